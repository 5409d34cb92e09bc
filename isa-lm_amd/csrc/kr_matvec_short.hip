// The normalizing decode matvecs whose rmsnorm sums at most SC_SHORT terms
// (k_matvec with SH). A code object of their own: in the same one as the
// kernels of longer rows they made those slower (the 8B shape's attention
// block 41.4 -> 42.1 us, its own kernels' code and offsets unchanged; where a
// process's code and buffers lie alone moves that block between 41.0 and 41.9).
#include <cstring>

#include "kr_matvec.h"

void kr_matvec_short(int epi, bool mixed, int type, int d16, const void *args, size_t bytes, int grid, size_t lds) {
    MvArgs a;
    static_assert(std::is_trivially_copyable<MvArgs>::value, "copied as bytes");
    if (bytes != sizeof a) {
        kr_fail(ML_E_SHAPE, "matvec arguments", hipSuccess);
        return;
    }
    memcpy(&a, args, sizeof a);
    auto go = [&](auto kern) { hipLaunchKernelGGL(kern, dim3(grid), dim3(MV_THREADS), lds, kr_stream(), a); };
    auto pick = [&](auto e) {
        constexpr int EPI = decltype(e)::value;
        if (type == ML_Q8_0) {
            if (d16) go(k_matvec<EPI, ML_Q8_0, 1, true>); else go(k_matvec<EPI, ML_Q8_0, 0, true>);
        } else {
            if (d16) go(k_matvec<EPI, ML_Q4_0, 1, true>); else go(k_matvec<EPI, ML_Q4_0, 0, true>);
        }
    };
    if (mixed) {   // q|k|v
        if (d16) go(k_matvec<EPI_QKV, QT_MIXED, 1, true>); else go(k_matvec<EPI_QKV, QT_MIXED, 0, true>);
    } else if (epi == EPI_QKV) {
        pick(std::integral_constant<int, EPI_QKV>{});
    } else if (epi == EPI_SWIGLU) {
        pick(std::integral_constant<int, EPI_SWIGLU>{});
    } else {
        pick(std::integral_constant<int, EPI_STORE>{});
    }
}
