// Decode-step kernels for gfx950 (one token at a time, batch 1).
//
// Matvec (k_matvec): HBM-streaming, no MFMA. A workgroup owns R output rows
// (of up to three matrices that share the input, or the w1/w3 row pairs of
// SwiGLU). Its 256 threads walk the rows' 32-element blocks in memory order,
// so each wave reads one contiguous span per step (2 x 16-byte loads per
// lane for Q8, one for Q4), and form the exact int32 block dot with v_dot4
// against the Q8_0 activation staged in LDS. The per-block term
// ((float)s * wd) * xd is computed in parallel into LDS; one lane per row then
// adds the terms in block order, which is the reference's float order
// (kernels/scalar/k_scalar.c:13, :34). Fused epilogues: plain store,
// residual add, QKV bias + RoPE + KV-cache write, SwiGLU + Q8_0 quantize.
#include "kr_matvec.h"

namespace {

KMat to_kmat(const krh_mat *m) {
    KMat k = { (const uint8_t *)m->q, m->d, m->rows, m->cols, m->type, m->d16 };
    return k;
}

// workgroups resident at once: mv_wgs_per_cu per compute unit of this
// device (768 on an MI355X's 256 CUs)
int mv_resident(int epi = EPI_STORE) { return mv_wgs_per_cu(epi) * (krh_device_cus() > 0 ? krh_device_cus() : 256); }

// Rows per tile (one wave's): the largest power of two (at most cap, even for
// the RoPE pairs) that still gives every resident wave a tile; blocks per
// chunk: as many as MV_NPT slots per lane allow (a multiple of 4, for the
// 16-byte term reads).
constexpr int MV_MAX_LOC = 8;   // local rows per tile: a row's chunk then spans >= MV_NPT * 8 blocks

int mv_rows(int K, int total_rows, int local_per_row, int cap, int epi = EPI_STORE) {
    (void)K;
    int R = cap / local_per_row;
    if (R * local_per_row > 64) R = 64 / local_per_row;
    if (R * local_per_row > MV_MAX_LOC) R = MV_MAX_LOC / local_per_row;
    while (R > 2 && (total_rows + R - 1) / R < mv_resident(epi) * MV_WAVES) R /= 2;
    if (R > 1) R &= ~1;
    return R < 1 ? 1 : R;
}

int mv_chunk(int nb, int nloc) {
    int c = (MV_NPT * 64 / nloc) & ~3;
    if (c < 4) c = 4;
    return c < nb ? c : nb;
}

template <int EPI>
void launch_mv(MvArgs &a, const KMat &W) {
    const int nb = a.K / KR_QK;
    const int nloc = EPI == EPI_SWIGLU ? 2 * a.R : a.R;
    a.nbc = mv_chunk(nb, nloc);
    a.touch = 1;
    for (int i = 0; i < a.nmat; i++)
        if ((size_t)a.m[i].rows * (size_t)a.K >= ((size_t)1 << 32) / 32 * 32) a.touch = 0;
    const size_t lds = mv_lds(a.K, nloc, a.nbc, a.nw != nullptr).total;
    const int ntiles = a.tile0[a.nmat];
    const int wgs = (ntiles + MV_WAVES - 1) / MV_WAVES;
    const int grid = wgs > mv_resident(EPI) ? mv_resident(EPI) : wgs;
    if (a.K % KR_QK || lds > 64 * 1024 || grid <= 0 || nloc > 64 || nloc * a.nbc > MV_NPT * 64 ||
        (!a.xq && !a.xf)) {
        kr_fail(ML_E_SHAPE, "matvec shape", hipSuccess);
        return;
    }
    auto go = [&](auto kern) {
        hipLaunchKernelGGL(kern, dim3(grid), dim3(MV_THREADS), lds, kr_stream(), a);
    };
    bool mixed = false;
    for (int i = 1; i < a.nmat; i++) mixed = mixed || a.m[i].type != a.m[0].type;
    if (mixed && EPI != EPI_QKV) {
        kr_fail(ML_E_SHAPE, "matvec: matrices of one launch differ in type", hipSuccess);
        return;
    }
    if (EPI != EPI_ADD && a.nw && a.K <= SC_SHORT) {
        kr_matvec_short(EPI, mixed, W.type, W.d16, &a, sizeof a, grid, lds);
        kr_check_launch("matvec");
        return;
    }
    if constexpr (EPI == EPI_QKV) {
        if (mixed) {
            if (W.d16) go(k_matvec<EPI, QT_MIXED, 1>); else go(k_matvec<EPI, QT_MIXED, 0>);
            kr_check_launch("matvec");
            return;
        }
    }
    if (W.type == ML_Q8_0) {
        if (W.d16) go(k_matvec<EPI, ML_Q8_0, 1>); else go(k_matvec<EPI, ML_Q8_0, 0>);
    } else {
        if (W.d16) go(k_matvec<EPI, ML_Q4_0, 1>); else go(k_matvec<EPI, ML_Q4_0, 0>);
    }
    kr_check_launch("matvec");
}

// ---- rmsnorm + quantize, quantize ----

// One workgroup per token; each thread keeps its float4 slices of x and w in
// registers (n <= RN_MAX); see rmsnorm_q8_block.
// V4: float4 slices of x and w per thread (n <= RN_THREADS * V4 * 4): 4 for
// rows up to 4096 keep the kernel at a quarter of the registers of 16, so
// four times the tokens are in flight (each token's ordered sum is latency)
template <int V4>
__global__ void __launch_bounds__(RN_THREADS) k_rmsnorm_q8(int8_t *q, float *d, int dld, float *xb, const float *x,
                                                           const float *w, int n, float eps, int norm) {
    const size_t t = blockIdx.x;
    // scales [t][n / 32], or transposed [n / 32][dld] when dld > 0
    extern __shared__ __align__(16) float rn_smem[];
    rmsnorm_q8_block<RN_THREADS, V4>(q + t * n, d + (dld > 0 ? t : t * (n / KR_QK)), dld > 0 ? (size_t)dld : 1,
                                     xb ? xb + t * n : nullptr, x + t * n, w, n, eps, norm != 0, rn_smem);
}

// Q8_0 of ntok rows of n floats, QZ_CHUNK values per workgroup: thread t
// takes 4 consecutive values, 8 threads a 32-block (k_scalar.c:39-57).
constexpr int QZ_CHUNK = 1024;
__global__ void __launch_bounds__(256) k_quantize_q8(int8_t *q, size_t ldq, float *d, size_t ldd, int dld,
                                                    const float *x, size_t ldx, int n) {
    const size_t row = blockIdx.y;
    const int i = blockIdx.x * QZ_CHUNK + 4 * threadIdx.x;
    if (i >= n) return;   // n % 32 == 0: 8-thread groups are all in or all out
    const float4 v = *(const float4 *)(x + row * ldx + i);
    float m = fmaxf(fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w))), 0.0f);   // seeded with 0
    m = fmaxf(m, __shfl_xor(m, 1, 8));
    m = fmaxf(m, __shfl_xor(m, 2, 8));
    m = fmaxf(m, __shfl_xor(m, 4, 8));
    int packed = 0;
    float dd = 0.0f;
    if (!(m < KR_QUANT_TINY)) {
        const float id = kr_fdiv(127.0f, m);
        dd = kr_fdiv(m, 127.0f);
        packed = (kr_q8_elem(v.x, id) & 0xff) | (kr_q8_elem(v.y, id) & 0xff) << 8 |
                 (kr_q8_elem(v.z, id) & 0xff) << 16 | (int)((unsigned)kr_q8_elem(v.w, id) << 24);
    }
    *(int *)(q + row * ldq + i) = packed;
    if ((i & 31) == 0) {
        if (dld > 0) d[(size_t)(i >> 5) * dld + row] = dd;
        else d[row * ldd + (i >> 5)] = dd;
    }
}

// ---- embedding ----

__global__ void k_embed(float *x, const KMat e, const int *tok, float scale) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= e.cols) return;
    const int nb = e.cols / KR_QK, row = *tok, b = i / KR_QK, j = i % KR_QK;
    const float d = kr_scale(e.d, (size_t)row * nb + b, e.d16);
    int v;
    if (e.type == ML_Q8_0) {
        v = ((const int8_t *)e.q)[(size_t)row * e.cols + i];
    } else {
        const uint8_t p = e.q[((size_t)row * nb + b) * 16 + (j & 15)];
        v = (j < 16 ? (p & 0xF) : (p >> 4)) - 8;
    }
    float o = kr_fmul((float)v, d);
    if (scale != 1.0f) o = kr_fmul(o, scale);
    x[i] = o;
}

// ---- greedy pick ----

// First index of the maximum (model/sampler.c:57-61): NaN entries never win,
// and a NaN at index 0 keeps 0, as the sequential loop does.
// Greedy pick (model/sampler.c:57-61): the first index of the largest value,
// NaNs never chosen, index 0 when v[0] is NaN or every value is NaN. Each
// workgroup reduces a span of float4s (all its loads in flight together) to
// (value, smallest index among equal values); the last workgroup to finish
// (a counter it resets, so graph replays need no memset) reduces the
// partials. The partials live in static device memory: calls that overlap on
// one device race.
constexpr int AM_THREADS = 256, AM_V4 = 4;   // float4s per thread
constexpr int AM_MAX_WG = 1024;
__device__ float g_am_v[AM_MAX_WG];
__device__ int g_am_i[AM_MAX_WG];
__device__ unsigned g_am_count;

__device__ __forceinline__ void am_take(float &bv, int &bi, float v, int i) {
    if (v > bv || (v == bv && i < bi)) { bv = v; bi = i; }
}

__device__ __forceinline__ void am_reduce_block(float &bv, int &bi, float *sv, int *si) {
    for (int o = 32; o >= 1; o >>= 1) am_take(bv, bi, __shfl_xor(bv, o), __shfl_xor(bi, o));
    const int w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) { sv[w] = bv; si[w] = bi; }
    __syncthreads();
    if (threadIdx.x == 0)
        for (int k = 1; k < AM_THREADS / 64; k++) am_take(bv, bi, sv[k], si[k]);
}

__global__ void __launch_bounds__(AM_THREADS) k_argmax(int *tok, const float *v, int n, int *pos, int *log) {
    __shared__ float sv[AM_THREADS / 64];
    __shared__ int si[AM_THREADS / 64];
    __shared__ bool last;
    float bv = -INFINITY;
    int bi = INT_MAX;   // -inf with no index: any real value, -inf included, replaces it
    const int n4 = n / 4;
    const int base = blockIdx.x * AM_THREADS * AM_V4 + threadIdx.x;
    float4 x[AM_V4];
    if (n4 > 0) {
#pragma unroll
        for (int k = 0; k < AM_V4; k++) {
            const int i = base + k * AM_THREADS;
            x[k] = ((const float4 *)v)[min(i, n4 - 1)];
        }
    }
#pragma unroll
    for (int k = 0; k < AM_V4; k++) {
        const int i = base + k * AM_THREADS;
        if (i < n4) {
            am_take(bv, bi, x[k].x, 4 * i);
            am_take(bv, bi, x[k].y, 4 * i + 1);
            am_take(bv, bi, x[k].z, 4 * i + 2);
            am_take(bv, bi, x[k].w, 4 * i + 3);
        }
    }
    if (blockIdx.x == gridDim.x - 1 && threadIdx.x < n - 4 * n4) am_take(bv, bi, v[4 * n4 + threadIdx.x], 4 * n4 + threadIdx.x);
    am_reduce_block(bv, bi, sv, si);
    if (threadIdx.x == 0) {
        g_am_v[blockIdx.x] = bv;
        g_am_i[blockIdx.x] = bi;
        __threadfence();
        last = atomicAdd(&g_am_count, 1u) == gridDim.x - 1;
    }
    __syncthreads();
    if (!last) return;
    __threadfence();
    bv = -INFINITY;
    bi = INT_MAX;
    for (int k = threadIdx.x; k < (int)gridDim.x; k += AM_THREADS) am_take(bv, bi, g_am_v[k], g_am_i[k]);
    am_reduce_block(bv, bi, sv, si);
    if (threadIdx.x == 0) {
        g_am_count = 0;
        if (bi == INT_MAX || v[0] != v[0]) bi = 0;
        *tok = bi;
        if (pos) {
            const int p = *pos + 1;
            if (log) log[p] = bi;
            *pos = p;
        }
    }
}

__global__ void k_take_token(int *tok, const int *prompt, const int *pos) { *tok = prompt[*pos]; }
__global__ void k_advance(int *pos) { *pos += 1; }

__global__ void k_math_batch(int op, float *y, const float *a, const float *b, size_t n) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    switch (op) {
    case KRH_MATH_EXPF: y[i] = kr_expf(a[i]); break;
    case KRH_MATH_SQRT: y[i] = kr_fsqrt(a[i]); break;
    case KRH_MATH_DIV: y[i] = kr_fdiv(a[i], b[i]); break;
    case KRH_MATH_RMS_INV: y[i] = kr_fdiv(1.0f, kr_fsqrt(kr_fadd(kr_fdiv(a[i], b[i]), 1e-5f))); break;
    case KRH_MATH_F2H: y[i] = __uint_as_float(kr_f2h(a[i])); break;   // the half's bits in the low 16
    default: y[i] = 0.0f;
    }
}
__global__ void __launch_bounds__(256) k_ordered_sum(float *out, const float *t, int n, float s0) {
    extern __shared__ __align__(16) float os_t[];
    for (int i = threadIdx.x; i < n; i += 256) os_t[sc_at(i, sc_log_len(n))] = t[i];
    __syncthreads();
    const float s = kr_spec_sum<256>(os_t, n, (unsigned char *)(os_t + sc_terms_cap(n)), s0);
    if (threadIdx.x == 0) *out = s;
}
// the same with fewer reads in flight (the long-row prefill softmax's form)
__global__ void __launch_bounds__(256) k_ordered_sum_lean(float *out, const float *t, int n, float s0) {
    extern __shared__ __align__(16) float osl_t[];
    for (int i = threadIdx.x; i < n; i += 256) osl_t[sc_at(i, sc_log_len(n))] = t[i];
    __syncthreads();
    const float s = kr_spec_sum<256, false, false, true>(osl_t, n, (unsigned char *)(osl_t + sc_terms_cap(n)), s0);
    if (threadIdx.x == 0) *out = s;
}
// the same by 1024 threads, the decode softmax's workgroup
__global__ void __launch_bounds__(1024) k_ordered_sum_1024(float *out, const float *t, int n, float s0) {
    extern __shared__ __align__(16) float osk_t[];
    for (int i = threadIdx.x; i < n; i += 1024) osk_t[sc_at(i, sc_log_len(n))] = t[i];
    __syncthreads();
    const float s = kr_spec_sum<1024>(osk_t, n, (unsigned char *)(osk_t + sc_terms_cap(n)), s0);
    if (threadIdx.x == 0) *out = s;
}
// the single-wave mode, run by the second wave of the workgroup (its lanes
// and LDS are not the workgroup's first)
__global__ void __launch_bounds__(128) k_ordered_sum_wave(float *out, const float *t, int n, float s0) {
    extern __shared__ __align__(16) float osw_t[];
    if (threadIdx.x < 64) return;
    const int lane = threadIdx.x & 63, sh = sc_log_len(n);
    for (int i = lane; i < n; i += 64) osw_t[sc_at(i, sh)] = t[i];
    kr_wave_sync();
    const float s = kr_spec_sum<64, false, true>(osw_t, n, (unsigned char *)(osw_t + sc_terms_cap(n)), s0);
    if (lane == 0) *out = s;
}
__global__ void k_h2f_batch(float *y, const uint16_t *h, size_t n) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) y[i] = kr_h2f(h[i]);
}
__global__ void k_block_dots(int32_t *out, const KMat W, const int8_t *xq) {
    const int nb = W.cols / KR_QK;
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (size_t)W.rows * nb) return;
    const int b = (int)(i % nb);
    int4 w0, w1 = make_int4(0, 0, 0, 0);
    int s;
    __align__(16) int8_t xb[32];
    for (int j = 0; j < 32; j++) xb[j] = xq[b * 32 + j];
    if (W.type == ML_Q8_0) {
        w0 = ((const int4 *)(W.q + i * 32))[0];
        w1 = ((const int4 *)(W.q + i * 32))[1];
        s = block_dot<ML_Q8_0>(w0, w1, xb);
    } else {
        w0 = *(const int4 *)(W.q + i * 16);
        s = block_dot<ML_Q4_0>(w0, w1, xb);
    }
    out[i] = s;
}

}  // namespace

// ---- C ABI ----

extern "C" void krh_embed(float *x, const krh_mat *emb, const int *tok, float embed_scale) {
    hipLaunchKernelGGL(k_embed, dim3((emb->cols + 255) / 256), dim3(256), 0, kr_stream(), x, to_kmat(emb), tok,
                       embed_scale);
    kr_check_launch("embed");
}

extern "C" void krh_rmsnorm_q8(int8_t *q, float *d, float *xb, const float *x, const float *w, int n, float eps,
                               int ntok) {
    krh_rmsnorm_q8_t(q, d, 0, xb, x, w, n, eps, ntok);
}

extern "C" void krh_rmsnorm_q8_t(int8_t *q, float *d, int dld, float *xb, const float *x, const float *w, int n,
                                 float eps, int ntok) {
    // LDS: the squares and the ordered sum's scratch, within 64 KB
    const size_t lds = sizeof(float) * (size_t)sc_terms_cap(n) + sc_lds_bytes(n, RN_THREADS);
    if (n % KR_QK || n > RN_MAX || lds > 64 * 1024 || ntok <= 0 || (dld > 0 && dld < ntok)) {
        kr_fail(ML_E_SHAPE, "rmsnorm shape", hipSuccess);
        return;
    }
    if (n <= RN_THREADS * 4 * 4)
        hipLaunchKernelGGL(k_rmsnorm_q8<4>, dim3(ntok), dim3(RN_THREADS), lds, kr_stream(), q, d, dld, xb, x, w, n,
                           eps, 1);
    else
        hipLaunchKernelGGL(k_rmsnorm_q8<RN_V4>, dim3(ntok), dim3(RN_THREADS), lds, kr_stream(), q, d, dld, xb, x, w,
                           n, eps, 1);
    kr_check_launch("rmsnorm_q8");
}

extern "C" void krh_quantize_q8(int8_t *q, float *d, const float *x, int n, int ntok) {
    krh_quantize_q8_t(q, d, 0, x, n, ntok);
}

extern "C" void krh_quantize_q8_t(int8_t *q, float *d, int dld, const float *x, int n, int ntok) {
    if (n % KR_QK || n <= 0 || ntok <= 0 || (dld > 0 && dld < ntok)) {
        kr_fail(ML_E_SHAPE, "quantize shape", hipSuccess);
        return;
    }
    hipLaunchKernelGGL(k_quantize_q8, dim3((n + QZ_CHUNK - 1) / QZ_CHUNK, ntok), dim3(256), 0, kr_stream(), q,
                       (size_t)n, d, (size_t)(n / KR_QK), dld, x, (size_t)n, n);
    kr_check_launch("quantize_q8");
}

extern "C" void krh_quantize_q8_rows(int8_t *q, size_t ldq, float *d, size_t ldd, const float *x, size_t ldx, int n,
                                     int rows) {
    if (n % KR_QK || n <= 0 || rows < 0 || rows > KRH_ROWS_MAX || ldq % 4 || ldx % 4 || ((uintptr_t)x & 15) ||
        ((uintptr_t)q & 3)) {
        kr_fail(ML_E_SHAPE, "quantize_q8 rows: shape or alignment", hipSuccess);
        return;
    }
    if (rows == 0) return;
    hipLaunchKernelGGL(k_quantize_q8, dim3((n + QZ_CHUNK - 1) / QZ_CHUNK, rows), dim3(256), 0, kr_stream(), q, ldq, d,
                       ldd, 0, x, ldx, n);
    kr_check_launch("quantize_q8");
}

// the prologue results a launch also stores (MvArgs::keep_*): for a float
// input of any length (the register prologue and the one staged through LDS
// both store them), the normalized x only with a norm
struct MvKeep {
    float *xb;
    int8_t *xq;
    float *xd;
};

static bool keep_ok(const MvKeep &k, const float *xf, const float *nw, int K) {
    if (!k.xb && !k.xq) return true;
    const bool ok = xf && (k.xq != nullptr) == (k.xd != nullptr) && (!k.xb || nw) && !((uintptr_t)k.xq & 15) &&
                    !((uintptr_t)k.xb & 15);
    if (!ok) kr_fail(ML_E_SHAPE, "matvec keep: a float input, 16-byte aligned outputs", hipSuccess);
    return ok;
}

static void set_keep(MvArgs &a, const MvKeep &k) {
    a.keep_xb = k.xb;
    a.keep_xq = k.xq;
    a.keep_xd = k.xd;
}

static void mv_plain(float *y, const krh_mat *W, const int8_t *xq, const float *xd, const float *xf,
                     const float *nw, float eps, int accumulate, float *keep = nullptr, MvKeep kp = {}) {
    if (!keep_ok(kp, xf, nw, W->cols)) return;
    MvArgs a = {};
    a.keep = keep;
    set_keep(a, kp);
    a.m[0] = to_kmat(W);
    a.nmat = 1;
    a.R = mv_rows(W->cols, W->rows, 1, 64);
    // one-row tiles when two-row ones would give at most half of the
    // resident waves a tile (the 0.5B and 1B shapes' wo and w2: twice the
    // waves, a shorter chain of items each): 0.5B decode 888 -> 904 tok/s,
    // 1B 858 -> 866; the 8B's 4096-row matrices keep two rows (one-row
    // tiles measured slower there)
    if (a.R == 2 && (W->rows + 1) / 2 * 2 <= mv_resident() * MV_WAVES) a.R = 1;
    a.tile0[0] = 0;
    a.tile0[1] = (W->rows + a.R - 1) / a.R;
    a.xq = xq;
    a.xd = xd;
    a.xf = xf;
    a.nw = nw;
    a.eps = eps;
    a.K = W->cols;
    a.y[0] = y;
    if (accumulate) launch_mv<EPI_ADD>(a, a.m[0]);
    else launch_mv<EPI_STORE>(a, a.m[0]);
}

extern "C" void krh_matvec(float *y, const krh_mat *W, const int8_t *xq, const float *xd, int accumulate) {
    mv_plain(y, W, xq, xd, nullptr, nullptr, 0.0f, accumulate);
}

extern "C" void krh_matvec_residual(float *r, float *y, const krh_mat *W, const int8_t *xq, const float *xd) {
    mv_plain(r, W, xq, xd, nullptr, nullptr, 0.0f, 1, y);
}

extern "C" void krh_matvec_f_residual_keep(float *r, float *y, const krh_mat *W, const float *x, int8_t *xq,
                                           float *xd) {
    mv_plain(r, W, nullptr, nullptr, x, nullptr, 0.0f, 1, y, MvKeep{ nullptr, xq, xd });
}

extern "C" void krh_matvec_multi(float *const *y, const krh_mat *const *W, int nmat, const int8_t *xq,
                                 const float *xd) {
    if (nmat < 1 || nmat > 3) {
        kr_fail(ML_E_SHAPE, "matvec_multi: 1 to 3 matrices", hipSuccess);
        return;
    }
    for (int i = 1; i < nmat; i++)
        if (W[i]->cols != W[0]->cols || W[i]->type != W[0]->type || W[i]->d16 != W[0]->d16) {
            kr_fail(ML_E_SHAPE, "matvec_multi: one input length, type and scale kind", hipSuccess);
            return;
        }
    MvArgs a = {};
    int rows = 0;
    for (int i = 0; i < nmat; i++) rows += W[i]->rows;
    a.nmat = nmat;
    a.R = mv_rows(W[0]->cols, rows, 1, 64);
    a.tile0[0] = 0;
    for (int i = 0; i < nmat; i++) {
        a.m[i] = to_kmat(W[i]);
        a.y[i] = y[i];
        a.tile0[i + 1] = a.tile0[i] + (W[i]->rows + a.R - 1) / a.R;
    }
    a.xq = xq;
    a.xd = xd;
    a.K = W[0]->cols;
    launch_mv<EPI_STORE>(a, a.m[0]);
}

extern "C" void krh_matvec_f(float *y, const krh_mat *W, const float *x, int accumulate) {
    mv_plain(y, W, nullptr, nullptr, x, nullptr, 0.0f, accumulate);
}

extern "C" void krh_rmsnorm_matvec(float *y, const krh_mat *W, const float *x, const float *nw, float eps,
                                   int accumulate) {
    mv_plain(y, W, nullptr, nullptr, x, nw, eps, accumulate);
}

// k and v go to row *pos of the F32 cache (kv16: of the F16 cache, rounded
// to halves), or with stage set to the staging rows kc, vc of a Q8 cache
// (model/transformer.c:262-263)
static void qkv(float *q, float *kc, float *vc, const krh_mat *wq, const krh_mat *wk, const krh_mat *wv,
                const float *bq, const float *bk, const float *bv, const int8_t *xq, const float *xd, const float *xf,
                const float *nw, float eps, const float *rope_cos, const float *rope_sin, int head_dim,
                const int *pos, bool stage = false, bool kv16 = false, MvKeep kp = {}) {
    if (wq->cols != wk->cols || wq->cols != wv->cols || wk->rows != wv->rows || head_dim % 2 || wq->rows % 2 ||
        wk->rows % 2 || wq->type != wk->type || wq->d16 != wk->d16 || wv->d16 != wq->d16) {
        kr_fail(ML_E_SHAPE, "qkv shapes", hipSuccess);
        return;
    }
    if (!keep_ok(kp, xf, nw, wq->cols)) return;
    MvArgs a = {};
    a.m[0] = to_kmat(wq);
    a.m[1] = to_kmat(wk);
    a.m[2] = to_kmat(wv);
    a.nmat = 3;
    a.R = mv_rows(wq->cols, wq->rows + 2 * wk->rows, 1, 64, EPI_QKV);
    a.tile0[0] = 0;
    a.tile0[1] = (wq->rows + a.R - 1) / a.R;
    a.tile0[2] = a.tile0[1] + (wk->rows + a.R - 1) / a.R;
    a.tile0[3] = a.tile0[2] + (wv->rows + a.R - 1) / a.R;
    a.xq = xq;
    a.xd = xd;
    a.xf = xf;
    a.nw = nw;
    a.eps = eps;
    a.K = wq->cols;
    a.y[0] = q;
    a.y[1] = kc;
    a.y[2] = vc;
    a.bias[0] = bq;
    a.bias[1] = bk;
    a.bias[2] = bv;
    a.rope_cos = rope_cos;
    a.rope_sin = rope_sin;
    a.head_dim = head_dim;
    a.ld_cache = stage ? 0 : wk->rows;
    a.pos = pos;
    a.kv16 = kv16;
    set_keep(a, kp);
    // wv may be Q8 in a Q4 model: the launch then reads each matrix's type
    launch_mv<EPI_QKV>(a, a.m[0]);
}

extern "C" void krh_matvec_qkv(float *q, float *kc, float *vc, const krh_mat *wq, const krh_mat *wk,
                               const krh_mat *wv, const float *bq, const float *bk, const float *bv, const int8_t *xq,
                               const float *xd, const float *rope_cos, const float *rope_sin, int head_dim,
                               const int *pos) {
    qkv(q, kc, vc, wq, wk, wv, bq, bk, bv, xq, xd, nullptr, nullptr, 0.0f, rope_cos, rope_sin, head_dim, pos);
}

extern "C" void krh_rmsnorm_matvec_qkv(float *q, float *kc, float *vc, const krh_mat *wq, const krh_mat *wk,
                                       const krh_mat *wv, const float *bq, const float *bk, const float *bv,
                                       const float *x, const float *nw, float eps, const float *rope_cos,
                                       const float *rope_sin, int head_dim, const int *pos) {
    qkv(q, kc, vc, wq, wk, wv, bq, bk, bv, nullptr, nullptr, x, nw, eps, rope_cos, rope_sin, head_dim, pos);
}

extern "C" void krh_rmsnorm_matvec_qkv_f16(float *q, uint16_t *kc, uint16_t *vc, const krh_mat *wq,
                                           const krh_mat *wk, const krh_mat *wv, const float *bq, const float *bk,
                                           const float *bv, const float *x, const float *nw, float eps,
                                           const float *rope_cos, const float *rope_sin, int head_dim,
                                           const int *pos) {
    qkv(q, (float *)kc, (float *)vc, wq, wk, wv, bq, bk, bv, nullptr, nullptr, x, nw, eps, rope_cos, rope_sin,
        head_dim, pos, false, true);
}

extern "C" void krh_rmsnorm_matvec_qkv_keep(float *q, float *k, float *v, const krh_mat *wq, const krh_mat *wk,
                                            const krh_mat *wv, const float *bq, const float *bk, const float *bv,
                                            const float *x, const float *nw, float eps, const float *rope_cos,
                                            const float *rope_sin, int head_dim, const int *pos, float *xb,
                                            int8_t *xq, float *xd) {
    qkv(q, k, v, wq, wk, wv, bq, bk, bv, nullptr, nullptr, x, nw, eps, rope_cos, rope_sin, head_dim, pos, true, false,
        MvKeep{ xb, xq, xd });
}

extern "C" void krh_rmsnorm_matvec_qkv_stage(float *q, float *k, float *v, const krh_mat *wq, const krh_mat *wk,
                                             const krh_mat *wv, const float *bq, const float *bk, const float *bv,
                                             const float *x, const float *nw, float eps, const float *rope_cos,
                                             const float *rope_sin, int head_dim, const int *pos) {
    qkv(q, k, v, wq, wk, wv, bq, bk, bv, nullptr, nullptr, x, nw, eps, rope_cos, rope_sin, head_dim, pos, true);
}

static void swiglu(float *h, const krh_mat *w1, const krh_mat *w3, const int8_t *xq, const float *xd, const float *xf,
                   const float *nw, float eps, float *keep = nullptr, MvKeep kp = {}) {
    if (!keep_ok(kp, xf, nw, w1->cols)) return;
    if (w1->rows != w3->rows || w1->cols != w3->cols || w1->type != w3->type || w1->d16 != w3->d16) {
        kr_fail(ML_E_SHAPE, "swiglu shapes", hipSuccess);
        return;
    }
    MvArgs a = {};
    a.m[0] = to_kmat(w1);
    a.m[1] = to_kmat(w3);
    a.nmat = 1;
    a.R = mv_rows(w1->cols, w1->rows, 2, 4);   // 2 rows of w1 and w3 a tile: measured fastest
    a.tile0[0] = 0;
    a.tile0[1] = (w1->rows + a.R - 1) / a.R;
    a.xq = xq;
    a.xd = xd;
    a.xf = xf;
    a.nw = nw;
    a.eps = eps;
    a.K = w1->cols;
    a.y[0] = h;
    a.keep = keep;
    set_keep(a, kp);
    launch_mv<EPI_SWIGLU>(a, a.m[0]);
}

extern "C" void krh_rmsnorm_matvec_swiglu_keep(float *h, float *u, const krh_mat *w1, const krh_mat *w3,
                                               const float *x, const float *nw, float eps, float *xb, int8_t *xq,
                                               float *xd) {
    swiglu(h, w1, w3, nullptr, nullptr, x, nw, eps, u, MvKeep{ xb, xq, xd });
}

extern "C" void krh_matvec_swiglu_keep(float *h, float *u, const krh_mat *w1, const krh_mat *w3, const int8_t *xq,
                                       const float *xd) {
    swiglu(h, w1, w3, xq, xd, nullptr, nullptr, 0.0f, u);
}

extern "C" void krh_matvec_swiglu(float *h, const krh_mat *w1, const krh_mat *w3, const int8_t *xq, const float *xd) {
    swiglu(h, w1, w3, xq, xd, nullptr, nullptr, 0.0f);
}

extern "C" void krh_rmsnorm_matvec_swiglu(float *h, const krh_mat *w1, const krh_mat *w3, const float *x,
                                          const float *nw, float eps) {
    swiglu(h, w1, w3, nullptr, nullptr, x, nw, eps);
}

extern "C" void krh_argmax(int *tok, const float *logits, int n, int *pos, int *log) {
    const int per_wg = AM_THREADS * AM_V4 * 4;
    const int grid = (n + per_wg - 1) / per_wg;
    if (n < 1 || grid > AM_MAX_WG) {
        kr_fail(ML_E_SHAPE, "argmax size", hipSuccess);
        return;
    }
    hipLaunchKernelGGL(k_argmax, dim3(grid), dim3(AM_THREADS), 0, kr_stream(), tok, logits, n, pos, log);
    kr_check_launch("argmax");
}

extern "C" void krh_take_token(int *tok, const int *prompt, const int *pos) {
    hipLaunchKernelGGL(k_take_token, dim3(1), dim3(1), 0, kr_stream(), tok, prompt, pos);
    kr_check_launch("take_token");
}

extern "C" void krh_advance(int *pos) {
    hipLaunchKernelGGL(k_advance, dim3(1), dim3(1), 0, kr_stream(), pos);
    kr_check_launch("advance");
}

extern "C" void krh_math_batch(int op, float *y, const float *a, const float *b, size_t n) {
    hipLaunchKernelGGL(k_math_batch, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, kr_stream(), op, y, a, b, n);
    kr_check_launch("math_batch");
}

extern "C" void krh_ordered_sum(float *out, const float *t, int n, float s0) {
    if (n < 1 || n > KRH_ORDERED_SUM_MAX) {
        kr_fail(ML_E_SHAPE, "ordered_sum size", hipSuccess);
        return;
    }
    const size_t lds = sizeof(float) * (size_t)sc_terms_cap(n) + sc_lds_bytes(n, RN_THREADS);
    hipLaunchKernelGGL(k_ordered_sum, dim3(1), dim3(256), lds, kr_stream(), out, t, n, s0);
    kr_check_launch("ordered_sum");
}

extern "C" void krh_ordered_sum_lean(float *out, const float *t, int n, float s0) {
    if (n < 1 || n > KRH_ORDERED_SUM_MAX) {
        kr_fail(ML_E_SHAPE, "ordered_sum_lean size", hipSuccess);
        return;
    }
    const size_t lds = sizeof(float) * (size_t)sc_terms_cap(n) + sc_lds_bytes(n, RN_THREADS);
    hipLaunchKernelGGL(k_ordered_sum_lean, dim3(1), dim3(256), lds, kr_stream(), out, t, n, s0);
    kr_check_launch("ordered_sum_lean");
}

extern "C" void krh_ordered_sum_1024(float *out, const float *t, int n, float s0) {
    if (n < 1 || n > KRH_ORDERED_SUM_MAX) {
        kr_fail(ML_E_SHAPE, "ordered_sum_1024 size", hipSuccess);
        return;
    }
    const size_t lds = sizeof(float) * (size_t)sc_terms_cap(n) + sc_lds_bytes(n, 1024);
    hipLaunchKernelGGL(k_ordered_sum_1024, dim3(1), dim3(1024), lds, kr_stream(), out, t, n, s0);
    kr_check_launch("ordered_sum_1024");
}
extern "C" void krh_ordered_sum_wave(float *out, const float *t, int n, float s0) {
    if (n < 1 || n > KRH_ORDERED_SUM_WAVE_MAX) {
        kr_fail(ML_E_SHAPE, "ordered_sum_wave size", hipSuccess);
        return;
    }
    const size_t lds = sizeof(float) * (size_t)sc_terms_cap(n) + sc_lds_bytes(n, 64);
    hipLaunchKernelGGL(k_ordered_sum_wave, dim3(1), dim3(128), lds, kr_stream(), out, t, n, s0);
    kr_check_launch("ordered_sum_wave");
}

extern "C" void krh_h2f_batch(float *y, const uint16_t *h, size_t n) {
    hipLaunchKernelGGL(k_h2f_batch, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, kr_stream(), y, h, n);
    kr_check_launch("h2f_batch");
}

extern "C" void krh_block_dots(int32_t *s, const krh_mat *W, const int8_t *xq) {
    const size_t n = (size_t)W->rows * (W->cols / KR_QK);
    hipLaunchKernelGGL(k_block_dots, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, kr_stream(), s, to_kmat(W),
                       xq);
    kr_check_launch("block_dots");
}
