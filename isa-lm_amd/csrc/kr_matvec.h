// The decode matvec's kernel (see kr_decode.hip's head comment), for the two
// translation units that instantiate it: kr_decode.hip, and kr_matvec_short.hip
// with the short norm sums.
#pragma once
#include <type_traits>

#include "kr_internal.h"
#include "kr_numerics.h"
#include "kr_chain.h"

namespace {

struct KMat {
    const uint8_t *q;
    const void *d;
    int rows, cols, type, d16;
};

enum { EPI_STORE = 0, EPI_ADD = 1, EPI_QKV = 2, EPI_SWIGLU = 3 };
// weight type template argument: ML_Q8_0, ML_Q4_0, or QT_MIXED, the type of
// each matrix read from its KMat at run time (q|k|v of a Q4 model with its
// v in Q8: one launch and one prologue; an item lies in one matrix, so the
// branch is uniform across the wave)
constexpr int QT_MIXED = 7;
template <int QT> __device__ __forceinline__ bool qt_is_q8(int type) {
    return QT == QT_MIXED ? type == ML_Q8_0 : QT == ML_Q8_0;
}

struct MvArgs {
    KMat m[3];
    int tile0[4];        // first workgroup of matrix i; tile0[nmat] = grid size
    int nmat;
    int R;               // output rows per tile
    int nbc;             // blocks per chunk (set by launch_mv)
    const int8_t *xq;    // Q8_0 activation; or NULL: quantize xf in the prologue,
    const float *xd;     // after rmsnorm with weight nw when nw is set
    const float *xf;
    const float *nw;
    float eps;
    int K;
    float *y[3];
    const float *bias[3];
    const float *rope_cos, *rope_sin;
    int head_dim, ld_cache;
    const int *pos;
    int kv16;            // EPI_QKV: k and v rows are the F16 cache's (halves)
    float *keep;         // EPI_ADD: receives the product W x as well; EPI_SWIGLU: receives w3 x
    // workgroup 0 stores the prologue's results when set (float inputs):
    // the normalized x (with nw) and its Q8_0 quants and scales, as the
    // reference's separate rmsnorm and quantize_q8 calls leave them in memory
    float *keep_xb;
    int8_t *keep_xq;
    float *keep_xd;
    int touch;           // touches ahead (set by launch_mv: every matrix below 4 GiB)
};

constexpr int MV_THREADS = 256;
constexpr int MV_NPT = 2;   // weight blocks per thread per work item
constexpr int MV_DEPTH = 2;    // work items in flight per wave: a wave that issues more loads than the
                               // memory pipeline holds stalls at issue
#ifndef KR_MV_TOUCH
#define KR_MV_TOUCH 2
#endif
// Items a wave touches ahead (the item MV_TOUCH after the one whose dots run;
// 1: none): a 2-byte read per 128-byte line of an item's quants and per row
// of its scales, so that the lines are in this XCD's L2 (and the Infinity
// Cache) when the item's own loads go out, above all under a prologue, when
// the register-loaded item is the only other memory traffic. 2 or 4; 4
// (three items touched) was slower: a wave's loads return in order, so the
// item loads wait behind touches further out.
constexpr int MV_TOUCH = KR_MV_TOUCH;
// Activations held in registers by the prologue (longer ones are staged
// through LDS from memory): sized so that the kernel fits 128 VGPRs, four
// workgroups per CU
constexpr int MV_XQ_MAX = 8192;   // quantized activations up to this length are staged from registers
constexpr int MV_XF_MAX = 4096;    // float activations up to this length are normalized and quantized from registers
constexpr int MV_XF_PLAIN_MAX = 16384;  // float activations without a norm: quantized from registers up to this length,
constexpr int MV_XF_PASS = 4096;        // in passes of this many

template <typename T> __device__ __forceinline__ T pick3(int i, T a, T b, T c) { return i == 0 ? a : (i == 1 ? b : c); }

// Exact int32 dot of one weight block with the activation block in LDS.
template <int QT>
__device__ __forceinline__ int block_dot(const int4 w0, const int4 w1, const int8_t *xb) {
    const int4 xa = *(const int4 *)xb, xc = *(const int4 *)(xb + 16);
    int s = 0;
    if (QT == ML_Q8_0) {
        s = kr_dot4(w0.x, xa.x, s); s = kr_dot4(w0.y, xa.y, s);
        s = kr_dot4(w0.z, xa.z, s); s = kr_dot4(w0.w, xa.w, s);
        s = kr_dot4(w1.x, xc.x, s); s = kr_dot4(w1.y, xc.y, s);
        s = kr_dot4(w1.z, xc.z, s); s = kr_dot4(w1.w, xc.w, s);
    } else {
        // byte j holds element j (low nibble) and j+16 (high); nibble n is
        // weight n-8, so the dot is sum(n x) - 8 sum(x), all exact in int32
        const unsigned M = 0x0F0F0F0Fu;
        s = kr_dot4((int)((unsigned)w0.x & M), xa.x, s); s = kr_dot4((int)((unsigned)w0.y & M), xa.y, s);
        s = kr_dot4((int)((unsigned)w0.z & M), xa.z, s); s = kr_dot4((int)((unsigned)w0.w & M), xa.w, s);
        s = kr_dot4((int)(((unsigned)w0.x >> 4) & M), xc.x, s); s = kr_dot4((int)(((unsigned)w0.y >> 4) & M), xc.y, s);
        s = kr_dot4((int)(((unsigned)w0.z >> 4) & M), xc.z, s); s = kr_dot4((int)(((unsigned)w0.w >> 4) & M), xc.w, s);
        const int one = 0x01010101;
        int sx = 0;
        sx = kr_dot4(one, xa.x, sx); sx = kr_dot4(one, xa.y, sx); sx = kr_dot4(one, xa.z, sx); sx = kr_dot4(one, xa.w, sx);
        sx = kr_dot4(one, xc.x, sx); sx = kr_dot4(one, xc.y, sx); sx = kr_dot4(one, xc.z, sx); sx = kr_dot4(one, xc.w, sx);
        s -= 8 * sx;
    }
    return s;
}

// Q8_0 of the 4 values v = x[i..i+3] (k_scalar.c:39-57): 8 consecutive
// lanes hold a 32-block (all 8 must call together); the block max is exact in
// any order. q[i..i+3] receive the values, d[(i / 32) * dstep] the scale.
__device__ __forceinline__ void kr_quant4(float4 v, int i, int8_t *q, float *d, size_t dstep) {
    // seeded with 0 as the reference's loop is: NaNs never raise the max
    float m = fmaxf(fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w))), 0.0f);
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
    *(int *)(q + i) = packed;
    if ((i & 31) == 0) d[(size_t)(i >> 5) * dstep] = dd;
}

// Q8_0 of the 16 values v = x[i..i+15] held by this lane (k_scalar.c:39-57):
// a 32-block is two lanes' halves, lanes 2j and 2j + 1 (both must call
// together; i % 32 == 16 in the odd one). The block max is exact in any
// order; the two divisions are paid once per 16 values instead of per 4.
// q[i..i+15] receive the values, d[i / 32] the scale.
__device__ __forceinline__ void kr_quant16(const float4 (&v)[4], int i, int8_t *q, float *d) {
    float m = 0.0f;   // seeded with 0 as the reference's loop is: NaNs never raise the max
#pragma unroll
    for (int k = 0; k < 4; k++)
        m = fmaxf(fmaxf(m, fmaxf(fabsf(v[k].x), fabsf(v[k].y))), fmaxf(fabsf(v[k].z), fabsf(v[k].w)));
    m = fmaxf(m, __uint_as_float((unsigned)__builtin_amdgcn_mov_dpp((int)__float_as_uint(m), 0xB1, 0xF, 0xF, false)));
    int4 packed = make_int4(0, 0, 0, 0);
    float dd = 0.0f;
    if (!(m < KR_QUANT_TINY)) {
        const float id = kr_fdiv(127.0f, m);
        dd = kr_fdiv(m, 127.0f);
        auto p4 = [&](float4 x) {
            return (kr_q8_elem(x.x, id) & 0xff) | (kr_q8_elem(x.y, id) & 0xff) << 8 |
                   (kr_q8_elem(x.z, id) & 0xff) << 16 | (int)((unsigned)kr_q8_elem(x.w, id) << 24);
        };
        packed = make_int4(p4(v[0]), p4(v[1]), p4(v[2]), p4(v[3]));
    }
    *(int4 *)(q + i) = packed;
    if ((i & 31) == 0) d[i >> 5] = dd;
}

// the rmsnorm output (x * inv) * w (k_scalar.c:63)
__device__ __forceinline__ float4 kr_norm4(float4 x, float inv, float4 w) {
    return make_float4(kr_fmul(kr_fmul(x.x, inv), w.x), kr_fmul(kr_fmul(x.y, inv), w.y),
                       kr_fmul(kr_fmul(x.z, inv), w.z), kr_fmul(kr_fmul(x.w, inv), w.w));
}

// Q8_0 of K floats into LDS: each thread takes 4 consecutive values, 8
// threads a 32-block. K % 32 == 0, x 16-byte aligned. With w: the rmsnorm
// output (x * inv) * w is quantized, and also stored into xb when it is set.
__device__ __forceinline__ void quantize_to_lds(const float *x, int K, int8_t *xs, float *xds,
                                                const float *w = nullptr, float inv = 1.0f, float *xb = nullptr) {
    constexpr int B = 4;   // float4 loads in flight per thread
    for (int base = 0; base < K; base += 4 * B * MV_THREADS) {
        float4 vs[B], ws[B];
#pragma unroll
        for (int k = 0; k < B; k++) {
            const int i = base + 4 * (k * MV_THREADS + threadIdx.x);
            if (i < K) {
                vs[k] = *(const float4 *)(x + i);
                if (w) ws[k] = *(const float4 *)(w + i);
            }
        }
#pragma unroll
        for (int k = 0; k < B; k++) {
            const int i = base + 4 * (k * MV_THREADS + threadIdx.x);   // K % 32 == 0: 8-lane groups all in or all out
            if (i < K) {
                const float4 o = w ? kr_norm4(vs[k], inv, ws[k]) : vs[k];
                kr_quant4(o, i, xs, xds, 1);
                if (xb) *(float4 *)(xb + i) = o;
            }
        }
    }
}

// rmsnorm + Q8_0 of one row of n floats by the NT threads of a workgroup
// (n <= NT * V4 * 4, n % 32 == 0, rows 16-byte aligned): every thread keeps
// its float4 slices of x and w in registers; the squares x_i * x_i (each one
// rounded product, as in the scalar loop) go to LDS (sq: sc_terms_cap(n)
// floats and then sc_lds_bytes(n, NT) bytes) for the ordered sum
// (k_scalar.c:59-64); then every thread forms (x * inv) * w for its values
// and 8-thread groups quantize their 32-element blocks (k_scalar.c:39-57).
// q[i] and d[(i / 32) * dstep] receive them, xb (nullable) the floats.
constexpr int RN_THREADS = 256, RN_V4 = 16, RN_MAX = RN_THREADS * RN_V4 * 4;

template <int NT, int V4>
__device__ __forceinline__ void rmsnorm_q8_block(int8_t *q, float *d, size_t dstep, float *xb, const float *x,
                                                 const float *w, int n, float eps, bool norm, float *sq) {
    const int tid = threadIdx.x;
    float4 xv[V4], wv[V4];
#pragma unroll
    for (int k = 0; k < V4; k++) {
        const int i = min((k * NT + tid) * 4, n - 4);
        xv[k] = *(const float4 *)(x + i);
        if (norm) wv[k] = *(const float4 *)(w + i);
    }
    float inv = 1.0f;
    if (norm) {
        const int sh = sc_log_len(n);
#pragma unroll
        for (int k = 0; k < V4; k++) {
            const int i = (k * NT + tid) * 4;
            if (i < n)
                *(float4 *)(sq + sc_at(i, sh)) = make_float4(kr_fmul(xv[k].x, xv[k].x), kr_fmul(xv[k].y, xv[k].y),
                                                  kr_fmul(xv[k].z, xv[k].z), kr_fmul(xv[k].w, xv[k].w));
        }
        __syncthreads();
        const float ss = kr_spec_sum<NT>(sq, n, (unsigned char *)(sq + sc_terms_cap(n)));
        inv = kr_fdiv(1.0f, kr_fsqrt(kr_fadd(kr_fdiv(ss, (float)n), eps)));
    }
#pragma unroll
    for (int k = 0; k < V4; k++) {
        const int i = (k * NT + tid) * 4;
        if (i < n) {   // n % 32 == 0: 8-thread groups are all in or all out
            const float4 o = norm ? kr_norm4(xv[k], inv, wv[k]) : xv[k];
            if (xb) *(float4 *)(xb + i) = o;
            kr_quant4(o, i, q, d, dstep);
        }
    }
}

// Loads of one work item (row tile, block chunk) by one wave: slot k of lane
// l is local block l + 64 k of the item, blocks fastest, so each load
// instruction reads contiguous spans (a Q8_0 block as two 16-byte loads, a
// Q4_0 block as one). Every slot loads (slots past the item re-read its first
// block and are not used), so no load waits on a branch.
struct MvSlots {
    int4 w0[MV_NPT], w1[MV_NPT];
    uint32_t wd[MV_NPT];   // raw scale bits: widened at use, after every load is in flight
};

// Where a work item lies: matrix mi, first row, rows, local rows (SwiGLU's w3
// rows follow its w1 rows), first block and block count of the chunk.
struct MvItem {
    int mi, row0, nr, nloc, c0, nbc;
};

template <int EPI>
__device__ __forceinline__ MvItem mv_item(const MvArgs &a, int tile, int chunk, int nb) {
    // constant indices only: a runtime index into the argument block makes
    // the compiler read it with a vector load, whose wait would drain the
    // weight loads in flight
    MvItem it;
    it.mi = 0;
    if (EPI != EPI_SWIGLU)
        it.mi = (a.nmat > 1 && tile >= a.tile0[1]) + (a.nmat > 2 && tile >= a.tile0[2]);
    const int rows = pick3(it.mi, a.m[0].rows, a.m[1].rows, a.m[2].rows);
    it.row0 = (tile - pick3(it.mi, a.tile0[0], a.tile0[1], a.tile0[2])) * a.R;
    it.nr = min(a.R, rows - it.row0);
    it.nloc = EPI == EPI_SWIGLU ? 2 * it.nr : it.nr;
    it.c0 = chunk * a.nbc;
    it.nbc = min(a.nbc, nb - it.c0);
    return it;
}

template <int EPI, int QT, int D16>
__device__ __forceinline__ void mv_load(MvSlots &S, const MvArgs &a, const MvItem &it, int nb, int lane) {
    const KMat W = pick3(it.mi, a.m[0], a.m[1], a.m[2]);
    const KMat W2 = a.m[1];
    const int n = it.nloc * it.nbc;
    int lr = lane / it.nbc, b = lane - lr * it.nbc;
    const int sr = 64 / it.nbc, sb = 64 - sr * it.nbc;
#pragma unroll
    for (int k = 0; k < MV_NPT; k++) {
        const bool in = lane + k * 64 < n;
        const bool second = EPI == EPI_SWIGLU && in && lr >= it.nr;
        const uint8_t *q = second ? W2.q : W.q;
        const void *d = second ? W2.d : W.d;
        const size_t blk = in ? (size_t)(it.row0 + (second ? lr - it.nr : lr)) * nb + it.c0 + b
                              : (size_t)it.row0 * nb + it.c0;
        if (qt_is_q8<QT>(W.type)) {
            const int4 *p = (const int4 *)(q + blk * 32);
            S.w0[k] = p[0];
            S.w1[k] = p[1];
        } else {
            S.w0[k] = *(const int4 *)(q + blk * 16);
            S.w1[k] = make_int4(0, 0, 0, 0);
        }
        S.wd[k] = D16 ? (uint32_t)((const uint16_t *)d)[blk] : ((const uint32_t *)d)[blk];
        b += sb;
        lr += sr;
        if (b >= it.nbc) { b -= it.nbc; lr++; }
    }
}

// One dword per lane from one of the item's lines (a touch: the value is not
// used): lanes l < n / 4 read local block 4 l (a 128-byte line of Q8_0 quants,
// half of one of Q4_0), the next lanes the first and the middle scale of each
// local row. The local blocks map to rows and blocks as in mv_load. Offsets
// are 32-bit: the launcher sets touch only when every matrix's quants and
// scales stay below 4 GiB.
// (a 2-byte read of the block's first quants or of the scale itself)
template <int EPI, int QT, int D16>
__device__ __forceinline__ int mv_touch(const MvArgs &a, const MvItem &it, int nb, int lane) {
    const KMat W = pick3(it.mi, a.m[0], a.m[1], a.m[2]);
    const KMat W2 = a.m[1];
    const int n = max(it.nloc * it.nbc, 1), nql = (n + 3) >> 2;
    const bool scale = lane >= nql;
    const int sl = lane - nql;
    int j = scale ? min(sl >> 1, max(it.nloc, 1) - 1) * it.nbc + (sl & 1) * (it.nbc >> 1) : 4 * lane;
    j = min(j, n - 1);
    const int lr = j / it.nbc, b = j - lr * it.nbc;
    const bool second = EPI == EPI_SWIGLU && lr >= it.nr;
    const unsigned blk = (unsigned)(it.row0 + (second ? lr - it.nr : lr)) * (unsigned)nb + (unsigned)(it.c0 + b);
    const uint8_t *base = scale ? (const uint8_t *)(second ? W2.d : W.d) : (second ? W2.q : W.q);
    const unsigned off = scale ? blk * (D16 ? 2u : 4u) : blk * (qt_is_q8<QT>(W.type) ? 32u : 16u);
    return *(const uint16_t *)(base + off);   // 2 bytes: in bounds for every block and scale
}

// LDS layout of k_matvec (byte offsets, every region 16-byte aligned): the
// Q8_0 activation and its scales, each wave's chunk terms (rows of ts floats:
// a multiple of 4 plus 4, for 16-byte reads with a 4-bank shift between
// rows) and row sums, and for a normalizing launch the squares and the
// ordered sum's scratch.
constexpr int MV_WAVES = MV_THREADS / 64;
struct MvLds {
    int ts, xds, t2, sums, sq, total;
};
__host__ __device__ constexpr int mv_align16(int b) { return (b + 15) & ~15; }
__host__ __device__ inline MvLds mv_lds(int K, int maxloc, int nbc, bool norm) {
    MvLds l = {};
    l.ts = (nbc + 3) / 4 * 4 + 4;
    l.xds = mv_align16(K);
    l.t2 = mv_align16(l.xds + 4 * (K / KR_QK));
    l.sums = mv_align16(l.t2 + 4 * MV_WAVES * maxloc * l.ts);
    l.sq = mv_align16(l.sums + 4 * MV_WAVES * maxloc);
    l.total = norm ? l.sq + 4 * sc_terms_cap(K) + sc_lds_bytes(K, MV_THREADS) : l.sq;
    return l;
}

// Orders one wave's LDS writes before its later reads for the compiler (a
// wave's LDS operations execute in order).

// y rows [row0, row0 + R) of up to three matrices sharing the activation
// (QKV), or the w1 and w3 rows [row0, row0 + R) (SwiGLU). Each wave streams
// its own row tiles (tiles gw, gw + GW, ... of the GW waves of the grid),
// each split into chunks of nbc blocks, and issues the loads of item i + 1
// before it uses item i's; waves never wait for each other, so the weight
// stream never stops for the dots, the ordered sums or the epilogues. Per
// item: the exact int32 block dots and their terms ((float)s * wd) * xd go to
// the wave's LDS rows; one lane per row continues its row's ordered sum over
// the chunk's terms, in block order (kernels/scalar/k_scalar.c:13, :34). On a
// tile's last chunk the sums go through the epilogue. Before the first item's
// dots the workgroup stages the activation into LDS (while the first loads
// are in flight): copied, quantized, or normalized first (rmsnorm's ordered
// sum, k_scalar.c:59-64) and quantized.
// workgroups of a launch resident on one CU: three (up to 168 VGPRs, three
// waves a SIMD). With the prologue's Q8_0 in half-blocks per lane and one
// item touched ahead, the 8B decode ran at 316.0 tok/s with four (128
// VGPRs) and 319.3 with three; with the 4-value quantization and no
// touches, four had been ahead (307.5 against 310.9 with three and
// touches). The q|k|v grid of the 8B shape is 768 workgroups in any case
// (3,072 two-row tiles).
#ifndef KR_MV_WGS
#define KR_MV_WGS 3
#endif
constexpr int mv_wgs_per_cu(int epi) { return epi == EPI_QKV ? 3 : KR_MV_WGS; }

// SH: a normalizing launch whose sum is short (K <= SC_SHORT). A kernel of
// its own: as a branch it made the 8B shape's attention block 0.8 us slower.
template <int EPI, int QT, int D16, bool SH = false>
__global__ void __launch_bounds__(MV_THREADS, mv_wgs_per_cu(EPI)) k_matvec(const MvArgs a) {
    extern __shared__ __align__(16) unsigned char smem[];
    const int K = a.K, nb = K / KR_QK, tid = threadIdx.x;
    const int ntiles = a.nmat == 1 ? a.tile0[1] : a.nmat == 2 ? a.tile0[2] : a.tile0[3];
    const int lane = tid & 63, wave = tid >> 6;
    const int gw = blockIdx.x * MV_WAVES + wave, GW = gridDim.x * MV_WAVES;   // this wave; waves in the grid
    const int pos = EPI == EPI_QKV ? *a.pos : 0;
    const int maxloc = EPI == EPI_SWIGLU ? 2 * a.R : a.R;
    const MvLds L = mv_lds(K, maxloc, a.nbc, a.nw != nullptr);
    const int ts = L.ts;
    int8_t *xs = (int8_t *)smem;
    float *xds = (float *)(smem + L.xds);
    float *T = (float *)(smem + L.t2) + wave * maxloc * ts;   // this wave's terms [maxloc][ts]
    float *sums = (float *)(smem + L.sums) + wave * maxloc;   // and row sums
    float *sq = (float *)(smem + L.sq);      // rmsnorm prologue only: the squares, then the ordered sum's scratch
    if ((int)blockIdx.x * MV_WAVES >= ntiles) return;
    const int nch = (nb + a.nbc - 1) / a.nbc;

    // items are loaded MV_DEPTH - 1 ahead of the one whose dots run: S[P]
    // holds item P of every MV_DEPTH; (ltile, lchunk) is the next item to load
    int tile = gw, chunk = 0, ltile = gw, lchunk = 0;
    auto next_item = [&](int &t, int &c) {
        if (++c == nch) { c = 0; t += GW; }
    };
    auto load_item = [&](MvSlots &dst, MvItem &it) {
        // past the last item: an item of no rows, whose slots all read one
        // block (not used), so the prefetch beyond the end costs one line
        it = mv_item<EPI>(a, min(ltile, ntiles - 1), ltile < ntiles ? lchunk : 0, nb);
        it.nloc = ltile < ntiles ? it.nloc : 0;
        mv_load<EPI, QT, D16>(dst, a, it, nb, lane);
        next_item(ltile, lchunk);
    };
    MvSlots S[MV_DEPTH];
    MvItem I[MV_DEPTH];
    // touches: item i + MV_TOUCH is touched in item i's step, into slot
    // i % MV_TOUCH, whose value (item i's touch, older than item i's own
    // loads, so already back when item i's dots have run) is folded into sink
    // first; the prologue touches items 1 .. MV_TOUCH - 1
    int tv[MV_TOUCH > 1 ? MV_TOUCH : 1] = {};
    int sink = 0, ttile = gw, tchunk = 0;
    auto touch_item = [&]() -> int {
        MvItem it = mv_item<EPI>(a, min(ttile, ntiles - 1), ttile < ntiles ? tchunk : 0, nb);
        next_item(ttile, tchunk);
        return a.touch ? mv_touch<EPI, QT, D16>(a, it, nb, lane) : 0;
    };
    auto prime_touch = [&]() {
        if (MV_TOUCH > 1) {
            next_item(ttile, tchunk);
#pragma unroll
            for (int t = 1; t < MV_TOUCH; t++) tv[t] = touch_item();
        }
    };
    if (a.xq && K <= MV_XQ_MAX) {
        // a quantized activation (just written by the previous launch, so
        // not yet in this die's L2): it is read and stored to LDS before the
        // weight stream starts, so it never queues behind it
        int4 xv[MV_XQ_MAX / 16 / MV_THREADS];
        float xdv[MV_XQ_MAX / 32 / MV_THREADS];
#pragma unroll
        for (int k = 0; k < MV_XQ_MAX / 16 / MV_THREADS; k++)
            xv[k] = ((const int4 *)a.xq)[min(tid + k * MV_THREADS, K / 16 - 1)];
#pragma unroll
        for (int k = 0; k < MV_XQ_MAX / 32 / MV_THREADS; k++) xdv[k] = a.xd[min(tid + k * MV_THREADS, nb - 1)];
#pragma unroll
        for (int k = 0; k < MV_XQ_MAX / 16 / MV_THREADS; k++)
            if (tid + k * MV_THREADS < K / 16) ((int4 *)xs)[tid + k * MV_THREADS] = xv[k];
#pragma unroll
        for (int k = 0; k < MV_XQ_MAX / 32 / MV_THREADS; k++)
            if (tid + k * MV_THREADS < nb) xds[tid + k * MV_THREADS] = xdv[k];
#pragma unroll
        for (int d = 0; d < MV_DEPTH - 1; d++) load_item(S[d], I[d]);
        prime_touch();
    } else if (!a.xq && !a.nw && K <= MV_XF_PLAIN_MAX) {
        // a float activation without a norm (ao before wo, h before w2), in
        // passes of MV_XF_PASS floats held in registers: the first pass's
        // loads go out first, then the first item's weight loads, and the
        // first quantization waits on the activation alone; later passes
        // (h of more than MV_XF_PASS) follow
        // thread t takes the 16 values base + 16 t .. + 15, half of a
        // 32-block (kr_quant16)
        static_assert(MV_XF_PASS == 16 * MV_THREADS, "a pass is one half-block per thread");
        // Two passes' registers in turn: a pass's loads go out before the
        // pass ahead of it is quantized (h of 14,336 floats: four load round
        // trips in series otherwise).
        float4 xa[4], xb[4];
        auto pass_load = [&](float4 (&xv)[4], int base) {
            const int i = min(base + 16 * tid, K - 16);
#pragma unroll
            for (int k = 0; k < 4; k++) xv[k] = *(const float4 *)(a.xf + i + 4 * k);
        };
        auto pass_quant = [&](const float4 (&xv)[4], int base) {
            const int i = base + 16 * tid;   // K % 32 == 0: both halves of a block are in or out
            if (i < K) kr_quant16(xv, i, xs, xds);
        };
        pass_load(xa, 0);
        if (MV_XF_PASS < K) pass_load(xb, MV_XF_PASS);
#pragma unroll
        for (int d = 0; d < MV_DEPTH - 1; d++) load_item(S[d], I[d]);
        prime_touch();
        pass_quant(xa, 0);
        for (int base = MV_XF_PASS; base < K; base += 2 * MV_XF_PASS) {
            if (base + MV_XF_PASS < K) pass_load(xa, base + MV_XF_PASS);
            pass_quant(xb, base);
            if (base + MV_XF_PASS < K) {
                if (base + 2 * MV_XF_PASS < K) pass_load(xb, base + 2 * MV_XF_PASS);
                pass_quant(xa, base + MV_XF_PASS);
            }
        }
    } else if (!a.xq && K <= MV_XF_MAX) {
        // a float activation (normalized first when nw is set), held in
        // registers: its loads go out before the weight loads; the squares
        // and the quantization read the registers
        // thread t holds the 16 values 16 t .. 16 t + 15 (half of a
        // 32-block, kr_quant16) and their norm weights
        static_assert(MV_XF_MAX == 16 * MV_THREADS, "one half-block per thread");
        constexpr int XV = 4;
        float4 xv[XV], wv[XV];
        const int i0 = 16 * tid;
        const bool live = i0 < K;   // K % 32 == 0: both halves of a block are live or not
        {
            const int i = min(i0, K - 16);
#pragma unroll
            for (int k = 0; k < XV; k++) xv[k] = *(const float4 *)(a.xf + i + 4 * k);
        }
        float inv = 1.0f;
        if (a.nw) {
            // the squares wait on x alone; the weight stream then runs under
            // the ordered sum
            const int sh = sc_log_len(K);
            if (live) {
#pragma unroll
                for (int k = 0; k < XV; k++)   // 16 | chunk length: the 16 terms are contiguous in sq
                    *(float4 *)(sq + sc_at(i0, sh) + 4 * k) =
                        make_float4(kr_fmul(xv[k].x, xv[k].x), kr_fmul(xv[k].y, xv[k].y), kr_fmul(xv[k].z, xv[k].z),
                                    kr_fmul(xv[k].w, xv[k].w));
            }
            // the norm weights go out once x is in (every workgroup reads x
            // at once; the weights, needed only by the quantization, return
            // under the ordered sum), ahead of the weight stream, whose
            // loads return after them
            {
                const int i = min(i0, K - 16);
#pragma unroll
                for (int k = 0; k < XV; k++) wv[k] = *(const float4 *)(a.nw + i + 4 * k);
            }
#pragma unroll
            for (int d = 0; d < MV_DEPTH - 1; d++) load_item(S[d], I[d]);
            prime_touch();
            __syncthreads();
            unsigned char *sl = (unsigned char *)(sq + sc_terms_cap(K));
            float ss;
            if constexpr (SH) ss = kr_short_sum(sq, K, sl);
            else ss = kr_spec_sum<MV_THREADS>(sq, K, sl);
            inv = kr_fdiv(1.0f, kr_fsqrt(kr_fadd(kr_fdiv(ss, (float)K), a.eps)));
        }
        if (live) {
            float4 o[XV];
#pragma unroll
            for (int k = 0; k < XV; k++) o[k] = a.nw ? kr_norm4(xv[k], inv, wv[k]) : xv[k];
            kr_quant16(o, i0, xs, xds);
            if (a.keep_xb && blockIdx.x == 0) {
#pragma unroll
                for (int k = 0; k < XV; k++) *(float4 *)(a.keep_xb + i0 + 4 * k) = o[k];
            }
        }
        if (!a.nw) {
#pragma unroll
            for (int d = 0; d < MV_DEPTH - 1; d++) load_item(S[d], I[d]);
            prime_touch();
        }
    } else {
#pragma unroll
        for (int d = 0; d < MV_DEPTH - 1; d++) load_item(S[d], I[d]);
        prime_touch();
        if (a.xq) {
            for (int i = tid; i < K / 16; i += MV_THREADS) ((int4 *)xs)[i] = ((const int4 *)a.xq)[i];
            for (int i = tid; i < nb; i += MV_THREADS) xds[i] = a.xd[i];
        } else if (a.nw) {
            for (int i = 4 * tid; i < K; i += 4 * MV_THREADS) {
                const float4 v = *(const float4 *)(a.xf + i);
                *(float4 *)(sq + sc_at(i, sc_log_len(K))) = make_float4(kr_fmul(v.x, v.x), kr_fmul(v.y, v.y), kr_fmul(v.z, v.z),
                                                  kr_fmul(v.w, v.w));
            }
            __syncthreads();
            const float ss = kr_spec_sum<MV_THREADS>(sq, K, (unsigned char *)(sq + sc_terms_cap(K)));
            const float inv = kr_fdiv(1.0f, kr_fsqrt(kr_fadd(kr_fdiv(ss, (float)K), a.eps)));
            quantize_to_lds(a.xf, K, xs, xds, a.nw, inv, blockIdx.x == 0 ? a.keep_xb : nullptr);
        } else {
            quantize_to_lds(a.xf, K, xs, xds);
        }
    }
    __syncthreads();
    if (a.keep_xq && blockIdx.x == 0) {   // the prologue's Q8_0 of x, from LDS
        for (int i = tid; i < K / 16; i += MV_THREADS) ((int4 *)a.keep_xq)[i] = ((const int4 *)xs)[i];
        for (int i = tid; i < nb; i += MV_THREADS) a.keep_xd[i] = xds[i];
    }

    float acc = 0.0f;   // row sum of lane < nloc
    // one item (step P4 of an unrolled group of 2 or 4): S[P4 % MV_DEPTH] holds it;
    // the slot before receives the loads MV_DEPTH - 1 ahead
    auto step = [&](auto P4_) -> bool {
        constexpr int P4 = decltype(P4_)::value, P = P4 % MV_DEPTH;
        const MvItem cur = I[P];
        load_item(S[(P + MV_DEPTH - 1) % MV_DEPTH], I[(P + MV_DEPTH - 1) % MV_DEPTH]);
        int ntile = tile, nchunk = chunk;
        next_item(ntile, nchunk);
        // the epilogue's inputs for this tile's rows, read before this
        // step's item loads go out, so the epilogue waits on them alone;
        // every lane reads (a clamped row; a missing bias reads the RoPE
        // table and is not used): no load sits in a branch
        float ep0 = 0.0f, ep1 = 0.0f, ep2 = 0.0f;
        {
            const int row = cur.row0 + min(lane, cur.nr - 1);
            if (EPI == EPI_ADD) ep0 = pick3(cur.mi, a.y[0], a.y[1], a.y[2])[row];
            if (EPI == EPI_QKV) {
                const float *bias = pick3(cur.mi, a.bias[0], a.bias[1], a.bias[2]);
                ep0 = *(bias ? bias + row : a.rope_cos);
                const int hd = a.head_dim, h2 = hd >> 1, j = row % hd;
                ep1 = a.rope_cos[(size_t)pos * h2 + (j >> 1)];
                ep2 = a.rope_sin[(size_t)pos * h2 + (j >> 1)];
            }
        }

        {
            int lr = lane / cur.nbc, b = lane - lr * cur.nbc;
            const int sr = 64 / cur.nbc, sb = 64 - sr * cur.nbc;
            const int n = cur.nloc * cur.nbc;
#pragma unroll
            for (int k = 0; k < MV_NPT; k++) {
                if (lane + k * 64 < n) {
                    const int bb = cur.c0 + b;
                    const int sdot = QT != QT_MIXED ? block_dot<QT>(S[P].w0[k], S[P].w1[k], xs + bb * 32)
                                     : qt_is_q8<QT>(pick3(cur.mi, a.m[0].type, a.m[1].type, a.m[2].type))
                                         ? block_dot<ML_Q8_0>(S[P].w0[k], S[P].w1[k], xs + bb * 32)
                                         : block_dot<ML_Q4_0>(S[P].w0[k], S[P].w1[k], xs + bb * 32);
                    const float sc = D16 ? kr_h2f((uint16_t)S[P].wd[k]) : __uint_as_float(S[P].wd[k]);
                    T[lr * ts + b] = kr_fmul(kr_fmul((float)sdot, sc), xds[bb]);
                }
                b += sb;
                lr += sr;
                if (b >= cur.nbc) { b -= cur.nbc; lr++; }
            }
        }
        if (MV_TOUCH > 1) {
            constexpr int TS = P4 % (MV_TOUCH > 1 ? MV_TOUCH : 1);
            sink ^= tv[TS];
            tv[TS] = touch_item();
        }
        kr_wave_sync();
        if (lane < cur.nloc) {
            if (chunk == 0) acc = 0.0f;
            const float *p = T + lane * ts;
            int j = 0;
            for (; j + 32 <= cur.nbc; j += 32) {
                float4 r[8];
#pragma unroll
                for (int k = 0; k < 8; k++) r[k] = *(const float4 *)(p + j + 4 * k);
#pragma unroll
                for (int k = 0; k < 8; k++) {
                    acc = kr_fadd(acc, r[k].x);
                    acc = kr_fadd(acc, r[k].y);
                    acc = kr_fadd(acc, r[k].z);
                    acc = kr_fadd(acc, r[k].w);
                }
            }
            for (; j + 4 <= cur.nbc; j += 4) {   // under 32 left (a 896-wide row's 28): 16-byte reads
                const float4 r = *(const float4 *)(p + j);
                acc = kr_fadd(acc, r.x);
                acc = kr_fadd(acc, r.y);
                acc = kr_fadd(acc, r.z);
                acc = kr_fadd(acc, r.w);
            }
            for (; j < cur.nbc; j++) acc = kr_fadd(acc, p[j]);
        }
        if (nchunk == 0) {   // the tile's last chunk: epilogue
            if (lane < cur.nloc) sums[lane] = acc;
            kr_wave_sync();
            const int mi = cur.mi, row0 = cur.row0, nr = cur.nr;
            if (EPI == EPI_STORE) {
                if (lane < nr) pick3(mi, a.y[0], a.y[1], a.y[2])[row0 + lane] = sums[lane];
            } else if (EPI == EPI_ADD) {
                if (lane < nr) {
                    pick3(mi, a.y[0], a.y[1], a.y[2])[row0 + lane] = kr_fadd(ep0, sums[lane]);
                    if (a.keep) a.keep[row0 + lane] = sums[lane];
                }
            } else if (EPI == EPI_QKV) {
                // bias (model/transformer.c:276-277), then RoPE on q and k
                // (k_scalar.c:79-94: pairs 2i, 2i+1 of each head, unfused)
                const float *bias = pick3(mi, a.bias[0], a.bias[1], a.bias[2]);
                float v = 0.0f;
                if (lane < nr) {
                    v = sums[lane];
                    if (bias) v = kr_fadd(v, ep0);
                }
                kr_wave_sync();
                if (lane < nr) sums[lane] = v;
                kr_wave_sync();
                if (lane < nr) {
                    const int row = row0 + lane;
                    float o = v;
                    if (mi < 2) {
                        const float c = ep1, sn = ep2;
                        const float pa = sums[lane & ~1], pb = sums[lane | 1];
                        o = (lane & 1) == 0 ? kr_fsub(kr_fmul(pa, c), kr_fmul(pb, sn))
                                            : kr_fadd(kr_fmul(pa, sn), kr_fmul(pb, c));
                    }
                    if (mi == 0) a.y[0][row] = o;
                    else if (a.kv16)   // store_kv's rounding (model/transformer.c:195-197)
                        ((uint16_t *)pick3(mi, a.y[0], a.y[1], a.y[2]))[(size_t)pos * a.ld_cache + row] = kr_f2h(o);
                    else pick3(mi, a.y[0], a.y[1], a.y[2])[(size_t)pos * a.ld_cache + row] = o;
                }
            } else if (EPI == EPI_SWIGLU) {
                // g = g / (1 + expf(-g)) * u (k_scalar.c:96-98)
                if (lane < nr) {
                    const float h1 = sums[lane], h3 = sums[nr + lane];
                    a.y[0][row0 + lane] = kr_fmul(kr_fdiv(h1, kr_fadd(1.0f, kr_expf(-h1))), h3);
                    if (a.keep) a.keep[row0 + lane] = h3;
                }
            }
        }
        tile = ntile;
        chunk = nchunk;
        return tile < ntiles;
    };
    static_assert(MV_DEPTH == 2, "the step loop is unrolled by 2 or 4");
    static_assert(MV_TOUCH == 1 || MV_TOUCH == 2 || MV_TOUCH == 4, "touch slots divide the unrolled 4");
    if (gw >= ntiles) return;   // a wave with no tile (after the workgroup's one barrier)
    if (MV_TOUCH == 4) {
        while (step(std::integral_constant<int, 0>()) && step(std::integral_constant<int, 1>()) &&
               step(std::integral_constant<int, 2>()) && step(std::integral_constant<int, 3>())) {
        }
    } else {
        while (step(std::integral_constant<int, 0>()) && step(std::integral_constant<int, 1>())) {
        }
    }
    if (MV_TOUCH > 1) {
        // keeps the touches (their values are never otherwise used)
#pragma unroll
        for (int t = 0; t < MV_TOUCH; t++) sink ^= tv[t];
        if (sink == 0x5bd1e995 && K < 0) a.y[0][0] = 0.0f;
    }
}

}  // namespace
