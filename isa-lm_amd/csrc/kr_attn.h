// What the decode and the batched attention launches share (kr_attn.hip,
// kr_attn_prefill.hip): the cache view, the per-token score kernels and the
// per-row softmax.
#pragma once
#include <algorithm>
#include "kr_internal.h"
#include "kr_numerics.h"
#include "kr_chain.h"

// The cache a launch reads (ml_kv_layer, ops/ops.h:16-22, of one layer): K
// and V rows [max_seq][kv_dim] of floats, halves or int8, and for the Q8
// cache the row scales kd, vd [max_seq][n_kv_heads] (model/transformer.c:169-180).
enum { KV_F32 = 0, KV_F16 = 1, KV_Q8 = 2 };
struct KvView {
    const void *k, *v;
    const float *kd, *vd;
    int n_kv;
    const float *ks, *vs;   // Q8 decode: row *pos's K and V, still to be stored (else null)
};

// kr_attn_prefill.hip: the attention of ntok > 1 positions *pos + t over a
// cache of type kt (KV_*); shapes checked by the caller
void kr_attn_prefill(int kt, float *ao, float *att, const float *q, const KvView &kv, int n_heads, int n_kv_heads,
                     int head_dim, int max_seq, int window, float scale, const int *pos, int ntok, int max_pos,
                     float cap);

namespace {

// ---- attention (F32 cache) ----
//
// Per layer and position (ops/ops.c:124-155): for query head h (KV head
// h / group), s_t = (sum_i q_i k_t,i in index order) * scale
// (k_scalar.c:111-117), softmax over t (k_scalar.c:66-77: max, expf(x - max),
// the sum in position order, then x * (1 / sum)), and out_i = 0,
// out_i += a_t v_t,i in position order (k_scalar.c:119-122). The ordered
// chains run from LDS; the loads feeding them are wide and parallel.

constexpr int AT_T = 64;          // positions per score tile of a batched (prefill) launch
constexpr int AT_TD = 16;         // of a decode launch: more, smaller tiles hide the K loads better
constexpr int AT_THREADS = 256;

// positions attended by token blockIdx.z of the launch, at position *pos_p + blockIdx.z
__device__ __forceinline__ void attn_range(const int *pos_p, int window, int *first, int *n) {
    const int pos = *pos_p + (int)blockIdx.z;
    *first = window && pos >= window ? pos + 1 - window : 0;
    *n = pos + 1 - *first;
}

// Where a windowed token's scores start in its row of the scratch: a batched
// launch (prefill) stores position p's score at index p, so that the tokens
// of a block, whose windows start one position apart, share position tiles
// and aligned reads; a decode launch packs the row from its first attended
// position. Without a window both are position 0. (BATCH is a template
// argument: reading it from the launch's grid cost the decode kernels 0.7 us
// of the 41 us an 8B-shape attention block takes.)
template <bool BATCH> __device__ __forceinline__ int attn_row0(int first) { return BATCH ? first : 0; }
// the first position token position pos attends
__device__ __forceinline__ int attn_first(int pos, int window) { return window && pos >= window ? pos + 1 - window : 0; }

// 4 consecutive cache elements: the registers as loaded, and widened to
// floats (halves exactly, k_scalar.c:124-135; int8 to its value, :148-155)
template <int KT> struct Kv4;
template <> struct Kv4<KV_F32> {
    using T = float4;
    static constexpr int REGS = 4;
    __device__ static T load(const void *p, size_t i) { return *(const float4 *)((const float *)p + i); }
    __device__ static float4 wide(T v) { return v; }
};
template <> struct Kv4<KV_F16> {
    using T = uint2;
    static constexpr int REGS = 2;
    __device__ static T load(const void *p, size_t i) { return *(const uint2 *)((const uint16_t *)p + i); }
    __device__ static float4 wide(T v) {
        return make_float4(kr_h2f((uint16_t)v.x), kr_h2f((uint16_t)(v.x >> 16)), kr_h2f((uint16_t)v.y),
                           kr_h2f((uint16_t)(v.y >> 16)));
    }
};
template <> struct Kv4<KV_Q8> {
    using T = int;
    static constexpr int REGS = 1;
    __device__ static T load(const void *p, size_t i) { return *(const int *)((const int8_t *)p + i); }
    __device__ static float4 wide(T v) {
        return make_float4((float)(int8_t)v, (float)(int8_t)(v >> 8), (float)(int8_t)(v >> 16), (float)(v >> 24));
    }
};

// Scores of one KV head's query heads for TT positions. The K tile is staged
// in LDS as floats (F16 rows widened exactly, k_scalar.c:124-129), rows hd + 4
// floats apart so that the 16-byte reads of 8 consecutive lanes cover all
// banks once; thread (t, j) computes heads j, j + 4, ... of the group for
// position t, adding the products in index order.
template <int KT, int TT, bool BATCH>
__device__ __forceinline__ void attn_scores(float *att, const float *q, const KvView kv, int group, int hd, int kv_dim,
                                            int max_seq, int window, float scale, const int *pos_p) {
    extern __shared__ __align__(16) float at_smem[];
    int first, n;
    attn_range(pos_p, window, &first, &n);
    att += (size_t)blockIdx.z * gridDim.x * group * max_seq + attn_row0<BATCH>(first);   // token z: [n_heads][max_seq]
    q += (size_t)blockIdx.z * gridDim.x * group * hd;
    const int g = blockIdx.x, t0 = blockIdx.y * TT, tid = threadIdx.x;
    if (t0 >= n) return;
    const int nt = min(TT, n - t0), ks = hd + 4, h4 = hd / 4;
    float *qs = at_smem, *kt = at_smem + group * hd;
    const float4 *qg = (const float4 *)(q + (size_t)g * group * hd);
    for (int i = tid; i < group * h4; i += AT_THREADS) ((float4 *)qs)[i] = qg[i];
    for (int e = tid; e < nt * h4; e += AT_THREADS) {
        const int r = e / h4, c = e - r * h4;
        *(float4 *)(kt + r * ks + 4 * c) =
            Kv4<KT>::wide(Kv4<KT>::load(kv.k, (size_t)(first + t0 + r) * kv_dim + (size_t)g * hd + 4 * c));
    }
    __syncthreads();
    const int t = tid % TT;
    if (t >= nt) return;
    const float *kr = kt + t * ks;
    for (int j = tid / TT; j < group; j += AT_THREADS / TT) {
        const float *qh = qs + j * hd;
        float acc = 0.0f;
#pragma unroll 4
        for (int i = 0; i < hd; i += 4) {
            const float4 a = *(const float4 *)(qh + i), b = *(const float4 *)(kr + i);
            acc = kr_fadd(acc, kr_fmul(a.x, b.x));
            acc = kr_fadd(acc, kr_fmul(a.y, b.y));
            acc = kr_fadd(acc, kr_fmul(a.z, b.z));
            acc = kr_fadd(acc, kr_fmul(a.w, b.w));
        }
        att[(size_t)(g * group + j) * max_seq + t0 + t] = kr_fmul(acc, scale);
    }
}

// the F32 cache (its own argument list: the view is built on the device)
template <int TT, bool BATCH = false>
__global__ void __launch_bounds__(AT_THREADS) k_attn_scores(float *att, const float *q, const float *kc, int group,
                                                            int hd, int kv_dim, int max_seq, int window, float scale,
                                                            const int *pos_p) {
    const KvView kv = { kc, nullptr, nullptr, nullptr, 0 };
    attn_scores<KV_F32, TT, BATCH>(att, q, kv, group, hd, kv_dim, max_seq, window, scale, pos_p);
}

template <int KT, int TT, bool BATCH = false>
__global__ void __launch_bounds__(AT_THREADS) k_attn_scores_kv(float *att, const float *q, const KvView kv, int group,
                                                               int hd, int kv_dim, int max_seq, int window, float scale,
                                                               const int *pos_p) {
    attn_scores<KT, TT, BATCH>(att, q, kv, group, hd, kv_dim, max_seq, window, scale, pos_p);
}

// One query head of hd floats as the Q8 rule does it for the score
// (ops/ops.c:81-96): the max |x| from 0, one scale for the head, each value
// trunc(x * 127 / max + copysign(0.5, x)); a head of zeros (max below the
// rule's tiny) has scale 0 and zero quants. One wave; lane 0 writes the scale.
__device__ __forceinline__ void q8_head(const float *x, int hd, int8_t *dst, float *dd, int lane) {
    float m = 0.0f;
    for (int i = lane; i < hd; i += 64) m = fmaxf(m, fabsf(x[i]));
    for (int o = 32; o >= 1; o >>= 1) m = fmaxf(m, __shfl_xor(m, o));
    const bool zero = m < KR_QUANT_TINY;
    const float id = zero ? 0.0f : kr_fdiv(127.0f, m);
    for (int i = lane; i < hd; i += 64) dst[i] = zero ? (int8_t)0 : (int8_t)kr_q8_elem(x[i], id);
    if (lane == 0) *dd = zero ? 0.0f : kr_fdiv(m, 127.0f);
}

// Scores over the Q8 cache (ops/ops.c:171-173, k_scalar.c:137-146): each query
// head of the group quantized with one scale (ops/ops.c:81-96; every
// workgroup quantizes its group's heads itself, the same bits), then per
// position the exact int32 dot of the int8 rows (v_dot4) and
// ((float)sum * (dq * scale)) * dk_t. K rows are staged in LDS with a stride
// of hd + 4 bytes (33 words for hd 128: the lanes of a wave spread over the
// banks).
template <bool BATCH = false>
__global__ void __launch_bounds__(AT_THREADS) k_attn_scores_q8(float *att, const float *q, const KvView kv, int group,
                                                               int hd, int kv_dim, int max_seq, int window, float scale,
                                                               const int *pos_p) {
    extern __shared__ __align__(16) float at_smem[];
    int first, n;
    attn_range(pos_p, window, &first, &n);
    att += (size_t)blockIdx.z * gridDim.x * group * max_seq + attn_row0<BATCH>(first);
    q += (size_t)blockIdx.z * gridDim.x * group * hd;
    const int g = blockIdx.x, t0 = blockIdx.y * AT_T, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    if (t0 >= n) return;
    const int nt = min(AT_T, n - t0), ks = hd + 4;
    float *qd = at_smem;                            // [16] query scales
    int8_t *qs = (int8_t *)(at_smem + 16);          // [group][hd]
    int8_t *kt = qs + (group * hd + 15) / 16 * 16;  // [AT_T][ks]
    for (int j = wave; j < group; j += AT_THREADS / 64) q8_head(q + (size_t)(g * group + j) * hd, hd, qs + j * hd, qd + j, lane);
    // store_kv folded into decode (model/transformer.c:198-203): the tile
    // holding the current position quantizes its KV head's K row (wave 0,
    // straight into the tile as well) and V row (wave 1) into the cache
    __shared__ float fresh_dk;
    const bool fresh = kv.ks && t0 + nt == n;
    if (fresh && wave < 2) {
        const float *x = (wave ? kv.vs : kv.ks) + (size_t)g * hd;
        float m = 0.0f;
        for (int i = lane; i < hd; i += 64) m = fmaxf(m, fabsf(x[i]));
        for (int o = 32; o >= 1; o >>= 1) m = fmaxf(m, __shfl_xor(m, o));
        const bool zero = m < KR_QUANT_TINY;
        const float id = zero ? 0.0f : kr_fdiv(127.0f, m), d = zero ? 0.0f : kr_fdiv(m, 127.0f);
        const size_t row = (size_t)(first + n - 1);
        int8_t *dst = (int8_t *)(wave ? kv.v : kv.k) + row * kv_dim + (size_t)g * hd;
        for (int i = lane; i < hd; i += 64) {
            const int8_t qv = zero ? (int8_t)0 : (int8_t)kr_q8_elem(x[i], id);
            dst[i] = qv;
            if (wave == 0) kt[(nt - 1) * ks + i] = qv;
        }
        if (lane == 0) {
            ((float *)(wave ? kv.vd : kv.kd))[row * kv.n_kv + g] = d;
            if (wave == 0) fresh_dk = d;
        }
    }
    const int h4 = hd / 4;
    for (int e = tid; e < nt * h4; e += AT_THREADS) {
        const int r = e / h4, c = e - r * h4;
        if (fresh && r == nt - 1) continue;   // written above
        *(int *)(kt + r * ks + 4 * c) =
            *(const int *)((const int8_t *)kv.k + (size_t)(first + t0 + r) * kv_dim + (size_t)g * hd + 4 * c);
    }
    __syncthreads();
    const int t = tid % AT_T;
    if (t >= nt) return;
    const int8_t *kr = kt + t * ks;
    const float dk = fresh && t == nt - 1 ? fresh_dk : kv.kd[(size_t)(first + t0 + t) * kv.n_kv + g];
    for (int j = tid / AT_T; j < group; j += AT_THREADS / AT_T) {
        const int8_t *qh = qs + j * hd;
        int sum = 0;
        for (int i = 0; i < hd; i += 4) sum = kr_dot4(*(const int *)(qh + i), *(const int *)(kr + i), sum);
        const float c = kr_fmul(qd[j], scale);
        att[(size_t)(g * group + j) * max_seq + t0 + t] = kr_fmul(kr_fmul((float)sum, c), dk);
    }
}

// Softmax of one head's n scores in place (k_scalar.c:66-77): the max, the
// exponentials x - max, their ordered sum (kr_spec_sum: the sequential
// loop's bits), x * (1 / sum). Up to AT_CHUNK scores stay in registers
// between one batched read and one write (every load issued at once, from an
// index clamped into the row); longer rows go AT_CHUNK at a time through LDS,
// the sum continuing from chunk to chunk.
// NT threads a row, CH scores of it in registers at once: the decode launch
// spreads its loads, exponentials and stores over 1024 threads; prefill rows
// of up to 4096 scores take 256 (the ordered sum needs 4 waves, and a small
// workgroup lets 8 rows share a CU's LDS and SIMDs).
constexpr int SMX_THREADS = 1024, AT_CHUNK = 8192;   // the decode launch
template <int NT, int CH, bool LEAN = false, bool BATCH = LEAN>
__global__ void __launch_bounds__(NT) k_attn_softmax(float *att, int max_seq, int window, const int *pos_p) {
    constexpr int SMX_THREADS = NT, AT_CHUNK = CH, AT_V = CH / NT;
    __shared__ __align__(16) float es[sc_terms_cap(AT_CHUNK)];
    __shared__ __align__(16) unsigned char scr[sc_lds_bytes(AT_CHUNK, SMX_THREADS)];
    __shared__ float red[SMX_THREADS / 64];
    __shared__ uint64_t xtab[32];   // expf's table
    int first, n;
    attn_range(pos_p, window, &first, &n);
    float *a = att + ((size_t)blockIdx.z * gridDim.x + blockIdx.x) * max_seq + attn_row0<BATCH>(first);
    const int tid = threadIdx.x;
    if (tid < 32) xtab[tid] = kr_exp2_tab[tid];
    const bool fits = n <= AT_CHUNK;
    float v[AT_V];
    float m = -INFINITY;
    if (fits) {
        // slots past the row's end are skipped (a uniform test); the last
        // live slot's index is clamped: repeats change no max
#pragma unroll
        for (int k = 0; k < AT_V; k++)
            if (k * SMX_THREADS < n) v[k] = a[min(k * SMX_THREADS + tid, n - 1)];
#pragma unroll
        for (int k = 0; k < AT_V; k++)
            if (k * SMX_THREADS < n) m = fmaxf(m, v[k]);
    } else {
        for (int t = tid; t < n; t += SMX_THREADS) m = fmaxf(m, a[t]);
    }
    for (int o = 32; o >= 1; o >>= 1) m = fmaxf(m, __shfl_xor(m, o));
    if ((tid & 63) == 0) red[tid >> 6] = m;
    __syncthreads();
    float mx = red[0];
    for (int k = 1; k < SMX_THREADS / 64; k++) mx = fmaxf(mx, red[k]);
    if (mx == -INFINITY) {   // every score -inf: the scalar loop's 1/n
        for (int t = tid; t < n; t += SMX_THREADS) a[t] = kr_fdiv(1.0f, (float)n);
        return;
    }
    if (fits) {
        const int sh = sc_log_len(n);
#pragma unroll
        for (int k = 0; k < AT_V; k++) {
            if (k * SMX_THREADS >= n) break;   // the rest of the slots are clamped repeats
            const int t = k * SMX_THREADS + tid;
            v[k] = kr_expf_tab(kr_fsub(v[k], mx), xtab);
            if (t < n) es[sc_at(t, sh)] = v[k];
        }
        __syncthreads();
        const float inv = kr_fdiv(1.0f, kr_spec_sum<SMX_THREADS, false, false, LEAN>(es, n, scr));
#pragma unroll
        for (int k = 0; k < AT_V; k++) {
            if (k * SMX_THREADS >= n) break;
            const int t = k * SMX_THREADS + tid;
            if (t < n) a[t] = kr_fmul(v[k], inv);
        }
        return;
    }
    float sum = 0.0f;
    for (int c0 = 0; c0 < n; c0 += AT_CHUNK) {
        const int cn = min(AT_CHUNK, n - c0), sh = sc_log_len(cn);
        for (int t = tid; t < cn; t += SMX_THREADS) {
            const float e = kr_expf_tab(kr_fsub(a[c0 + t], mx), xtab);
            es[sc_at(t, sh)] = e;
            a[c0 + t] = e;
        }
        __syncthreads();
        sum = kr_spec_sum<SMX_THREADS, false, false, LEAN>(es, cn, scr, sum);   // ends with a barrier: es is free again
    }
    const float inv = kr_fdiv(1.0f, sum);
    for (int t = tid; t < n; t += SMX_THREADS) a[t] = kr_fmul(a[t], inv);
}

__device__ __forceinline__ void kr_lds_order() { asm volatile("" ::: "memory"); }

// the per-token score kernels' LDS: the group's queries and a K tile of
// tt positions. F32/F16 tiles of wide heads (Gemma's 256) take AT_TD
// positions; the int8 Q8 tile fits at AT_T up to heads of 512 and more.
template <int KT> size_t attn_tile_lds(int group, int head_dim, int tt) {
    return KT == KV_Q8 ? 64 + (size_t)(group * head_dim + 15) / 16 * 16 + (size_t)tt * (head_dim + 4)
                       : sizeof(float) * ((size_t)group * head_dim + (size_t)tt * (head_dim + 4));
}
// the positions of such a tile, 0: none fits
template <int KT> int attn_tile(int group, int head_dim) {
    return attn_tile_lds<KT>(group, head_dim, AT_T) <= 64 * 1024                       ? AT_T
           : KT != KV_Q8 && attn_tile_lds<KT>(group, head_dim, AT_TD) <= 64 * 1024 ? AT_TD
                                                                                   : 0;
}

}   // namespace
