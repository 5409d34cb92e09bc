// Batched (prefill) attention over one layer's KV cache for gfx950: the
// scores, softmax and mix of many tokens at once (see kr_attn.hip's head
// comment; every float operation is the reference's, in its order). A code
// object of its own, which leaves the decode kernels' small.
#include <cmath>
#include "kr_attn.h"

namespace {

// Batched (prefill) scores over the F32 or F16 cache, a block of AT_TB tokens
// at a time (F16 rows widened exactly as the K tile is staged). The block's
// tiles start at the tile that holds its first token's first attended
// position; one K tile of AT_T positions, staged once in LDS, serves the
// whole block (the per-token kernel stages it again for every token). The queries of QB
// tokens at a time follow in LDS; thread (position t, head j) runs the QB
// chains of those tokens in one pass over the head's dims, one K read feeding
// them all (QB independent chains: the LDS latency hides under them). Each
// chain is the per-token kernel's: s = sum_i q_i k_i in index order, then
// * scale; a token stores only the positions it attends. HD: the head size
// when it is 64 or 128, else 0 (any). TP: positions per K tile, AT_T, or
// AT_T / 2 for heads whose AT_T-position tile and queries exceed 64 KB of
// LDS (Gemma's 256-wide heads).
//
// WIN, here and in the other batched kernels: with a window. A launch without one
// keeps the shorter loop conditions and its registers (through the windowed
// forms 6 heads of 48, 16 tokens at position 2000 took 70 us against 67, and the
// 1B shape's prompt step ran 1% slower).
constexpr int AT_TB = 16;
template <int HD, int QB, int KT, int TP, bool WIN>
__global__ void __launch_bounds__(AT_THREADS) k_attn_scores_blk(float *att, const float *q, const KvView kv, int group,
                                                                int hd_arg, int kv_dim, int max_seq, int window_arg,
                                                                float scale, const int *pos_p, int ntok) {
    const int window = WIN ? window_arg : 0;
    extern __shared__ __align__(16) float at_smem[];
    const int hd = HD ? HD : hd_arg;
    const int g = blockIdx.x, z0 = blockIdx.z * AT_TB, tid = threadIdx.x;
    const int pos0 = *pos_p, zn = min(AT_TB, ntok - z0);
    const int t0 = attn_first(pos0 + z0, window) / TP * TP + blockIdx.y * TP;
    const int nlast = pos0 + z0 + zn;   // positions the block's last token attends
    if (t0 >= nlast) return;
    const int nt = min(TP, nlast - t0), ks = hd + 4, h4 = hd / 4, n_heads = gridDim.x * group;
    float *kt = at_smem, *qs = at_smem + TP * ks;   // K tile [TP][ks]; queries [QB][group][hd]
    for (int e = tid; e < nt * h4; e += AT_THREADS) {
        const int r = e / h4, c = e - r * h4;
        *(float4 *)(kt + r * ks + 4 * c) =
            Kv4<KT>::wide(Kv4<KT>::load(kv.k, (size_t)(t0 + r) * kv_dim + (size_t)g * hd + 4 * c));
    }
    const int t = tid % TP, p = t0 + t;   // this thread's position
    const size_t qstride = (size_t)group * hd;   // floats between two tokens' queries in LDS
    for (int zb = 0; zb < zn; zb += QB) {
        const int qn = min(QB, zn - zb), gh4 = group * h4;
        __syncthreads();   // the last queries are read
        for (int e = tid; e < qn * gh4; e += AT_THREADS) {
            const int zz = e / gh4, r = e - zz * gh4;
            ((float4 *)qs)[e] = ((const float4 *)(q + (size_t)(z0 + zb + zz) * n_heads * hd + (size_t)g * group * hd))[r];
        }
        __syncthreads();
        if (t >= nt) continue;
        const float *kr = kt + t * ks;
        for (int j = tid / TP; j < group; j += AT_THREADS / TP) {
            // tokens zb + u, u < QB (slots past qn read an earlier block's
            // queries and are not stored)
            const float *qh = qs + (size_t)j * hd;
            float acc[QB];
#pragma unroll
            for (int u = 0; u < QB; u++) acc[u] = 0.0f;
#pragma unroll 2
            for (int i = 0; i < hd; i += 4) {
                const float4 b = *(const float4 *)(kr + i);
#pragma unroll
                for (int u = 0; u < QB; u++) {
                    const float4 a = *(const float4 *)(qh + u * qstride + i);
                    acc[u] = kr_fadd(acc[u], kr_fmul(a.x, b.x));
                    acc[u] = kr_fadd(acc[u], kr_fmul(a.y, b.y));
                    acc[u] = kr_fadd(acc[u], kr_fmul(a.z, b.z));
                    acc[u] = kr_fadd(acc[u], kr_fmul(a.w, b.w));
                }
            }
#pragma unroll
            for (int u = 0; u < QB; u++) {
                const int z = z0 + zb + u;
                if (u < qn && p <= pos0 + z && p >= attn_first(pos0 + z, window))
                    att[((size_t)z * n_heads + (size_t)g * group + j) * max_seq + p] = kr_fmul(acc[u], scale);
            }
        }
    }
}

// Batched (prefill) scores for heads of HD dims, blocked in registers: the
// rows (token z, query head j) of KV head g, numbered z * group + j, go to
// workgroups RB_R at a time, each over a chunk of pc tiles of RB_T positions
// (from the tile of its first row's first attended position). The workgroup
// stages its rows' queries in LDS once and each K tile in turn (F16 rows
// widened exactly), rows HS + 4 floats apart; lane (row group rg, position
// group pg) owns the scores of rows 4 rg .. 4 rg + 3 at positions pg + 16 k
// (k < 4): per 4 dims it reads 4 query and 4 K 16-byte values, which feed 64
// multiplies and 64 adds, each of its 16 sums s = sum_i q_i k_i in index
// order, then * scale, as in the per-token kernel. A row stores only the
// positions its token attends. The next tile's loads are in flight while a
// tile is summed. HS < HD (256-dim heads, whose tiles would fill the LDS):
// the queries and K are staged HS dims at a time, the sums carried along.
constexpr int RB_R = 64, RB_T = 64;   // rows of a register-blocked workgroup; positions of its tiles
constexpr int RB_PC = 8;             // K tiles per scores workgroup, at most
static bool rb_dims(int hd) { return hd == 48 || hd == 64 || hd == 80 || hd == 96 || hd == 128 || hd == 256; }
constexpr int RB_NT128 = 512;        // threads of the 128-dim heads' workgroups (4 outputs' rows a lane, LDS for 2
                                     // workgroups a CU: 4 waves a SIMD; 256 threads gave 2 and measured the same)
template <int HD, int KT, int NT, bool WIN, int HS = HD>
__global__ void __launch_bounds__(NT) k_attn_scores_rb(float *att, const float *q, const KvView kv, int group,
                                                       int kv_dim, int max_seq, int window_arg, float scale,
                                                       const int *pos_p, int ntok, int pc) {
    const int window = WIN ? window_arg : 0;
    constexpr int S = HS + 4;                     // LDS row stride (floats)
    constexpr int NS = HD / HS;                   // dim slices
    constexpr int NPG = NT / 16, PPL = RB_T / NPG;   // position groups; positions a lane (pg + NPG k)
    constexpr int NL = RB_T * HS / 4 / NT;        // 4-element K loads a thread stages per tile
    constexpr int NQL = RB_R * HS / 4 / NT;       // query float4 a thread stages
    static_assert(NS * HS == HD && NL * NT * 4 == RB_T * HS && NQL * NT * 4 == RB_R * HS, "whole loads");
    __shared__ __align__(16) float qs[RB_R * S];
    __shared__ __align__(16) float ks[RB_T * S];
    const int g = blockIdx.x, tid = threadIdx.x, pg = tid % NPG, rg = tid / NPG;
    const int nrow = ntok * group, R0 = blockIdx.y * RB_R;
    const int pos0 = *pos_p, n_heads = gridDim.x * group;
    const int nlast = pos0 + (min(R0 + RB_R, nrow) - 1) / group + 1;   // positions the block's last row attends
    const int p0 = attn_first(pos0 + R0 / group, window) / RB_T * RB_T + blockIdx.z * pc * RB_T;
    if (p0 >= nlast) return;
    const int ntl = min(pc, (nlast - p0 + RB_T - 1) / RB_T);
    auto q_load = [&](int u, int c0) {
        const int e = tid + NT * u, rr = e / (HS / 4), c4 = e % (HS / 4);
        const int R = min(R0 + rr, nrow - 1), z = R / group, j = R - z * group;
        return *(const float4 *)(q + ((size_t)z * n_heads + (size_t)g * group + j) * HD + c0 + 4 * c4);
    };
    auto q_store = [&](int u, float4 v) {
        const int e = tid + NT * u, rr = e / (HS / 4), c4 = e % (HS / 4);
        *(float4 *)(qs + rr * S + 4 * c4) = v;
    };
    typename Kv4<KT>::T kr[NL];
    float4 qr[NS > 1 ? NQL : 1];
    auto load = [&](int t0, int c0) {
#pragma unroll
        for (int u = 0; u < NL; u++) {
            const int e = tid + NT * u, p = e / (HS / 4), c4 = e % (HS / 4);
            kr[u] = Kv4<KT>::load(kv.k, (size_t)min(t0 + p, nlast - 1) * kv_dim + (size_t)g * HD + c0 + 4 * c4);
        }
        if constexpr (NS > 1) {
#pragma unroll
            for (int u = 0; u < NQL; u++) qr[u] = q_load(u, c0);
        }
    };
    if constexpr (NS == 1) {
#pragma unroll
        for (int u = 0; u < NQL; u++) q_store(u, q_load(u, 0));
    }
    int zr[4], lo[4];   // the tokens of the lane's rows (past the last row: -1) and the first positions they attend
#pragma unroll
    for (int r = 0; r < 4; r++) {
        const int R = R0 + 4 * rg + r;
        zr[r] = R < nrow ? R / group : -1;
        lo[r] = attn_first(pos0 + R / group, window);
    }
    load(p0, 0);
    for (int ti = 0; ti < ntl; ti++) {
        const int t0 = p0 + ti * RB_T;
        float acc[4][PPL];
#pragma unroll
        for (int r = 0; r < 4; r++)
#pragma unroll
            for (int k = 0; k < PPL; k++) acc[r][k] = 0.0f;
#pragma unroll 1
        for (int sl = 0; sl < NS; sl++) {
            __syncthreads();   // the last tile is read
#pragma unroll
            for (int u = 0; u < NL; u++) {
                const int e = tid + NT * u, p = e / (HS / 4), c4 = e % (HS / 4);
                *(float4 *)(ks + p * S + 4 * c4) = Kv4<KT>::wide(kr[u]);
            }
            if constexpr (NS > 1) {
#pragma unroll
                for (int u = 0; u < NQL; u++) q_store(u, qr[u]);
            }
            __syncthreads();
            if (sl + 1 < NS) load(t0, (sl + 1) * HS);
            else if (ti + 1 < ntl) load(t0 + RB_T, 0);
            const float *qp = qs + 4 * rg * S, *kp = ks + pg * S;
#pragma unroll 4
            for (int i = 0; i < HS; i += 4) {
                float4 a[4], b[PPL];
#pragma unroll
                for (int r = 0; r < 4; r++) a[r] = *(const float4 *)(qp + r * S + i);
#pragma unroll
                for (int k = 0; k < PPL; k++) b[k] = *(const float4 *)(kp + NPG * k * S + i);
#pragma unroll
                for (int r = 0; r < 4; r++)
#pragma unroll
                    for (int k = 0; k < PPL; k++) acc[r][k] = kr_fadd(acc[r][k], kr_fmul(a[r].x, b[k].x));
#pragma unroll
                for (int r = 0; r < 4; r++)
#pragma unroll
                    for (int k = 0; k < PPL; k++) acc[r][k] = kr_fadd(acc[r][k], kr_fmul(a[r].y, b[k].y));
#pragma unroll
                for (int r = 0; r < 4; r++)
#pragma unroll
                    for (int k = 0; k < PPL; k++) acc[r][k] = kr_fadd(acc[r][k], kr_fmul(a[r].z, b[k].z));
#pragma unroll
                for (int r = 0; r < 4; r++)
#pragma unroll
                    for (int k = 0; k < PPL; k++) acc[r][k] = kr_fadd(acc[r][k], kr_fmul(a[r].w, b[k].w));
            }
        }
#pragma unroll
        for (int r = 0; r < 4; r++) {
            if (zr[r] < 0) continue;
            const int R = R0 + 4 * rg + r, j = R - zr[r] * group;
            float *dst = att + ((size_t)zr[r] * n_heads + (size_t)g * group + j) * max_seq;
#pragma unroll
            for (int k = 0; k < PPL; k++) {
                const int p = t0 + pg + NPG * k;
                if (p <= pos0 + zr[r] && p >= lo[r]) dst[p] = kr_fmul(acc[r][k], scale);
            }
        }
    }
}

// Batched (prefill) scores over the Q8 cache, a block of AT_TB tokens at a
// time: the int8 K tile of AT_T positions and its row
// scales are staged once for the block; then, QB tokens at a time, the
// workgroup quantizes those tokens' query heads of its group into LDS
// (q8_head: the per-token kernel's bits) and thread (position t, head j)
// runs the QB exact int32 dots against its K row in one pass, each finished
// as in the per-token kernel: ((float)sum * (dq * scale)) * dk_t.
template <int QB, bool WIN>
__global__ void __launch_bounds__(AT_THREADS) k_attn_scores_blk_q8(float *att, const float *q, const KvView kv,
                                                                   int group, int hd, int kv_dim, int max_seq,
                                                                   int window_arg, float scale, const int *pos_p,
                                                                   int ntok) {
    const int window = WIN ? window_arg : 0;
    extern __shared__ __align__(16) float at_smem[];
    const int g = blockIdx.x, z0 = blockIdx.z * AT_TB, tid = threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6;
    const int pos0 = *pos_p, zn = min(AT_TB, ntok - z0);
    const int t0 = attn_first(pos0 + z0, window) / AT_T * AT_T + blockIdx.y * AT_T;
    const int nlast = pos0 + z0 + zn;   // positions the block's last token attends
    if (t0 >= nlast) return;
    const int nt = min(AT_T, nlast - t0), ks = hd + 4, n_heads = gridDim.x * group, h4 = hd / 4;
    float *dks = at_smem;                                   // [AT_T] K row scales
    float *qd = dks + AT_T;                                 // [QB][group] query head scales
    int8_t *kt = (int8_t *)(qd + (QB * group + 3) / 4 * 4);   // [AT_T][ks]
    int8_t *qs = kt + (AT_T * ks + 15) / 16 * 16;          // [QB][group][hd]
    for (int e = tid; e < nt * h4; e += AT_THREADS) {
        const int r = e / h4, c = e - r * h4;
        *(int *)(kt + r * ks + 4 * c) =
            *(const int *)((const int8_t *)kv.k + (size_t)(t0 + r) * kv_dim + (size_t)g * hd + 4 * c);
    }
    for (int r = tid; r < nt; r += AT_THREADS) dks[r] = kv.kd[(size_t)(t0 + r) * kv.n_kv + g];
    const int t = tid % AT_T, p = t0 + t;   // this thread's position
    for (int zb = 0; zb < zn; zb += QB) {
        const int qn = min(QB, zn - zb);
        __syncthreads();   // the last queries are read
        for (int h = wave; h < qn * group; h += AT_THREADS / 64) {
            const int zz = h / group, jj = h - zz * group;
            q8_head(q + ((size_t)(z0 + zb + zz) * n_heads + (size_t)g * group + jj) * hd, hd, qs + (size_t)h * hd,
                    qd + h, lane);
        }
        __syncthreads();
        if (t >= nt) continue;
        const int8_t *kr = kt + t * ks;
        const float dk = dks[t];
        for (int j = tid / AT_T; j < group; j += AT_THREADS / AT_T) {
            // tokens zb + u, u < QB (slots past qn hold an earlier block's
            // queries and are not stored)
            int acc[QB];
#pragma unroll
            for (int u = 0; u < QB; u++) acc[u] = 0;
            for (int i = 0; i < hd; i += 4) {
                const int k4 = *(const int *)(kr + i);
#pragma unroll
                for (int u = 0; u < QB; u++) acc[u] = kr_dot4(*(const int *)(qs + ((size_t)u * group + j) * hd + i), k4, acc[u]);
            }
#pragma unroll
            for (int u = 0; u < QB; u++) {
                const int z = z0 + zb + u;
                if (u < qn && p <= pos0 + z && p >= attn_first(pos0 + z, window)) {
                    const float c = kr_fmul(qd[u * group + j], scale);
                    att[((size_t)z * n_heads + (size_t)g * group + j) * max_seq + p] = kr_fmul(kr_fmul((float)acc[u], c), dk);
                }
            }
        }
    }
}

// Batched (prefill) softmax, one row per wave and RW rows per workgroup:
// rows r = token * n_heads + head of up to SM_WN = 4096 entries (the
// single-wave ordered sum's limit). Per row, as k_attn_softmax: the max,
// the exponentials x - max, their ordered sum (kr_spec_sum in single-wave
// mode), x * (1 / sum); an all -inf row becomes 1/n. The per-row kernel keeps
// three of its four waves idle in the ordered sum of rows this short; here
// every wave sums its own row. SV: register slots per lane (rows of at most
// 64 SV entries). The launch takes rows up to 2048 (32 slots: fewer
// registers, more rows in flight); longer rows measured faster on the
// per-row kernel with 256 threads (64 slots a lane here leave each CU two
// waves a SIMD, its LDS then holding 8 rows' terms).
constexpr int SM_WN = SC_CPW << SC_LOG_LMIN, SM_V = SM_WN / 64;
template <int RW, int SV = SM_V>
__global__ void __launch_bounds__(64 * RW) k_attn_softmax_rows(float *att, int n_heads, int max_seq, int window,
                                                               const int *pos_p, int nrows, int terms_cap,
                                                               int scr_bytes) {
    extern __shared__ __align__(16) unsigned char sm_lds[];
    __shared__ uint64_t xtab[32];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    if (threadIdx.x < 32) xtab[threadIdx.x] = kr_exp2_tab[threadIdx.x];
    __syncthreads();
    const int r = blockIdx.x * RW + wave;
    if (r >= nrows) return;
    const int z = r / n_heads, pos = *pos_p + z;
    const int first = attn_first(pos, window), n = pos + 1 - first;
    float *a = att + (size_t)r * max_seq + first;
    float *es = (float *)(sm_lds + (size_t)wave * (4 * terms_cap + scr_bytes));
    unsigned char *scr = (unsigned char *)(es + terms_cap);
    float v[SV];
    float m = -INFINITY;
#pragma unroll
    for (int k = 0; k < SV; k++)
        if (k * 64 < n) v[k] = a[min(k * 64 + lane, n - 1)];   // the last live slot clamped: repeats change no max
#pragma unroll
    for (int k = 0; k < SV; k++)
        if (k * 64 < n) m = fmaxf(m, v[k]);
    for (int o = 32; o >= 1; o >>= 1) m = fmaxf(m, __shfl_xor(m, o));
    if (m == -INFINITY) {   // every score -inf: the scalar loop's 1/n
        for (int t = lane; t < n; t += 64) a[t] = kr_fdiv(1.0f, (float)n);
        return;
    }
    const int sh = sc_log_len(n);
#pragma unroll
    for (int k = 0; k < SV; k++) {
        if (k * 64 >= n) break;
        const int t = k * 64 + lane;
        v[k] = kr_expf_tab(kr_fsub(v[k], m), xtab);
        if (t < n) es[sc_at(t, sh)] = v[k];
    }
    kr_wave_sync();
    const float inv = kr_fdiv(1.0f, kr_spec_sum<64, false, true>(es, n, scr));
#pragma unroll
    for (int k = 0; k < SV; k++) {
        if (k * 64 >= n) break;
        const int t = k * 64 + lane;
        if (t < n) a[t] = kr_fmul(v[k], inv);
    }
}


// The same for a batch of positions (prefill: one workgroup per position and
// head chunk, so throughput, not one chain's latency, is what counts), one wave
// per workgroup: lane = (head j of the group, dim d), DW = 64 / (group rounded up
// to a power of two). Each lane runs its ordered chain o += a_t * v_t,d
// (k_scalar.c:119-122). ao is written as floats (its quantization happens
// where it is consumed).
//
// The chain is the bound (one dependent add per position), so everything else
// is pipelined under it: tiles of MB_T positions of V and of the heads' weights
// are loaded MB_DEPTH tiles ahead into registers; tile t + 1 is staged into
// the other half of a double LDS buffer while tile t is read, V transposed
// ([dim][position]) so one 16-byte LDS read feeds 4 steps; the reads of each
// 16-step chunk are issued before the adds of the chunk before it. The
// workgroup is one wave, whose LDS operations execute in order, so LDS needs
// only compiler ordering (kr_lds_order), not barriers.
constexpr int MB_T = 64, MB_TS = MB_T + 4;   // positions per tile; padded LDS row

template <int DW, int KT>
__device__ __forceinline__ void attn_mix_batch(float *ao, const float *att, const KvView kv, int group, int hd,
                                               int kv_dim, int max_seq, int window, const int *pos_p) {
    constexpr int GP = 64 / DW;                    // head slots per wave
    constexpr int NV = MB_T * DW / 4 / 64;         // float4 of V per lane per tile
    constexpr int NA = (GP * MB_T / 4 + 63) / 64;  // float4 of weights per lane per tile
    constexpr int MB_DEPTH = NV + NA > 8 ? 2 : 4;  // tiles in flight (even: LDS halves alternate)
    __shared__ __align__(16) float vt[2][DW * MB_TS];
    constexpr int AW = GP * MB_T > NA * 256 ? GP * MB_T : NA * 256;   // padded: every lane stores
    __shared__ __align__(16) float aw[2][AW];
    int first, n;
    attn_range(pos_p, window, &first, &n);
    const int g = blockIdx.x, c0 = blockIdx.y * DW, lane = threadIdx.x;
    const int j = lane / DW, d = lane % DW;
    const size_t vb = (size_t)first * kv_dim + (size_t)g * hd + c0;   // element offset of V row `first`
    const size_t q_dim = (size_t)gridDim.x * group * hd;
    const int row0 = attn_row0<true>(first), alim = max_seq - 4 - row0;   // the row's last float4, from its first score
    const float *abase = att + ((size_t)blockIdx.z * gridDim.x * group + (size_t)g * group) * max_seq + row0;
    ao += blockIdx.z * q_dim;
    const int ntiles = (n + MB_T - 1) / MB_T;
    const int cw = min(DW, hd - c0);   // valid dims of the chunk (a multiple of 4)

    // Every load is unconditional from an address clamped into the live
    // range (position n - 1, the chunk's last float4, the group's last head,
    // the row's last float4): values loaded for positions >= n, dims >= cw or
    // heads >= group only feed lanes and steps that are never stored or run,
    // and a branch-free load stream lets the compiler's wait counts keep the
    // loads of MB_DEPTH tiles in flight together.
    using VT = typename Kv4<KT>::T;
    constexpr int ND = KT == KV_Q8 ? NA : 1;   // Q8: V row scales at the weights' positions
    VT rv[MB_DEPTH][NV];
    float4 ra[MB_DEPTH][NA], rd[MB_DEPTH][ND];
    auto load = [&](int tile, VT *v, float4 *a, float4 *dv) {
        const int t0 = min(tile, ntiles - 1) * MB_T;
#pragma unroll
        for (int k = 0; k < NV; k++) {
            const int e = (k * 64 + lane) * 4, r = e / DW, c = min(e % DW, cw - 4);   // position r, dims c..c+3
            v[k] = Kv4<KT>::load(kv.v, vb + (size_t)min(t0 + r, n - 1) * kv_dim + c);
        }
#pragma unroll
        for (int k = 0; k < NA; k++) {
            const int e = (k * 64 + lane) * 4, jj = min(e / MB_T, group - 1), r = e % MB_T;
            const float *src = abase + (ptrdiff_t)((size_t)jj * max_seq) + min(t0 + r, alim);
            a[k] = make_float4(src[0], src[1], src[2], src[3]);
            if (KT == KV_Q8) {
                const float *d = kv.vd + (size_t)first * kv.n_kv + g;
                dv[k] = make_float4(d[(size_t)min(t0 + r, n - 1) * kv.n_kv], d[(size_t)min(t0 + r + 1, n - 1) * kv.n_kv],
                                    d[(size_t)min(t0 + r + 2, n - 1) * kv.n_kv], d[(size_t)min(t0 + r + 3, n - 1) * kv.n_kv]);
            }
        }
    };
    auto stage = [&](int buf, int tile, const VT *v, const float4 *a, const float4 *dv) {
        float *V = vt[buf], *A = aw[buf];
#pragma unroll
        for (int k = 0; k < NV; k++) {
            const int e = (k * 64 + lane) * 4, r = e / DW, c = e % DW;
            const float4 x = Kv4<KT>::wide(v[k]);
            V[(c + 0) * MB_TS + r] = x.x;
            V[(c + 1) * MB_TS + r] = x.y;
            V[(c + 2) * MB_TS + r] = x.z;
            V[(c + 3) * MB_TS + r] = x.w;
        }
#pragma unroll
        for (int k = 0; k < NA; k++) {
            const int e = (k * 64 + lane) * 4, r = e % MB_T;
            // a float4 clamped back from the row's end holds position p at
            // element p - alim: shift it down to element p - p0
            const int sh = tile * MB_T + r - min(tile * MB_T + r, alim);
            const float4 x = a[k];
            float4 y;
            y.x = sh == 0 ? x.x : sh == 1 ? x.y : sh == 2 ? x.z : x.w;
            y.y = sh == 0 ? x.y : sh == 1 ? x.z : x.w;
            y.z = sh == 0 ? x.z : x.w;
            y.w = x.w;
            if (KT == KV_Q8) {   // the weights a_t * dv_t (k_scalar.c:151)
                y.x = kr_fmul(y.x, dv[k].x);
                y.y = kr_fmul(y.y, dv[k].y);
                y.z = kr_fmul(y.z, dv[k].z);
                y.w = kr_fmul(y.w, dv[k].w);
            }
            *(float4 *)(A + e) = y;
        }
        kr_lds_order();
    };
    struct Chunk { float4 v[4], a[4]; };   // 16 steps of one lane
    auto read = [&](Chunk &c, int buf, int k) {
        const float *V = vt[buf] + d * MB_TS + 16 * k, *A = aw[buf] + j * MB_T + 16 * k;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            c.v[i] = *(const float4 *)(V + 4 * i);
            c.a[i] = *(const float4 *)(A + 4 * i);
        }
    };
    float o = 0.0f;
    auto chain = [&](const Chunk &c) {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            o = kr_fadd(o, kr_fmul(c.a[i].x, c.v[i].x));
            o = kr_fadd(o, kr_fmul(c.a[i].y, c.v[i].y));
            o = kr_fadd(o, kr_fmul(c.a[i].z, c.v[i].z));
            o = kr_fadd(o, kr_fmul(c.a[i].w, c.v[i].w));
        }
    };

#pragma unroll
    for (int s = 0; s < MB_DEPTH; s++) load(s, rv[s], ra[s], rd[s]);
    stage(0, 0, rv[0], ra[0], rd[0]);
    load(MB_DEPTH, rv[0], ra[0], rd[0]);
    Chunk c0r, c1r;
    read(c0r, 0, 0);
    // main loop: groups of MB_DEPTH full tiles; tile k0 + s sits in LDS half
    // s & 1 and its first chunk is in c0r when its step begins
    const int ngroups = n / (MB_T * MB_DEPTH);
    int k0 = 0;
    for (; k0 < ngroups * MB_DEPTH; k0 += MB_DEPTH) {
#pragma unroll
        for (int s = 0; s < MB_DEPTH; s++) {
            const int b = s & 1, nx = (s + 1) % MB_DEPTH;
            // phases fenced for the scheduler: a chunk's reads are issued
            // one phase before its products and adds, and the staging of
            // the next tile shares a phase with the first chunk's adds
            read(c1r, b, 1);
            __builtin_amdgcn_sched_barrier(0);
            chain(c0r);
            stage(b ^ 1, k0 + s + 1, rv[nx], ra[nx], rd[nx]);
            load(k0 + s + 1 + MB_DEPTH, rv[nx], ra[nx], rd[nx]);
            __builtin_amdgcn_sched_barrier(0);
            read(c0r, b, 2);
            __builtin_amdgcn_sched_barrier(0);
            chain(c1r);
            __builtin_amdgcn_sched_barrier(0);
            read(c1r, b, 3);
            __builtin_amdgcn_sched_barrier(0);
            chain(c0r);
            __builtin_amdgcn_sched_barrier(0);
            read(c0r, b ^ 1, 0);
            __builtin_amdgcn_sched_barrier(0);
            chain(c1r);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    // the last tiles (at most MB_DEPTH; tile k0 is staged in half 0, tile
    // k0 + s is in rv[s]); the last may be partial, and only its live steps
    // run: a zero weight would turn -0 to +0
#pragma unroll
    for (int s = 0; s < MB_DEPTH; s++) {
        const int tile = k0 + s;
        if (tile < ntiles) {
            if (s > 0) stage(s & 1, tile, rv[s], ra[s], rd[s]);
            const int nt = min(MB_T, n - tile * MB_T);
            const float *V = vt[s & 1] + d * MB_TS, *A = aw[s & 1] + j * MB_T;
            for (int r = 0; r < nt; r++) o = kr_fadd(o, kr_fmul(A[r], V[r]));
            kr_lds_order();
        }
    }
    if (j < group && d < cw) ao[(size_t)(g * group + j) * hd + c0 + d] = o;
}

// Batched (prefill) mix by blocks of MK_W x MK_U tokens: a
// workgroup per (KV head g, DW dims from c0, MK_W MK_U consecutive tokens),
// MK_U consecutive tokens per wave, lane = (head j of the group, dim d); each
// lane runs its tokens' chains o += a_t * v_t,d over positions t in order
// (k_scalar.c:119-122), each product rounded before its add. The block's waves
// share each V tile, staged once in LDS as [dim][position] so one 16-byte read
// gives a lane 4 positions, and each V value read serves the lane's MK_U
// chains, whose adds interleave (a chain's next add need not wait for its
// last). The weights take no LDS: a lane holds its head's weights of 16
// positions in one register a token (lane d of a 16-lane row holds position
// t0 + d), and a DPP row broadcast (row_newbcast) hands position t0 + k's
// weight to every lane of the row as the multiply's operand. So a row of 16
// lanes must hold one head: DW >= 16. Tiles are double-buffered: tile k + 1
// is stored while tile k is read, the loads of tile k + 2 already in flight.
// F16 and Q8 cache rows are widened exactly as they are staged; over the Q8
// cache a lane's weight is a_t * dv_t (the row's scale, k_scalar.c:151)
// before the broadcast, as in the per-token mix.
constexpr int MK_W = 4, MK_U = 2, MK_T = 64, MK_TS = MK_T + 4;

template <int K> __device__ __forceinline__ float row_bcast(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x150 + K, 0xF, 0xF, false));
}

// o[u] += a_{t0+4q+i} * v4.i for i < 4 and every token u, positions
// t0 + 4q + i of a 16-position block whose weights sit in a[u] (lane k of
// each row: position t0 + k); the tokens' adds of one position go out together
template <int Q, int U>
__device__ __forceinline__ void mk_quad(float (&o)[U], const float (&a)[U], float4 v) {
#pragma unroll
    for (int u = 0; u < U; u++) o[u] = kr_fadd(o[u], kr_fmul(row_bcast<4 * Q + 0>(a[u]), v.x));
#pragma unroll
    for (int u = 0; u < U; u++) o[u] = kr_fadd(o[u], kr_fmul(row_bcast<4 * Q + 1>(a[u]), v.y));
#pragma unroll
    for (int u = 0; u < U; u++) o[u] = kr_fadd(o[u], kr_fmul(row_bcast<4 * Q + 2>(a[u]), v.z));
#pragma unroll
    for (int u = 0; u < U; u++) o[u] = kr_fadd(o[u], kr_fmul(row_bcast<4 * Q + 3>(a[u]), v.w));
}

template <int DW, int KT, bool WIN>
__global__ void __launch_bounds__(64 * MK_W) k_attn_mix_blk(float *ao, const float *att, const KvView kv, int group,
                                                            int hd, int kv_dim, int max_seq, int window_arg,
                                                            const int *pos_p, int ntok) {
    const int window = WIN ? window_arg : 0;
    static_assert(DW >= 16, "a 16-lane row must hold one head");
    constexpr int U = MK_U;
    constexpr int QPR = DW / 4;                 // float4 per staged row of DW dims
    constexpr int RPP = 64 * MK_W / QPR;        // rows the workgroup stages per pass
    constexpr int NP = MK_T / RPP;              // passes per tile
    __shared__ __align__(16) float vt[2][DW * MK_TS];
    __shared__ float dvs[2][KT == KV_Q8 ? MK_T : 1];   // Q8: the tile's V row scales
    const int g = blockIdx.x, c0 = blockIdx.y * DW, z0 = blockIdx.z * MK_W * U, tid = threadIdx.x;
    const int wave = tid >> 6, lane = tid & 63, j = lane / DW, d = lane % DW;
    const int zw = z0 + wave * U, pos0 = *pos_p;      // the wave's first token
    const int nmax = pos0 + min(z0 + MK_W * U, ntok);   // positions the block's last token attends
    const int n_heads = gridDim.x * group, cw = min(DW, hd - c0);
    const int base = attn_first(pos0 + z0, window) / MK_T * MK_T;   // the block's first tile
    const int ntiles = (nmax - base + MK_T - 1) / MK_T;
    int n[U], f[U];   // token zw + u attends positions f .. n - 1 (n 0 past the last token)
    const float *arow[U];
#pragma unroll
    for (int u = 0; u < U; u++) {
        n[u] = zw + u < ntok ? pos0 + zw + u + 1 : 0;
        f[u] = attn_first(pos0 + zw + u, window);
        arow[u] = att + ((size_t)min(zw + u, ntok - 1) * n_heads + (size_t)g * group + min(j, group - 1)) * max_seq;
    }
    const size_t vbase = (size_t)g * hd + c0;   // element offset of the chunk in a V row
    // staging slot of this thread in pass p: row p * RPP + srow, dims scol .. scol + 3
    const int srow = tid / QPR, scol = min(4 * (tid % QPR), cw - 4);
    using VT = typename Kv4<KT>::T;
    VT sv[NP];
    float sd = 0.0f;
    auto stage_load = [&](int tile) {
#pragma unroll
        for (int p = 0; p < NP; p++)
            sv[p] = Kv4<KT>::load(kv.v, vbase + (size_t)min(base + tile * MK_T + p * RPP + srow, nmax - 1) * kv_dim + scol);
        if (KT == KV_Q8 && tid < MK_T) sd = kv.vd[(size_t)min(base + tile * MK_T + tid, nmax - 1) * kv.n_kv + g];
    };
    auto stage_store = [&](int buf) {
        float *V = vt[buf];
#pragma unroll
        for (int p = 0; p < NP; p++) {
            const int r = p * RPP + srow, c = 4 * (tid % QPR);
            const float4 x = Kv4<KT>::wide(sv[p]);
            V[(c + 0) * MK_TS + r] = x.x;
            V[(c + 1) * MK_TS + r] = x.y;
            V[(c + 2) * MK_TS + r] = x.z;
            V[(c + 3) * MK_TS + r] = x.w;
        }
        if (KT == KV_Q8 && tid < MK_T) dvs[buf][tid] = sd;
    };
    // the weights of a tile, loaded two tiles ahead like V: one tile's adds
    // are shorter than a load's round trip
    auto a_load = [&](int tile, float (&a)[U][MK_T / 16]) {
#pragma unroll
        for (int u = 0; u < U; u++)
#pragma unroll
            for (int b = 0; b < MK_T / 16; b++) a[u][b] = arow[u][min(base + tile * MK_T + 16 * b + (lane & 15), max_seq - 1)];
    };
    float o[U];
#pragma unroll
    for (int u = 0; u < U; u++) o[u] = 0.0f;
    float acur[U][MK_T / 16], anext[U][MK_T / 16], anext2[U][MK_T / 16];
    stage_load(0);
    stage_store(0);
    a_load(0, acur);
    a_load(min(1, ntiles - 1), anext);
    if (ntiles > 1) stage_load(1);
    __syncthreads();
    for (int k = 0; k < ntiles; k++) {
        const int buf = k & 1, t0 = base + k * MK_T;
        if (k + 1 < ntiles) stage_store(buf ^ 1);   // its last reader finished before the last barrier
        a_load(min(k + 2, ntiles - 1), anext2);
        // unconditional (a clamped tile past the end is loaded and never
        // stored): with a fixed count of loads behind them, the waits for
        // the weights at the end of the step leave this load in flight
        stage_load(min(k + 2, ntiles - 1));
        const float *V = vt[buf] + d * MK_TS;
        float aw[MK_T / 16][U];   // the weights (Q8: a_t * dv_t)
#pragma unroll
        for (int b = 0; b < MK_T / 16; b++)
#pragma unroll
            for (int u = 0; u < U; u++)
                aw[b][u] = KT == KV_Q8 ? kr_fmul(acur[u][b], dvs[buf][KT == KV_Q8 ? 16 * b + (lane & 15) : 0]) : acur[u][b];
        if (t0 + MK_T <= n[0] && t0 >= f[U - 1]) {   // a full tile for every token of the wave (tokens past the last are not stored)
#pragma unroll
            for (int b = 0; b < MK_T / 16; b++) {
                const float4 v0 = *(const float4 *)(V + 16 * b), v1 = *(const float4 *)(V + 16 * b + 4);
                const float4 v2 = *(const float4 *)(V + 16 * b + 8), v3 = *(const float4 *)(V + 16 * b + 12);
                mk_quad<0>(o, aw[b], v0);
                mk_quad<1>(o, aw[b], v1);
                mk_quad<2>(o, aw[b], v2);
                mk_quad<3>(o, aw[b], v3);
            }
        } else {   // the first and last tiles: each token its live positions
#pragma unroll
            for (int u = 0; u < U; u++) {
                if (t0 >= n[u] || t0 + MK_T <= f[u]) continue;
#pragma unroll
                for (int b = 0; b < MK_T / 16; b++) {
                    const float ab = aw[b][u];
                    float w[16];
                    w[0] = row_bcast<0>(ab); w[1] = row_bcast<1>(ab); w[2] = row_bcast<2>(ab); w[3] = row_bcast<3>(ab);
                    w[4] = row_bcast<4>(ab); w[5] = row_bcast<5>(ab); w[6] = row_bcast<6>(ab); w[7] = row_bcast<7>(ab);
                    w[8] = row_bcast<8>(ab); w[9] = row_bcast<9>(ab); w[10] = row_bcast<10>(ab); w[11] = row_bcast<11>(ab);
                    w[12] = row_bcast<12>(ab); w[13] = row_bcast<13>(ab); w[14] = row_bcast<14>(ab); w[15] = row_bcast<15>(ab);
                    for (int i = 0; i < 16 && t0 + 16 * b + i < n[u]; i++)
                        if (t0 + 16 * b + i >= f[u]) o[u] = kr_fadd(o[u], kr_fmul(w[i], V[16 * b + i]));
                }
            }
        }
#pragma unroll
        for (int u = 0; u < U; u++)
#pragma unroll
            for (int b = 0; b < MK_T / 16; b++) {
                acur[u][b] = anext[u][b];
                anext[u][b] = anext2[u][b];
            }
        kr_lds_order();
        __syncthreads();
    }
    if (j < group && d < cw) {
#pragma unroll
        for (int u = 0; u < U; u++)
            if (zw + u < ntok) ao[(size_t)(zw + u) * n_heads * hd + (size_t)(g * group + j) * hd + c0 + d] = o[u];
    }
}

// Batched (prefill) mix blocked in registers: the rows (token z, query head
// j) of KV head g, numbered z * group + j, go to workgroups RB_R at a time
// (the longest first), CW of the head's dims each, and lane (row group rg,
// dim group dg) of a workgroup owns the 4 x 4 outputs of rows 4 rg ..
// 4 rg + 3 and dims 4 dg + i: one chain o += a_t * v_t,d per output over
// positions t in order (k_scalar.c:119-122), each product rounded before its
// add. Per tile of RB_T positions (from the tile of the first row's first
// attended position) the weights [row][position] (Q8: a_t * dv_t, the
// per-token kernel's product) and the V rows [position][dim] (F16 widened, Q8
// as its int8 values) are staged in LDS; per 4 positions a lane reads its
// rows' 4 weights and, per position, its dims' V values, 16-byte reads that
// feed every product they take part in (16 chains a lane, 2 reads for 16
// multiplies and as many adds: no broadcasts of a weight across lanes). In the
// tiles past some row's own positions, or before its window, a select leaves
// those terms out of that row's sums, so no weight or V value there (rows of
// later tokens, stale rows) reaches them. The next tile's loads are in flight
// while a tile is summed.
constexpr int rb_cw(int hd) { return hd == 256 ? 128 : hd; }   // dims of a workgroup
template <int HD, int KT, bool WIN>
__global__ void __launch_bounds__(4 * rb_cw(HD)) k_attn_mix_rb(float *ao, const float *att, const KvView kv, int group,
                                                               int kv_dim, int max_seq, int window_arg,
                                                               const int *pos_p, int ntok) {
    const int window = WIN ? window_arg : 0;
    constexpr int CW = rb_cw(HD), hd = HD;
    constexpr int NT = 4 * CW, NDG = CW / 4;          // threads; dim groups
    constexpr int AS = RB_T + 4;                      // weight row stride (floats)
    constexpr int NW4 = RB_R * RB_T / 4;              // a tile's 4-weight loads
    constexpr int NA = (NW4 + NT - 1) / NT;           // of them a thread's, at most
    constexpr int NV = RB_T * CW / 4 / NT;            // 4-element V loads a thread stages per tile
    __shared__ __align__(16) float as[RB_R * AS];
    __shared__ __align__(16) float vs[RB_T * CW];
    const int g = blockIdx.x, tid = threadIdx.x, wave = tid >> 6, dg = tid % NDG, rg = tid / NDG;
    const int nrow = ntok * group, R0 = (gridDim.y - 1 - blockIdx.y) * RB_R;
    const int pos0 = *pos_p, n_heads = gridDim.x * group;
    const int nlast = pos0 + (min(R0 + RB_R, nrow) - 1) / group + 1;   // positions the block's last row attends
    const int base = attn_first(pos0 + R0 / group, window) / RB_T * RB_T;   // the block's first tile
    const int ntl = (nlast - base + RB_T - 1) / RB_T, c0 = HD == CW ? 0 : blockIdx.z * CW;
    const int zw = (R0 + 4 * (64 * wave / NDG)) / group;   // the token of the wave's first row
    const int zlw = (min(R0 + 4 * ((64 * wave + 63) / NDG + 1), nrow) - 1) / group;   // of its last (within the rows)
    const int fw = attn_first(pos0 + zw, window), flw = attn_first(pos0 + zlw, window);   // the first positions they attend
    typename Kv4<KT>::T vr[NV];
    float4 ar[NA];
    float dv[NA][4];   // Q8: the V row scales of the staged weights' positions
    auto load = [&](int t0) {
#pragma unroll
        for (int u = 0; u < NV; u++) {
            const int e = tid + NT * u, p = e / (CW / 4), c4 = e % (CW / 4);
            vr[u] = Kv4<KT>::load(kv.v, (size_t)min(t0 + p, nlast - 1) * kv_dim + (size_t)g * hd + c0 + 4 * c4);
        }
#pragma unroll
        for (int u = 0; u < NA; u++) {
            const int e = min(tid + NT * u, NW4 - 1), rr = e / (RB_T / 4), q4 = e % (RB_T / 4);
            const int R = min(R0 + rr, nrow - 1), z = R / group, j = R - z * group;
            ar[u] = *(const float4 *)(att + ((size_t)z * n_heads + (size_t)g * group + j) * max_seq +
                                      min(t0 + 4 * q4, max_seq - 4));
            if (KT == KV_Q8) {
#pragma unroll
                for (int i = 0; i < 4; i++) dv[u][i] = kv.vd[(size_t)min(t0 + 4 * q4 + i, nlast - 1) * kv.n_kv + g];
            }
        }
    };
    float acc[4][4];
#pragma unroll
    for (int r = 0; r < 4; r++)
#pragma unroll
        for (int c = 0; c < 4; c++) acc[r][c] = 0.0f;
    load(base);
    for (int ti = 0; ti < ntl; ti++) {
        const int t0 = base + ti * RB_T;
        __syncthreads();   // the last tile is read
#pragma unroll
        for (int u = 0; u < NV; u++) {
            const int e = tid + NT * u;
            *(float4 *)(vs + 4 * e) = Kv4<KT>::wide(vr[u]);   // [position][dim]: e = p CW / 4 + c4
        }
#pragma unroll
        for (int u = 0; u < NA; u++) {
            const int e = tid + NT * u, rr = e / (RB_T / 4), q4 = e % (RB_T / 4);
            if (NW4 % NT && e >= NW4) break;
            float4 a = ar[u];
            if (KT == KV_Q8)
                a = make_float4(kr_fmul(a.x, dv[u][0]), kr_fmul(a.y, dv[u][1]), kr_fmul(a.z, dv[u][2]),
                                kr_fmul(a.w, dv[u][3]));
            *(float4 *)(as + rr * AS + 4 * q4) = a;
        }
        __syncthreads();
        if (ti + 1 < ntl) load(t0 + RB_T);
        const float *ap = as + 4 * rg * AS, *vp = vs + 4 * dg;
        // positions t .. t + 3 of the tile, every row's terms (OWN: each
        // row's own positions only)
        auto step = [&](int t, auto own, const int *lo, const int *lim) {
            constexpr bool OWN = decltype(own)::value;
            float4 a[4];
#pragma unroll
            for (int r = 0; r < 4; r++) a[r] = *(const float4 *)(ap + r * AS + t);
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const float4 x = *(const float4 *)(vp + (t + k) * CW);
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const float w = k == 0 ? a[r].x : k == 1 ? a[r].y : k == 2 ? a[r].z : a[r].w;
                    const bool in = !OWN || (t + k <= lim[r] && (!WIN || t + k >= lo[r]));
                    float *o = acc[r];
                    o[0] = in ? kr_fadd(o[0], kr_fmul(w, x.x)) : o[0];
                    o[1] = in ? kr_fadd(o[1], kr_fmul(w, x.y)) : o[1];
                    o[2] = in ? kr_fadd(o[2], kr_fmul(w, x.z)) : o[2];
                    o[3] = in ? kr_fadd(o[3], kr_fmul(w, x.w)) : o[3];
                }
            }
        };
        if (t0 + RB_T - 1 <= pos0 + zw && (!WIN || t0 >= flw)) {   // every position counts for every row of the wave
#pragma unroll 2
            for (int t = 0; t < RB_T; t += 4) step(t, std::false_type{}, nullptr, nullptr);
        } else {
            // a tile that holds the wave's own positions or its windows'
            // starts: whole steps where every row attends, masked steps
            // where some do, none outside
            const int full = pos0 + zw - t0, any = pos0 + zlw - t0;
            int lim[4], lo[4];   // in a masked step: position t0 + k counts for row r iff lo[r] <= k <= lim[r]
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int pr = pos0 + (R0 + 4 * rg + r) / group;
                lim[r] = pr - t0;
                lo[r] = attn_first(pr, window) - t0;
            }
            for (int t = WIN ? max(0, (fw - t0) / 4 * 4) : 0; t < RB_T && t <= any; t += 4) {
                if (t + 3 <= full && (!WIN || t >= flw - t0)) step(t, std::false_type{}, nullptr, nullptr);
                else step(t, std::true_type{}, lo, lim);
            }
        }
    }
#pragma unroll
    for (int r = 0; r < 4; r++) {
        const int R = R0 + 4 * rg + r;
        if (R >= nrow) continue;
        const int z = R / group, j = R - z * group;
        *(float4 *)(ao + ((size_t)z * n_heads + (size_t)g * group + j) * hd + c0 + 4 * dg) =
            make_float4(acc[r][0], acc[r][1], acc[r][2], acc[r][3]);
    }
}

template <int DW>
__global__ void __launch_bounds__(64) k_attn_mix_batch(float *ao, const float *att, const float *vc, int group, int hd,
                                                       int kv_dim, int max_seq, int window, const int *pos_p) {
    const KvView kv = { nullptr, vc, nullptr, nullptr, 0 };
    attn_mix_batch<DW, KV_F32>(ao, att, kv, group, hd, kv_dim, max_seq, window, pos_p);
}

template <int DW, int KT>
__global__ void __launch_bounds__(64) k_attn_mix_batch_kv(float *ao, const float *att, const KvView kv, int group,
                                                          int hd, int kv_dim, int max_seq, int window,
                                                          const int *pos_p) {
    attn_mix_batch<DW, KT>(ao, att, kv, group, hd, kv_dim, max_seq, window, pos_p);
}

// ---- launches ----

// the kernels of a launch's scores and mix (one workgroup a token and tile,
// blocks of tokens, register-blocked rows) and of its softmax (a row: 1024 or
// 256 threads, or a wave)
enum { AP_TOKEN, AP_BLOCK, AP_ROWS };
enum { AP_SMX_1024, AP_SMX_256, AP_SMX_WAVE };
struct AttnPlan {
    int scores, pc, softmax, mix;   // pc: the register-blocked scores' K tiles a workgroup
};
struct AttnShape {
    int kt, n_heads, n_kv, hd, max_seq, window, ntok, max_pos;
    int group() const { return n_heads / n_kv; }
    bool cut() const { return window && window <= max_pos; }         // some token attends less than its prefix
    int nmax() const { return cut() ? window : max_pos + 1; }        // positions a row attends, at most
    int row_blocks() const { return (ntok * group() + RB_R - 1) / RB_R; }
    // tiles of tp positions that tb consecutive tokens attend, at most
    int span_tiles(int tb, int tp) const {
        const int all = (max_pos + tp) / tp;
        return cut() ? std::min(all, (window + tb - 1 + tp - 1 + tp - 1) / tp) : all;
    }
    int row_tiles() const { return span_tiles((RB_R - 1) / group() + 2, RB_T); }
    // tokens whose queries (F32, F16: floats; Q8: quantized, with their scales)
    // fit in 64 KB of LDS beside the token blocks' K tile of tp positions; 0: none
    size_t tile_bytes(int tp) const { return sizeof(float) * (size_t)tp * (hd + 4); }
    size_t q8_bytes(int qb) const {
        return sizeof(float) * (AT_T + (size_t)(qb * group() + 3) / 4 * 4) + (size_t)(AT_T * (hd + 4) + 15) / 16 * 16 +
               (size_t)qb * group() * hd;
    }
    size_t block_bytes(int tp, int qb) const {
        return kt == KV_Q8 ? q8_bytes(qb) : tile_bytes(tp) + sizeof(float) * (size_t)qb * group() * hd;
    }
    int qb_at(int tp) const {
        for (int qb = kt == KV_Q8 ? 16 : 8; qb >= 4; qb /= 2)
            if (block_bytes(tp, qb) <= 64 * 1024) return qb;
        return 0;
    }
    int tp() const { return kt == KV_Q8 || qb_at(AT_T) ? AT_T : AT_T / 2; }
    int qb() const { return qb_at(tp()); }
    int dw() const {   // dims of a mix workgroup's lanes
        const int g = group(), gp = g <= 1 ? 1 : g <= 2 ? 2 : g <= 4 ? 4 : g <= 8 ? 8 : 16;
        return 64 / gp;
    }
    // what a stage's kernels take
    bool scores_block() const { return qb() != 0; }
    bool scores_rows() const { return kt != KV_Q8 && rb_dims(hd); }
    bool mix_block() const { return dw() >= 16; }
    bool mix_rows() const { return rb_dims(hd) && max_seq % 4 == 0; }
    int mix_row_blocks() const { return n_kv * row_blocks() * (hd / rb_cw(hd)); }
};

// The choice: for each stage the kernels with the least estimated time. The
// constants (us, on the 256 CUs of an MI355X) are fitted to the choice: every
// form of the three stages was timed for 21 head counts and sizes (1 to 32 heads
// over 1 to 16 KV heads of 32 to 256 dims), three cache types, prompts of 2 to 2000
// tokens at positions 0, 500 and 2000, without a window and with ones of 96 to
// 1024 positions: 5040 launches. The choice's three stages together cost 0.6%
// more than the best form of each, and 24 of the 5040 take over 4% longer than with
// the token blocks and register-blocked rows chosen by the grid's size alone
// and windows one token a workgroup; on average 25% less. Windowed batches of few
// tokens lose most in large blocks: 4 heads of 64, 101 tokens over a window of
// 70: 12.7 us one token a workgroup, 43 in blocks.
struct ApScores {      // one token a workgroup; token blocks
    float lat, lat_hd, tile_math, tile_stage, wide, tile, grid, blk_lat, blk_lat_hd, blk_step, blk_tile, blk_tile_step,
        q8_step;
};
constexpr ApScores AP_SC = { 6.0f, 0.014f, 3.4e-05f, 2e-05f, 1.4f, 5e-07f, 3.1e-06f, 5.8f, 0.00044f, 0.089f, 0.01f, 0.00015f, 0.0f };
constexpr ApScores AP_SC_Q8 = { 4.6f, 0.022f, 1.5e-05f, 0.0f, 1.0f, 0.00079f, 0.0004f, 6.0f, 0.02f, 0.095f, 0.0025f, 0.00021f, 0.014f };
struct ApRows {        // register-blocked rows of hd dims: workgroups a CU holds, scores, mix
    int hd, resident;
    float fixed, tile, shared, mix_tile;
};
constexpr ApRows AP_ROW[] = {
    { 48, 4, 6.3f, 3.2f, 1.3f, 0.011f },
    { 64, 4, 4.5f, 8.4f, 1.1f, 0.0092f },
    { 80, 3, 5.9f, 11.0f, 2.4f, 0.036f },
    { 96, 3, 6.6f, 13.0f, 4.0f, 0.022f },
    { 128, 2, 4.0f, 10.0f, 3.8f, 0.028f },
    { 256, 4, 2.0f, 41.0f, 16.0f, 0.03f },
};

// what a launch does, for the estimates
struct ApWork {
    double pairs;          // (token, position) pairs attended
    float n, navg;         // positions a token attends, at most and on average
    bool cut;              // a token attends less than its prefix
    bool full;             // every token a whole window
    int tb;                // tokens of a block of RB_R rows, at most
};

ApWork ap_work(const AttnShape &s) {
    ApWork w;
    const double T = s.ntok, p0 = s.max_pos + 1 - s.ntok;
    w.cut = s.cut();
    w.full = w.cut && p0 >= s.window;
    if (!w.cut) w.pairs = T * p0 + T * (T + 1) / 2;
    else if (w.full) w.pairs = T * s.window;
    else {
        const double k = s.window - p0;   // tokens below the window's length
        w.pairs = k * p0 + k * (k + 1) / 2 + (T - k) * s.window;
    }
    w.n = (float)s.nmax();
    w.navg = (float)(w.pairs / T);
    w.tb = std::min(s.ntok, (RB_R - 1) / s.group() + 1);
    return w;
}

const ApRows *ap_rows(int hd) {
    for (const ApRows &r : AP_ROW)
        if (r.hd == hd) return &r;
    return nullptr;
}

// the scores: one token a workgroup and tile, or blocks of AT_TB tokens a tile
float est_scores_token(const AttnShape &s, const ApWork &w) {
    const bool q8 = s.kt == KV_Q8;
    const ApScores &c = q8 ? AP_SC_Q8 : AP_SC;
    const float g4 = (float)((s.group() + 3) / 4), hd = (float)s.hd, kvt = (float)s.n_kv * s.ntok;
    const bool wide = !q8 && attn_tile<KV_F32>(s.group(), s.hd) == AT_TD;
    const float tp = wide ? AT_TD : AT_T;
    const float tiles = w.full ? kvt * ((s.window + 63) / 64) : (float)s.n_kv * (float)(w.pairs / 64 + 0.5 * s.ntok);
    const float x = (float)s.n_kv * hd * (float)(w.pairs / 64);
    const float thr = (x * (c.tile_math * g4 + c.tile_stage) + c.tile * tiles) * (wide ? c.wide : 1.0f) +
                      c.grid * kvt * std::ceil(w.n / tp);
    return std::max(c.lat + c.lat_hd * hd * g4, thr);
}
float est_scores_block(const AttnShape &s, const ApWork &w) {
    const bool q8 = s.kt == KV_Q8;
    const ApScores &c = q8 ? AP_SC_Q8 : AP_SC;
    const float hd = (float)s.hd;
    const int zn = std::min(s.ntok, AT_TB), qb = q8 ? AT_TB : s.qb();
    const float step = q8 ? (float)(zn * s.group()) * (1.0f + c.q8_step * hd)
                          : hd * (float)((zn + qb - 1) / qb) * (float)((s.group() + 3) / 4);
    const float tiles = (float)s.n_kv * ((s.ntok + AT_TB - 1) / AT_TB) * ((w.navg + 15) / s.tp() + 1);
    return std::max(c.blk_lat + c.blk_lat_hd * hd + c.blk_step * step, tiles * (c.blk_tile + c.blk_tile_step * step));
}
// register-blocked scores, pc tiles a workgroup
float est_scores_rows(const AttnShape &s, const ApWork &w, const ApRows &c, int pc) {
    const float nt = std::floor((w.n + w.tb - 1 + 63) / 64), tiles = (w.navg + w.tb - 1) / 64 + 1;
    const float pe = std::min((float)pc, nt), blocks = (float)s.n_kv * s.row_blocks();
    const float n = std::max(1.0f, blocks * std::min(std::ceil(nt / pc), tiles / pc + 0.5f) / 256);
    const float rounds = std::max(1.0f, n / c.resident);
    return rounds * (c.fixed + c.tile * pe) + (n - rounds) * c.shared * pe;
}

// the mix: a wave a token and DW dims, token blocks, register-blocked rows
float est_mix_token(const AttnShape &s, const ApWork &w) {
    const bool q8 = s.kt == KV_Q8;
    const int dw = s.dw(), k = dw == 64 ? 0 : dw == 32 ? 1 : 2;
    constexpr float per[2][3] = { { 6.7e-05f, 2e-05f, 1.2e-05f }, { 6.7e-05f, 2.1e-05f, 1.8e-05f } };
    const float lat = 1.8f + (q8 ? 0.19f : 0.0f) + (k == 0 ? 0.018f : 0.0098f) * w.n;
    return std::max(lat, per[q8][k] * (float)s.n_kv * ((s.hd + dw - 1) / dw) * (float)w.pairs);
}
float est_mix_block(const AttnShape &s, const ApWork &w) {
    const int dw = s.dw();
    const float lat = 2.0f + (w.cut ? 17.0f : 0.0f) + (dw == 64 ? 2.1f : 1.7f) * w.n / 64;
    const float wgs = (float)s.n_kv * ((s.hd + dw - 1) / dw) * ((s.ntok + MK_W * MK_U - 1) / (MK_W * MK_U));
    return std::max(lat, (dw == 64 ? 0.0039f : 0.0021f) * wgs * ((w.navg + 7) / 64 + 1 + (w.cut ? 2.7f : 0.0f)));
}
float est_mix_rows(const AttnShape &s, const ApWork &w, const ApRows &c) {
    const float lat = 1.6f + 6.6f * ((w.n + w.tb - 1) / 64 + (w.cut ? 0.35f : 0.0f));
    return std::max(lat, c.mix_tile * (float)s.mix_row_blocks() * ((w.navg + w.tb - 1) / 64 + 1)) * (s.kt == KV_Q8 ? 1.1f : 1.0f);
}

// krh_set_attn_rb_min: at other values than its default the grids alone decide
// between register-blocked rows and token blocks
constexpr int RB_MIN_WG = 512;
int g_rb_min_wg = RB_MIN_WG;
bool rb_fills(long wgs) { return 2 * wgs >= g_rb_min_wg; }

AttnPlan attn_plan(const AttnShape &s) {
    AttnPlan p = { AP_TOKEN, RB_PC, AP_SMX_1024, AP_TOKEN };
    if (g_rb_min_wg != RB_MIN_WG) {
        if (s.scores_block()) p.scores = AP_BLOCK;
        if (s.mix_block()) p.mix = AP_BLOCK;
        // a scores workgroup's K tiles are cut until the grid fills the device
        const long blocks = (long)s.n_kv * s.row_blocks();
        auto chunks = [&] { return (s.row_tiles() + p.pc - 1) / p.pc; };
        while (p.pc > 1 && !rb_fills(blocks * chunks() / 2)) p.pc /= 2;
        if (s.scores_rows() && rb_fills(blocks * chunks())) p.scores = AP_ROWS;
        if (s.mix_rows() && rb_fills(s.mix_row_blocks())) p.mix = AP_ROWS;
    } else {
        const ApWork w = ap_work(s);
        const ApRows *rows = ap_rows(s.hd);
        float t = est_scores_token(s, w);
        auto take = [&](float e, int &choice, int form) {
            if (e >= t) return false;
            t = e;
            choice = form;
            return true;
        };
        if (s.scores_block()) take(est_scores_block(s, w), p.scores, AP_BLOCK);
        for (int pc = 1; s.scores_rows() && pc <= RB_PC; pc *= 2)
            if (take(est_scores_rows(s, w, *rows, pc), p.scores, AP_ROWS)) p.pc = pc;
        t = est_mix_token(s, w);
        if (s.mix_block()) take(est_mix_block(s, w), p.mix, AP_BLOCK);
        if (s.mix_rows()) take(est_mix_rows(s, w, *rows), p.mix, AP_ROWS);
    }
    // a wave a row only for rows of up to 2048 scores that fill the device:
    // 1024 rows of 1000 scores take 9.9 us a wave each and 7.6 at 256 threads each,
    // 2048 rows 11.4 and 12.2; rows past 4096 scores take 1024 threads
    if (s.nmax() <= SM_WN / 2 && (long)s.ntok * s.n_heads > 1024) p.softmax = AP_SMX_WAVE;
    else if (s.nmax() <= 4096) p.softmax = AP_SMX_256;
    return p;
}

template <int V> using ic = std::integral_constant<int, V>;

// calls go(head size) with the head size as a constant
template <class F> void rb_switch(int hd, F &&go) {
    switch (hd) {
    case 48: go(ic<48>{}); break;
    case 64: go(ic<64>{}); break;
    case 80: go(ic<80>{}); break;
    case 96: go(ic<96>{}); break;
    case 128: go(ic<128>{}); break;
    default: go(ic<256>{}); break;
    }
}

template <int KT, bool WIN>
void launch_scores(const AttnShape &s, const AttnPlan &p, float *att, const float *q, const KvView &kv, float scale,
                   const int *pos) {
    const int group = s.group(), kv_dim = s.n_kv * s.hd;
    if (p.scores == AP_ROWS) {
        if constexpr (KT != KV_Q8) {
            const dim3 grid(s.n_kv, s.row_blocks(), (s.row_tiles() + p.pc - 1) / p.pc);
            rb_switch(s.hd, [&](auto dims) {
                constexpr int HD = decltype(dims)::value, NT = HD == 128 ? RB_NT128 : 256, HS = HD == 256 ? 64 : HD;
                hipLaunchKernelGGL((k_attn_scores_rb<HD, KT, NT, WIN, HS>), grid, dim3(NT), 0, kr_stream(), att, q, kv,
                                   group, kv_dim, s.max_seq, s.window, scale, pos, s.ntok, p.pc);
            });
        }
        return;
    }
    if (p.scores == AP_BLOCK) {   // blocks of AT_TB tokens share a K tile
        const int tp = s.tp(), qb = s.qb();
        const dim3 grid(s.n_kv, s.span_tiles(AT_TB, tp), (s.ntok + AT_TB - 1) / AT_TB);
        const size_t lds = s.block_bytes(tp, qb);
        if constexpr (KT == KV_Q8) {
            auto go = [&](auto kern) {
                hipLaunchKernelGGL(kern, grid, dim3(AT_THREADS), lds, kr_stream(), att, q, kv, group, s.hd, kv_dim,
                                   s.max_seq, s.window, scale, pos, s.ntok);
            };
            if (qb == 16) go(k_attn_scores_blk_q8<16, WIN>);
            else if (qb == 8) go(k_attn_scores_blk_q8<8, WIN>);
            else go(k_attn_scores_blk_q8<4, WIN>);
        } else {
            auto go = [&](auto kern) {
                hipLaunchKernelGGL(kern, grid, dim3(AT_THREADS), lds, kr_stream(), att, q, kv, group, s.hd, kv_dim,
                                   s.max_seq, s.window, scale, pos, s.ntok);
            };
            auto at = [&](auto q_) {
                constexpr int QB = decltype(q_)::value;
                if (tp != AT_T) go(k_attn_scores_blk<0, QB, KT, AT_T / 2, WIN>);
                else if (s.hd == 128) go(k_attn_scores_blk<128, QB, KT, AT_T, WIN>);
                else if (s.hd == 64) go(k_attn_scores_blk<64, QB, KT, AT_T, WIN>);
                else go(k_attn_scores_blk<0, QB, KT, AT_T, WIN>);
            };
            if (qb == 8) at(ic<8>{});
            else at(ic<4>{});
        }
        return;
    }
    // a workgroup for each token and tile of the positions it attends
    const int tt = attn_tile<KT>(group, s.hd);
    const size_t lds = attn_tile_lds<KT>(group, s.hd, tt);
    const dim3 grid(s.n_kv, (s.nmax() + tt - 1) / tt, s.ntok);
    auto go = [&](auto kern, auto k) {
        hipLaunchKernelGGL(kern, grid, dim3(AT_THREADS), lds, kr_stream(), att, q, k, group, s.hd, kv_dim, s.max_seq,
                           s.window, scale, pos);
    };
    if constexpr (KT == KV_Q8) {
        go(k_attn_scores_q8<true>, kv);
    } else if constexpr (KT == KV_F32) {
        if (tt == AT_T) go(k_attn_scores<AT_T, true>, (const float *)kv.k);
        else go(k_attn_scores<AT_TD, true>, (const float *)kv.k);
    } else {
        if (tt == AT_T) go(k_attn_scores_kv<KT, AT_T, true>, kv);
        else go(k_attn_scores_kv<KT, AT_TD, true>, kv);
    }
}

void launch_softmax(const AttnShape &s, const AttnPlan &p, float *att, const int *pos) {
    if (p.softmax == AP_SMX_WAVE) {   // rows of up to 2048 scores
        const int tcap = sc_terms_cap(s.nmax()), scr = (sc_lds_bytes(s.nmax(), 64) + 15) / 16 * 16;
        const size_t per_wave = 4 * (size_t)tcap + scr;
        const int nrows = s.n_heads * s.ntok;
        hipLaunchKernelGGL((k_attn_softmax_rows<4, SM_V / 2>), dim3((nrows + 3) / 4), dim3(256), 4 * per_wave,
                           kr_stream(), att, s.n_heads, s.max_seq, s.window, pos, nrows, tcap, scr);
        return;
    }
    auto go = [&](auto kern, int threads) {
        hipLaunchKernelGGL(kern, dim3(s.n_heads, 1, s.ntok), dim3(threads), 0, kr_stream(), att, s.max_seq, s.window,
                           pos);
    };
    // 256 threads: the ordered sum's lean form (90 VGPRs against 111: 5 waves a
    // SIMD; 1B-shape 4000-token prompt 64.5k -> 65.5k tok/s)
    if (p.softmax == AP_SMX_256) {
        if (s.window) go(k_attn_softmax<256, 4096, true, true>, 256);
        else go(k_attn_softmax<256, 4096, true, false>, 256);
    } else {
        go(k_attn_softmax<SMX_THREADS, AT_CHUNK, false, true>, SMX_THREADS);
    }
}

template <int KT, int DW, bool WIN>
void launch_mix(const AttnShape &s, const AttnPlan &p, float *ao, const float *att, const KvView &kv, const int *pos) {
    const int group = s.group(), kv_dim = s.n_kv * s.hd;
    if constexpr (DW >= 16) {
        if (p.mix == AP_BLOCK) {   // blocks of MK_W waves' tokens share the V tiles
            const dim3 grid(s.n_kv, (s.hd + DW - 1) / DW, (s.ntok + MK_W * MK_U - 1) / (MK_W * MK_U));
            hipLaunchKernelGGL((k_attn_mix_blk<DW, KT, WIN>), grid, dim3(64 * MK_W), 0, kr_stream(), ao, att, kv, group,
                               s.hd, kv_dim, s.max_seq, s.window, pos, s.ntok);
            return;
        }
    }
    const dim3 grid(s.n_kv, (s.hd + DW - 1) / DW, s.ntok);
    if constexpr (KT == KV_F32)
        hipLaunchKernelGGL(k_attn_mix_batch<DW>, grid, dim3(64), 0, kr_stream(), ao, att, (const float *)kv.v, group,
                           s.hd, kv_dim, s.max_seq, s.window, pos);
    else
        hipLaunchKernelGGL((k_attn_mix_batch_kv<DW, KT>), grid, dim3(64), 0, kr_stream(), ao, att, kv, group, s.hd,
                           kv_dim, s.max_seq, s.window, pos);
}

template <int KT, bool WIN>
void attn_prefill(const AttnShape &s, const AttnPlan &p, float *ao, float *att, const float *q, const KvView &kv,
                  float scale, const int *pos, float cap) {
    launch_scores<KT, WIN>(s, p, att, q, kv, scale, pos);
    if (cap > 0.0f) kr_softcap_scores(att, s.n_heads, s.max_seq, s.window, pos, s.ntok, cap);   // ops/ops.c:141
    launch_softmax(s, p, att, pos);
    if (p.mix == AP_ROWS) {
        const dim3 grid(s.n_kv, s.row_blocks(), s.hd / rb_cw(s.hd));
        rb_switch(s.hd, [&](auto dims) {
            constexpr int HD = decltype(dims)::value;
            hipLaunchKernelGGL((k_attn_mix_rb<HD, KT, WIN>), grid, dim3(4 * rb_cw(HD)), 0, kr_stream(), ao, att, kv,
                               s.group(), s.n_kv * s.hd, s.max_seq, s.window, pos, s.ntok);
        });
    } else {
        switch (s.dw()) {
        case 64: launch_mix<KT, 64, WIN>(s, p, ao, att, kv, pos); break;
        case 32: launch_mix<KT, 32, WIN>(s, p, ao, att, kv, pos); break;
        case 16: launch_mix<KT, 16, WIN>(s, p, ao, att, kv, pos); break;
        case 8: launch_mix<KT, 8, WIN>(s, p, ao, att, kv, pos); break;
        default: launch_mix<KT, 4, WIN>(s, p, ao, att, kv, pos); break;
        }
    }
    kr_check_launch("attention");
}

}   // namespace

void kr_attn_prefill(int kt, float *ao, float *att, const float *q, const KvView &kv, int n_heads, int n_kv_heads,
                     int head_dim, int max_seq, int window, float scale, const int *pos, int ntok, int max_pos,
                     float cap) {
    if (window > max_pos) window = 0;   // none of the tokens reaches its end
    const AttnShape s = { kt, n_heads, n_kv_heads, head_dim, max_seq, window, ntok, max_pos };
    const AttnPlan p = attn_plan(s);
    auto run = [&](auto kt_) {
        constexpr int KT = decltype(kt_)::value;
        if (window) attn_prefill<KT, true>(s, p, ao, att, q, kv, scale, pos, cap);
        else attn_prefill<KT, false>(s, p, ao, att, q, kv, scale, pos, cap);
    };
    if (kt == KV_F32) run(ic<KV_F32>{});
    else if (kt == KV_F16) run(ic<KV_F16>{});
    else run(ic<KV_Q8>{});
}

extern "C" int krh_attention_plan(int kv_type, int n_heads, int n_kv_heads, int head_dim, int max_seq, int window,
                                  int ntok, int last_pos) {
    const int kt = kv_type == ML_F32 ? KV_F32 : kv_type == ML_F16 ? KV_F16 : KV_Q8;
    if (n_kv_heads <= 0 || n_heads <= 0 || n_heads % n_kv_heads || n_heads / n_kv_heads > 16 || head_dim <= 0 ||
        head_dim % 4 || head_dim > 1024 || ntok <= 1 || last_pos < ntok - 1 || last_pos >= max_seq)
        return -1;
    const AttnPlan p = attn_plan({ kt, n_heads, n_kv_heads, head_dim, max_seq, window, ntok, last_pos });
    return p.scores + 4 * p.softmax + 16 * p.mix;
}

extern "C" void krh_set_attn_rb_min(int min_wg) { g_rb_min_wg = min_wg < 0 ? 0 : min_wg; }
