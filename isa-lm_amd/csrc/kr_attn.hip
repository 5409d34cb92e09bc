// Attention over one layer's KV cache for gfx950: scores, softmax and the
// position-ordered mix, for the F32, F16 and Q8 caches (ops/ops.c:124-238,
// kernels/scalar/k_scalar.c:66-77, :111-155), and the F16 / Q8 cache stores
// (model/transformer.c:191-205). Every float operation is the reference's,
// in its order.
#include "kr_attn.h"

namespace {

// out for one KV head's query heads and DW of their dims: lane = (head j of
// the group, dim d), DW = 64 / (group rounded up to a power of two). Each
// lane runs its ordered chain o += a_t * v_t,d (k_scalar.c:119-122). ao is
// written as floats (its quantization happens where it is consumed).
//
// The chain (one dependent add per position) is the bound, so the workgroup
// splits the work by role and keeps the adding wave free of everything else.
// Wave 0 only adds. MX_P producer waves load V and the weights, form the
// products a_t * v_t,d (each the rounded product, as in the scalar loop) and
// hand them over through a ring of three LDS tiles of MX_T positions, laid out
// [lane][position] so that one 16-byte read feeds 4 adds. Producer p owns
// positions [p MX_TH, (p + 1) MX_TH) of every tile and loads them MX_D tiles
// ahead into registers: a lane holds 4 dims of V at one position and the
// weights of every head at that position, and writes its products straight
// into the adder's layout (4-byte writes: the transpose costs no LDS reads).
// LDS bandwidth is what the roles share, so each product crosses LDS once each
// way. One barrier per step hands tiles over: producers write tile s in step
// s; the adder reads tile s into registers in step s + 1 and adds it in step
// s + 2, so no add waits on an LDS read.
// Three producers and the adder: one wave per SIMD of the CU (a fourth
// producer would share the adder's SIMD and slow its chain). The adder, not
// the producers, is the slower side: a tile's 96 dependent adds and its 24
// reads take about 800 cycles, the producers' products and loads 550-700.
// Rows of MX_TS = 100 floats put a 16-lane group's 16-byte reads on 64
// distinct banks.
constexpr int MX_P = 3, MX_TH = 32;                  // producers; their positions per tile
constexpr int MX_T = MX_P * MX_TH, MX_TS = MX_T + 4;   // positions per tile; padded product row

// Slot k of a producer lane: position r of the producer's MX_TH positions and
// first dim c of its 4 dims. Lanes 0-31 and 32-63 take neighbouring dim
// quads of the same 32 positions, so the 32 stores of a half-wave into the
// adder's rows (MX_TS floats apart: 4 quads = 16 banks) hit 32 distinct banks.
static_assert(MX_TH == 32, "the slot map covers 32 positions a slot");
template <int DW>
__device__ __forceinline__ void mx_slot(int k, int lane, int &r, int &c) {
    if (DW >= 8) {
        r = lane & 31;
        c = 4 * (2 * k + (lane >> 5));
    } else {   // one dim quad: lanes 32-63 hold no slot (r >= MX_TH)
        r = lane;
        c = 0;
    }
}

template <int DW, int KT>
__device__ __forceinline__ void attn_mix(float *ao, const float *att, const KvView kv, int group, int hd, int kv_dim,
                                         int max_seq, int window, const int *pos_p) {
    constexpr int GP = 64 / DW;                        // head slots
    constexpr int NV = (MX_TH * DW / 4 + 63) / 64;     // 4-element groups of V per producer lane per tile
    constexpr int ND = KT == KV_Q8 ? NV : 0;           // V row scales per producer lane per tile
    constexpr int PT = Kv4<KT>::REGS * NV + NV * GP + ND;   // registers per tile: V, the weights, the scales
    constexpr int LT = NV + NV * GP + ND;              // loads per tile
    // tiles in flight: within 128 registers and within the 63 loads the wait
    // counter can track (past that every wait would drain it)
    constexpr int DR = 128 / PT < 60 / LT ? 128 / PT : 60 / LT;
    constexpr int MX_D = DR > 8 ? 8 : DR < 2 ? 2 : DR;
    __shared__ __align__(16) float prod[4][64 * MX_TS];   // the ring, and a sink for steps past the end
    int first, n;
    attn_range(pos_p, window, &first, &n);
    const int g = blockIdx.x, c0 = blockIdx.y * DW, lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int j = lane / DW, d = lane % DW;
    const int ntiles = (n + MX_T - 1) / MX_T;
    if (c0 >= hd) {
        // a helper workgroup (grid rows past the head's dim chunks, decode
        // only): it reads one 2-byte word of every 128-byte line of KV head
        // g's V rows and of its query heads' weight rows, earliest positions
        // first, so that they wait in the L2 of this XCD (workgroups are
        // dealt to the 8 XCDs by linear id, so with 8 KV heads per launch
        // row all of head g's workgroups share one) before the producers ask
        constexpr int eb = KT == KV_F32 ? 4 : KT == KV_F16 ? 2 : 1;
        const int lpr = (hd * eb + 127) / 128, nhelp = gridDim.y - (hd + DW - 1) / DW;
        const int hi = (blockIdx.y - (hd + DW - 1) / DW) * (64 * (1 + MX_P)) + threadIdx.x, hn = nhelp * 64 * (1 + MX_P);
        const unsigned char *vb = (const unsigned char *)kv.v + ((size_t)first * kv_dim + (size_t)g * hd) * eb;
        const float *ab = att + (size_t)g * group * max_seq;
        const int vl = n * lpr, al = (n * 4 + 127) / 128;   // V lines; weight-row lines per head
        int sink = 0;
        for (int i = hi; i < vl + group * al; i += hn) {
            if (i < vl) {
                const int t = i / lpr;
                sink ^= *(const unsigned short *)(vb + (size_t)t * kv_dim * eb + (size_t)(i - t * lpr) * 128);
            } else {
                const int h = (i - vl) / al;
                sink ^= *(const unsigned short *)((const unsigned char *)(ab + (size_t)h * max_seq) + (size_t)(i - vl - h * al) * 128);
            }
        }
        if (sink == 0x5bd1 && max_seq < 0) ao[0] = 0.0f;   // keeps the reads (never true)
        return;
    }
    // Steps with a barrier: one per tile the producers write, rounded up to
    // MX_S (every wave runs as many barriers); the adder's last two steps
    // (the last tile's read, the last adds) follow without one. The
    // producers' loop runs in groups of MX_D steps (one per register slot)
    // and may stop after a third (or half) of a group: whole groups ran up
    // to 4 empty steps past the end (the 0.5B shape at 550 positions: 12
    // steps for 8); a test after every step measured no better than one per
    // third.
    constexpr int MX_S = MX_D % 3 == 0 ? MX_D / 3 : MX_D % 2 == 0 ? MX_D / 2 : MX_D;
    const int steps = (ntiles + MX_S - 1) / MX_S * MX_S;
    const size_t q_dim = (size_t)gridDim.x * group * hd;

    if (wave == 0) {
        // the adder: in step s it reads all of tile s - 1 into registers
        // (finished a step earlier) while it adds tile s - 2 from the
        // registers read in step s - 1, so every LDS read has a whole tile
        // of adds to arrive in
        float o = 0.0f;
        auto step = [&](int s, float4 *cur, float4 *nxt, bool bar = true) {
            if (s - 1 >= 0 && s - 1 < ntiles) {
                const float *P = prod[(s - 1) % 3] + lane * MX_TS;
#pragma unroll
                for (int i = 0; i < MX_T / 4; i++) nxt[i] = *(const float4 *)(P + 4 * i);
            }
            const int tile = s - 2;
            if (tile >= 0 && tile < ntiles) {
                const int nt = min(MX_T, n - tile * MX_T);
                if (nt == MX_T) {
#pragma unroll
                    for (int i = 0; i < MX_T / 4; i++) {
                        o = kr_fadd(o, cur[i].x);
                        o = kr_fadd(o, cur[i].y);
                        o = kr_fadd(o, cur[i].z);
                        o = kr_fadd(o, cur[i].w);
                    }
                } else {   // the last, partial tile: only its live steps (a zero would turn -0 to +0)
                    const float *P = prod[tile % 3] + lane * MX_TS;
                    for (int r = 0; r < nt; r++) o = kr_fadd(o, P[r]);
                }
            }
            if (bar) {
                kr_lds_order();
                __syncthreads();
            }
        };
        float4 ta[MX_T / 4], tb[MX_T / 4];
        for (int s = 0; s < steps; s += 2) {
            step(s, ta, tb);
            if (s + 1 < steps) step(s + 1, tb, ta);
        }
        for (int s = steps; s < steps + 2; s++) {   // the producers are done: no barrier
            if (s & 1) step(s, tb, ta, false);
            else step(s, ta, tb, false);
        }
        if (j < group && d < min(DW, hd - c0)) ao[blockIdx.z * q_dim + (size_t)(g * group + j) * hd + c0 + d] = o;
        return;
    }

    // producer p: lane slot k holds V dims c..c+3 at position r of its half
    // tile, and the weights of heads 0..GP-1 at that position
    const int p = wave - 1;
    const int cw = min(DW, hd - c0);   // valid dims of the chunk (a multiple of 4)
    const size_t vb = (size_t)first * kv_dim + (size_t)g * hd + c0;   // element offset of V row `first`
    const float *abase = att + ((size_t)blockIdx.z * gridDim.x * group + (size_t)g * group) * max_seq;
    // Every load is unconditional from an address clamped into the live
    // range (position n - 1, the chunk's last 4 elements, the group's last
    // head, the row's last element): values loaded for positions >= n, dims
    // >= cw or heads >= group only feed products that are never added or
    // stored, and a branch-free loop keeps the loads of MX_D tiles in flight.
    using VT = typename Kv4<KT>::T;
    VT rv[MX_D][NV];
    float ra[MX_D][NV][GP];
    float rd[MX_D][ND > 0 ? ND : 1];   // Q8: the V rows' scales
    auto load = [&](int tile, VT *v, float (*a)[GP], float *dv) {
        const int t0 = min(tile, ntiles - 1) * MX_T + p * MX_TH;
#pragma unroll
        for (int k = 0; k < NV; k++) {
            int r, c;
            mx_slot<DW>(k, lane, r, c);
            r = min(r, MX_TH - 1);
            c = min(c, cw - 4);
            const int t = min(t0 + r, n - 1);
            v[k] = Kv4<KT>::load(kv.v, vb + (size_t)t * kv_dim + c);
            if (KT == KV_Q8) dv[k] = kv.vd[(size_t)(first + t) * kv.n_kv + g];
            const int q = min(t0 + r, max_seq - 1);
#pragma unroll
            for (int jj = 0; jj < GP; jj++) a[k][jj] = abase[(size_t)min(jj, group - 1) * max_seq + q];
        }
    };
    auto products = [&](int tile, const VT *v, const float (*a)[GP], const float *dv) {
        float *P = prod[tile < ntiles ? tile % 3 : 3] + p * MX_TH;
#pragma unroll
        for (int k = 0; k < NV; k++) {
            int r, c;
            mx_slot<DW>(k, lane, r, c);
            if (r < MX_TH) {
                const float4 x = Kv4<KT>::wide(v[k]);
#pragma unroll
                for (int jj = 0; jj < GP; jj++) {
                    // Q8: the weight a_t * dv_t, then its products (k_scalar.c:151-153)
                    const float w = KT == KV_Q8 ? kr_fmul(a[k][jj], dv[k]) : a[k][jj];
                    float *o = P + (jj * DW + c) * MX_TS + r;
                    o[0] = kr_fmul(w, x.x);
                    o[MX_TS] = kr_fmul(w, x.y);
                    o[2 * MX_TS] = kr_fmul(w, x.z);
                    o[3 * MX_TS] = kr_fmul(w, x.w);
                }
            }
        }
        kr_lds_order();
    };
    // in slot order (the loop's waits count on slot 0 being the oldest)
#pragma unroll
    for (int u = 0; u < MX_D; u++) {
        load(u, rv[u], ra[u], rd[u]);
        __builtin_amdgcn_sched_barrier(0);
    }
    for (int s0 = 0; s0 < steps; s0 += MX_D) {
#pragma unroll
        for (int u = 0; u < MX_D; u++) {
            if (u > 0 && u % MX_S == 0 && s0 + u >= steps) break;   // a part group ends the loop
            const int s = s0 + u;   // tile s sits in slot u
            // fenced for the scheduler: a step's products wait on its own
            // slot's loads only
            __builtin_amdgcn_sched_barrier(0);
            products(s, rv[u], ra[u], rd[u]);   // past the end: into the sink, unread
            load(s + MX_D, rv[u], ra[u], rd[u]);
            __builtin_amdgcn_sched_barrier(0);
            __syncthreads();
        }
    }
}

template <int DW>
__global__ void __launch_bounds__(64 * (1 + MX_P)) k_attn_mix(float *ao, const float *att, const float *vc,
                                                              int group, int hd, int kv_dim, int max_seq, int window,
                                                              const int *pos_p) {
    const KvView kv = { nullptr, vc, nullptr, nullptr, 0 };
    attn_mix<DW, KV_F32>(ao, att, kv, group, hd, kv_dim, max_seq, window, pos_p);
}

template <int DW, int KT>
__global__ void __launch_bounds__(64 * (1 + MX_P)) k_attn_mix_kv(float *ao, const float *att, const KvView kv,
                                                                 int group, int hd, int kv_dim, int max_seq,
                                                                 int window, const int *pos_p) {
    attn_mix<DW, KT>(ao, att, kv, group, hd, kv_dim, max_seq, window, pos_p);
}

// ---- decode over a short context: one launch ----

// A query head's whole attention in one workgroup, for rows of scores whose K
// rows fit in LDS together (AS_LDS: 572 positions of 64 dims). The three
// launches of a longer row spend most of such a token on their gaps, their
// loads' latencies and the ordered sum's fixed cost: for 6 heads of 48 dims at
// positions up to 136 they took 14.7 us a layer and two gaps, this launch 6.7.
// It stays the faster up to the longest rows that fit (us a call, three
// launches and this one, F32): 64 dims, 572 positions, 14 or 32 heads 14.4 and
// 14.0; 48 dims, 710 positions 16.8 and 13.7; 128 dims, 292 positions, 32 heads
// 13.3 and 12.0; 256 dims, 140 positions 14.6 and 11.3. K and V are
// loaded together up front; V waits in registers while the scores run from
// K's LDS copy, then its products with the weights take that copy's place.
//   scores: a thread per position, its ordered dot from LDS;
//   softmax: max, exponentials, and their ordered sum one add at a time (the
//     speculative sum's fixed cost is more than these rows' chains);
//   mix: the products a_t * v_t,d by every thread into [position / 4][dim][4]
//     order (the 16-byte reads of a wave's dims are contiguous; each thread
//     stores its 4 dims rotated by its quad's number, which puts the 64
//     stores of a wave on 64 banks), then one lane per dim adds them in
//     position order.
constexpr int AS_NT = 1024, AS_LDS = 152 * 1024;   // threads; bytes of the K copy or the products
constexpr int AS_NP = 10;   // passes over the rows, at most: 4-element loads a thread holds, of K and of V
// positions whose K rows (hd + 4 floats) and products fit
constexpr int as_positions(int hd) {
    return std::min(std::min((AS_LDS / 4 / (hd + 4)) & ~3, AS_NT), AS_NT / (hd / 4) * AS_NP);
}

struct AsLds {
    __align__(16) float kt[AS_LDS / 4];   // K [position][hd + 4], then the products
    __align__(16) float w[AS_NT + 32];    // exponentials, then weights
    __align__(16) float qs[256];
    float red[AS_NT / 64];
    float sum;
    uint64_t xtab[32];
};

// NP: passes of AS_NT / (hd / 4) rows (every load unconditional: the compiler
// then waits for K without waiting for V)
template <int KT, int NP>
__device__ __forceinline__ void attn_short(AsLds &S, float *ao, const float *q, const KvView &kv, int group, int hd,
                                           int kv_dim, float scale, int first, int n) {
    float *kt = S.kt, *w = S.w, *qs = S.qs, *red = S.red;
    const int tid = threadIdx.x, lane = tid & 63, h = blockIdx.x, g = h / group, h4 = hd / 4, ks = hd + 4;
    const int rows = AS_NT / h4, r0 = tid / h4, c = tid - r0 * h4;   // pass u: row u * rows + r0, dims 4c ..
    const bool mine = r0 < rows;                                     // the threads past a pass's rows hold none
    const size_t base = (size_t)first * kv_dim + (size_t)g * hd + 4 * c;
    typename Kv4<KT>::T kr[NP], vr[NP];
#pragma unroll
    for (int u = 0; u < NP; u++) kr[u] = Kv4<KT>::load(kv.k, base + (size_t)min(u * rows + r0, n - 1) * kv_dim);
#pragma unroll
    for (int u = 0; u < NP; u++) vr[u] = Kv4<KT>::load(kv.v, base + (size_t)min(u * rows + r0, n - 1) * kv_dim);
    if (tid < h4) *(float4 *)(qs + 4 * tid) = *(const float4 *)(q + (size_t)h * hd + 4 * tid);
    if (tid >= AS_NT - 32) S.xtab[tid - (AS_NT - 32)] = kr_exp2_tab[tid - (AS_NT - 32)];
#pragma unroll
    for (int u = 0; u < NP; u++)
        if (mine && u * rows + r0 < n) *(float4 *)(kt + (u * rows + r0) * ks + 4 * c) = Kv4<KT>::wide(kr[u]);
    __syncthreads();
    // the score of position tid
    float x = -INFINITY;
    if (tid < n) {
        const float *k = kt + tid * ks;
        float acc = 0.0f;
#pragma unroll 4
        for (int i = 0; i < hd; i += 4) {
            const float4 a = *(const float4 *)(qs + i), b = *(const float4 *)(k + i);
            acc = kr_fadd(acc, kr_fmul(a.x, b.x));
            acc = kr_fadd(acc, kr_fmul(a.y, b.y));
            acc = kr_fadd(acc, kr_fmul(a.z, b.z));
            acc = kr_fadd(acc, kr_fmul(a.w, b.w));
        }
        x = kr_fmul(acc, scale);
    }
    float m = x;
    for (int o = 32; o >= 1; o >>= 1) m = fmaxf(m, __shfl_xor(m, o));
    if (lane == 0) red[tid >> 6] = m;
    __syncthreads();
    m = red[0];
    for (int k = 1; k < AS_NT / 64; k++) m = fmaxf(m, red[k]);
    float e = 0.0f;
    if (tid < n) {
        e = kr_expf_tab(kr_fsub(x, m), S.xtab);
        w[tid] = e;
    }
    __syncthreads();
    if (tid < 64) {   // the ordered sum: every lane the same chain, 4 B terms' reads ahead of their adds
        // B: half as many where 10 passes of floats wait in registers (with all 8
        // the kernel spilled 27 of them)
        constexpr int B = KT == KV_F32 && NP > 5 ? 4 : 8;
        float s = 0.0f;
        int t = 0;
        float4 a[B], b[B];
        auto read = [&](float4 (&v)[B], int t0) {
#pragma unroll
            for (int k = 0; k < B; k++) v[k] = *(const float4 *)(w + min(t0, AS_NT) + 4 * k);
        };
        auto add = [&](const float4 (&v)[B]) {
#pragma unroll
            for (int k = 0; k < B; k++) {
                s = kr_fadd(s, v[k].x);
                s = kr_fadd(s, v[k].y);
                s = kr_fadd(s, v[k].z);
                s = kr_fadd(s, v[k].w);
            }
        };
        read(a, 0);
        for (; t + 8 * B <= n; t += 8 * B) {
            read(b, t + 4 * B);
            __builtin_amdgcn_sched_barrier(0);
            add(a);
            read(a, t + 8 * B);
            __builtin_amdgcn_sched_barrier(0);
            add(b);
        }
        for (; t < n; t++) s = kr_fadd(s, w[t]);
        if (tid == 0) S.sum = s;
    }
    __syncthreads();
    // every score -inf: 1 / n (k_scalar.c:66-77)
    if (tid < n) w[tid] = m == -INFINITY ? kr_fdiv(1.0f, (float)n) : kr_fmul(e, kr_fdiv(1.0f, S.sum));
    __syncthreads();
    // products; position r, dims 4c ..: quad r / 4's floats [dim][r % 4]
    const int rot = (c >> 2) & 3;
#pragma unroll
    for (int u = 0; u < NP; u++) {
        const int r = u * rows + r0;
        if (mine && r < n) {
            const float a = w[r];
            const float4 v = Kv4<KT>::wide(vr[u]);
            const float p0 = kr_fmul(a, v.x), p1 = kr_fmul(a, v.y), p2 = kr_fmul(a, v.z), p3 = kr_fmul(a, v.w);
            // slot k: dim 4c + (k + rot) % 4
            const float a0 = rot & 1 ? p1 : p0, a1 = rot & 1 ? p2 : p1, a2 = rot & 1 ? p3 : p2, a3 = rot & 1 ? p0 : p3;
            float *d = kt + ((size_t)(r >> 2) * hd + 4 * c) * 4 + (r & 3);
            d[4 * (rot & 3)] = rot & 2 ? a2 : a0;
            d[4 * ((1 + rot) & 3)] = rot & 2 ? a3 : a1;
            d[4 * ((2 + rot) & 3)] = rot & 2 ? a0 : a2;
            d[4 * ((3 + rot) & 3)] = rot & 2 ? a1 : a3;
        }
    }
    __syncthreads();
    if (tid < hd) {
        const float4 *p = (const float4 *)kt + tid;   // quad k at p[k * hd]
        const int nq = n >> 2;
        float o = 0.0f;
        float4 a[8], b[8];
        auto read = [&](float4 (&v)[8], int k0) {
#pragma unroll
            for (int k = 0; k < 8; k++) v[k] = p[min(k0 + k, max(nq - 1, 0)) * hd];
        };
        auto add = [&](const float4 (&v)[8]) {
#pragma unroll
            for (int k = 0; k < 8; k++) {
                o = kr_fadd(o, v[k].x);
                o = kr_fadd(o, v[k].y);
                o = kr_fadd(o, v[k].z);
                o = kr_fadd(o, v[k].w);
            }
        };
        int k = 0;
        read(a, 0);
        for (; k + 16 <= nq; k += 16) {
            read(b, k + 8);
            __builtin_amdgcn_sched_barrier(0);
            add(a);
            read(a, k + 16);
            __builtin_amdgcn_sched_barrier(0);
            add(b);
        }
        for (; k < nq; k++) {
            const float4 v = p[k * hd];
            o = kr_fadd(o, v.x);
            o = kr_fadd(o, v.y);
            o = kr_fadd(o, v.z);
            o = kr_fadd(o, v.w);
        }
        const float *tail = (const float *)(p + nq * hd);   // a partial quad's live positions only
        for (int i = 0; i < (n & 3); i++) o = kr_fadd(o, tail[i]);
        ao[(size_t)h * hd + tid] = o;
    }
}

template <int KT>
__global__ void __launch_bounds__(AS_NT) k_attn_short(float *ao, const float *q, const KvView kv, int group, int hd,
                                                      int kv_dim, int window, float scale, const int *pos_p,
                                                      int nmax) {
    __shared__ AsLds S;
    const int pos = *pos_p, first = attn_first(pos, window), n = min(pos + 1 - first, nmax);
    const int np = (n + AS_NT / (hd / 4) - 1) / (AS_NT / (hd / 4));
    if (np <= 2) attn_short<KT, 2>(S, ao, q, kv, group, hd, kv_dim, scale, first, n);
    else if (np <= 5) attn_short<KT, 5>(S, ao, q, kv, group, hd, kv_dim, scale, first, n);
    else attn_short<KT, AS_NP>(S, ao, q, kv, group, hd, kv_dim, scale, first, n);
}

// ---- F16 / Q8 cache rows ----

// store_kv (model/transformer.c:191-205) for the positions *pos0 + t: the
// staging rows k, v [ntok][kv_dim] (the projections' output) into one
// layer's F16 cache (every value rounded to half precision, core/ml.c:39-53)
// or Q8 cache (each KV head's head_dim values with one scale,
// ops/ops.c:81-96). One wave per (KV head, K or V, token).
struct KvOut {
    void *k, *v;
    float *kd, *vd;
    int n_kv;
};

template <int KT>
__global__ void __launch_bounds__(64) k_store_kv(const KvOut o, const float *k, const float *v, int kv_dim, int hd,
                                                 const int *pos0) {
    const int h = blockIdx.x, which = blockIdx.y, t = blockIdx.z, lane = threadIdx.x;
    const float *x = (which ? v : k) + (size_t)t * kv_dim + (size_t)h * hd;
    const size_t at = (size_t)(*pos0 + t) * kv_dim + (size_t)h * hd;
    if (KT == KV_F16) {
        uint16_t *dst = (uint16_t *)(which ? o.v : o.k) + at;
        for (int i = lane; i < hd; i += 64) dst[i] = kr_f2h(x[i]);
        return;
    }
    int8_t *dst = (int8_t *)(which ? o.v : o.k) + at;
    float m = 0.0f;
    for (int i = lane; i < hd; i += 64) m = fmaxf(m, fabsf(x[i]));
    for (int sh = 32; sh >= 1; sh >>= 1) m = fmaxf(m, __shfl_xor(m, sh));
    const bool zero = m < KR_QUANT_TINY;
    const float id = zero ? 0.0f : kr_fdiv(127.0f, m);
    for (int i = lane; i < hd; i += 64) dst[i] = zero ? (int8_t)0 : (int8_t)kr_q8_elem(x[i], id);
    if (lane == 0) (which ? o.vd : o.kd)[(size_t)(*pos0 + t) * o.n_kv + h] = zero ? 0.0f : kr_fdiv(m, 127.0f);
}

// The one-launch kernels, then a token's three launches, first and together in
// the code object. A token's launches hold more code than the instruction cache, so
// where this code and a process's buffers lie moves the 8B shape's attention
// block by up to 0.9 us: over the performance cases in one process this order
// took 41.1 us (the block's projections in another object, 47.6 the 1B shape's
// Q8 block), the three launches first 42.0 (47.9); alone in a process 41.0 to
// 41.4 and 41.4 to 41.9.
template __global__ void k_attn_short<KV_F32>(float *, const float *, const KvView, int, int, int, int, float, const int *,
                                              int);
template __global__ void k_attn_short<KV_F16>(float *, const float *, const KvView, int, int, int, int, float, const int *,
                                              int);
template __global__ void k_attn_scores<AT_TD, false>(float *, const float *, const float *, int, int, int, int, int, float,
                                                     const int *);
template __global__ void k_attn_softmax<SMX_THREADS, AT_CHUNK, false, false>(float *, int, int, const int *);
template __global__ void k_attn_mix<16>(float *, const float *, const float *, int, int, int, int, int, const int *);
template __global__ void k_attn_mix<8>(float *, const float *, const float *, int, int, int, int, int, const int *);
template __global__ void k_attn_mix<32>(float *, const float *, const float *, int, int, int, int, int, const int *);
template __global__ void k_attn_mix<64>(float *, const float *, const float *, int, int, int, int, int, const int *);

}   // namespace

// ---- C ABI ----

template <int KT, int DW>
static void launch_mix(const dim3 &grid, float *ao, const float *att, const KvView &kv, int group, int hd, int kv_dim,
                       int max_seq, int window, const int *pos) {
    // helper rows fill the chip (about 256 workgroups in all)
    const int rows = grid.x ? 256 / (int)grid.x : 0;
    const dim3 hgrid(grid.x, rows > (int)grid.y ? rows : grid.y, 1);
    if constexpr (KT == KV_F32)
        hipLaunchKernelGGL(k_attn_mix<DW>, hgrid, dim3(64 * (1 + MX_P)), 0, kr_stream(), ao, att, (const float *)kv.v,
                           group, hd, kv_dim, max_seq, window, pos);
    else
        hipLaunchKernelGGL((k_attn_mix_kv<DW, KT>), hgrid, dim3(64 * (1 + MX_P)), 0, kr_stream(), ao, att, kv, group,
                           hd, kv_dim, max_seq, window, pos);
}

// scores, softmax and mix of ntok positions *pos + t over one layer's cache
// of type KT; max_pos (the last position) sizes the launch
template <int KT>
static void attention(float *ao, float *att, const float *q, const KvView &kv, int n_heads, int n_kv_heads,
                      int head_dim, int max_seq, int window, float scale, const int *pos, int ntok, int max_pos,
                      float cap = 0.0f) {
    if (n_kv_heads <= 0 || n_heads % n_kv_heads || head_dim % 4 || (n_heads * head_dim) % KR_QK ||
        n_heads / n_kv_heads > 16 || head_dim > 1024 || max_seq < 4) {
        kr_fail(ML_E_SHAPE, "attention shape", hipSuccess);
        return;
    }
    const int group = n_heads / n_kv_heads, kv_dim = n_kv_heads * head_dim;
    if constexpr (KT != KV_Q8) {   // decode whose rows, at most this long, run in one launch
        const int rows = window && window <= max_pos ? window : max_pos + 1;
        if (ntok == 1 && cap <= 0.0f && head_dim <= 256 && rows <= as_positions(head_dim)) {
            hipLaunchKernelGGL(k_attn_short<KT>, dim3(n_heads), dim3(AS_NT), 0, kr_stream(), ao, q, kv, group,
                               head_dim, kv_dim, window, scale, pos, rows);
            kr_check_launch("attention");
            return;
        }
    }
    const int tt = attn_tile<KT>(group, head_dim);
    if (!tt) {
        kr_fail(ML_E_SHAPE, "attention: head_dim too large for the score tile", hipSuccess);
        return;
    }
    if (ntok > 1) {
        kr_attn_prefill(KT, ao, att, q, kv, n_heads, n_kv_heads, head_dim, max_seq, window, scale, pos, ntok, max_pos,
                        cap);
        return;
    }
    const size_t lds = attn_tile_lds<KT>(group, head_dim, tt);
    const dim3 sgrid(n_kv_heads, (max_pos + tt) / tt, 1);
    auto gokv = [&](auto kern) {
        hipLaunchKernelGGL(kern, sgrid, dim3(AT_THREADS), lds, kr_stream(), att, q, kv, group, head_dim, kv_dim,
                           max_seq, window, scale, pos);
    };
    if constexpr (KT == KV_Q8) {
        gokv(k_attn_scores_q8<false>);
    } else if constexpr (KT == KV_F32) {   // tiles of AT_TD positions
        const dim3 dgrid(n_kv_heads, (max_pos + AT_TD) / AT_TD, 1);
        hipLaunchKernelGGL((k_attn_scores<AT_TD, false>), dgrid, dim3(AT_THREADS),
                           attn_tile_lds<KT>(group, head_dim, AT_TD), kr_stream(), att, q, (const float *)kv.k, group,
                           head_dim, kv_dim, max_seq, window, scale, pos);
    } else {
        if (tt == AT_T) gokv(k_attn_scores_kv<KT, AT_T, false>);
        else gokv(k_attn_scores_kv<KT, AT_TD, false>);
    }
    if (cap > 0.0f) kr_softcap_scores(att, n_heads, max_seq, window, pos, 1, cap);   // ops/ops.c:141
    hipLaunchKernelGGL((k_attn_softmax<SMX_THREADS, AT_CHUNK, false, false>), dim3(n_heads), dim3(SMX_THREADS), 0,
                       kr_stream(), att, max_seq, window, pos);
    const int gp = group <= 1 ? 1 : group <= 2 ? 2 : group <= 4 ? 4 : group <= 8 ? 8 : 16;
    const int dw = 64 / gp;
    const dim3 grid(n_kv_heads, (head_dim + dw - 1) / dw, 1);
    switch (dw) {
    case 64: launch_mix<KT, 64>(grid, ao, att, kv, group, head_dim, kv_dim, max_seq, window, pos); break;
    case 32: launch_mix<KT, 32>(grid, ao, att, kv, group, head_dim, kv_dim, max_seq, window, pos); break;
    case 16: launch_mix<KT, 16>(grid, ao, att, kv, group, head_dim, kv_dim, max_seq, window, pos); break;
    case 8: launch_mix<KT, 8>(grid, ao, att, kv, group, head_dim, kv_dim, max_seq, window, pos); break;
    default: launch_mix<KT, 4>(grid, ao, att, kv, group, head_dim, kv_dim, max_seq, window, pos); break;
    }
    kr_check_launch("attention");
}

static KvView f32_view(const float *kc, const float *vc) {
    KvView v = { kc, vc, nullptr, nullptr, 0 };
    return v;
}

extern "C" void krh_attention(float *ao, int8_t *aq, float *ad, float *att, const float *q, const float *kc,
                              const float *vc, int n_heads, int n_kv_heads, int head_dim, int max_seq, int window,
                              float scale, const int *pos) {
    attention<KV_F32>(ao, att, q, f32_view(kc, vc), n_heads, n_kv_heads, head_dim, max_seq, window, scale, pos, 1,
                      max_seq - 1);
    if (aq) krh_quantize_q8(aq, ad, ao, n_heads * head_dim, 1);
}

// ---- decode attention without a workspace argument ----
//
// The score rows live in one file-scope device array, `scratch`, of
// KRH_ATTN_SCRATCH_FLOATS floats (8 MiB), which each device holds for the
// life of the process. Host code never passes the array's name to a kernel
// (on the host it only names a stand-in): its device address, one per device,
// comes from hipGetSymbolAddress at set-up (kr_attn_setup, from krh_init).
// Every call on a device shares that device's array, so calls that overlap on
// one device race. No entry of it needs clearing: each call writes every
// score row entry it reads back.
static __device__ __align__(256) float scratch[KRH_ATTN_SCRATCH_FLOATS];
static float *g_scratch_ptr[KR_MAX_DEVICES];

ml_status kr_attn_setup(int dev) {
    if (dev < 0 || dev >= KR_MAX_DEVICES) return ML_E_ISA;
    if (g_scratch_ptr[dev]) return ML_OK;
    void *ptr = nullptr;
    const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !ptr) {
        kr_fail(ML_E_ISA, "hipGetSymbolAddress(scratch)", e);
        return ML_E_ISA;
    }
    g_scratch_ptr[dev] = (float *)ptr;
    return ML_OK;
}

extern "C" void krh_attention_noalloc(float *ao, const float *q, const float *kc, const float *vc, int n_heads,
                                      int n_kv_heads, int head_dim, int max_seq, int window, float scale,
                                      const int *pos) {
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= KR_MAX_DEVICES || !g_scratch_ptr[dev]) {
        kr_fail(ML_E_ISA, "attention_noalloc: the device's scratch address is not set up (krh_init)", hipSuccess);
        return;
    }
    if (n_heads <= 0 || max_seq <= 0 || (size_t)n_heads * (size_t)max_seq > (size_t)KRH_ATTN_SCRATCH_FLOATS) {
        kr_fail(ML_E_SHAPE, "attention_noalloc: n_heads * max_seq exceeds the static scratch of "
                            "KRH_ATTN_SCRATCH_FLOATS floats", hipSuccess);
        return;
    }
    attention<KV_F32>(ao, g_scratch_ptr[dev], q, f32_view(kc, vc), n_heads, n_kv_heads, head_dim, max_seq, window,
                      scale, pos, 1, max_seq - 1);
}

extern "C" int krh_attention_short(int head_dim, int kv_type) {
    return head_dim > 0 && head_dim <= 256 && head_dim % 4 == 0 && kv_type != ML_Q8_0 ? as_positions(head_dim) : 0;
}

extern "C" void krh_attention_batch(float *ao, float *att, const float *q, const float *kc, const float *vc,
                                    int n_heads, int n_kv_heads, int head_dim, int max_seq, int window, float scale,
                                    const int *pos0, int ntok, int last_pos) {
    if (ntok <= 0 || last_pos >= max_seq) {
        kr_fail(ML_E_SHAPE, "attention batch shape", hipSuccess);
        return;
    }
    attention<KV_F32>(ao, att, q, f32_view(kc, vc), n_heads, n_kv_heads, head_dim, max_seq, window, scale, pos0, ntok,
                      last_pos);
}

extern "C" void krh_attention_kv(float *ao, float *att, const float *q, const ml_kv_layer *kv, int n_heads,
                                 int n_kv_heads, int head_dim, int max_seq, float scale, const int *pos0, int ntok,
                                 int last_pos) {
    krh_attention_kv_softcap(ao, att, q, kv, n_heads, n_kv_heads, head_dim, max_seq, scale, pos0, ntok, last_pos, 0.0f);
}

extern "C" void krh_attention_kv_softcap(float *ao, float *att, const float *q, const ml_kv_layer *kv, int n_heads,
                                         int n_kv_heads, int head_dim, int max_seq, float scale, const int *pos0,
                                         int ntok, int last_pos, float cap) {
    if (ntok <= 0 || last_pos >= max_seq || !kv) {
        kr_fail(ML_E_SHAPE, "attention shape", hipSuccess);
        return;
    }
    if (kv->k && kv->v) {
        attention<KV_F32>(ao, att, q, f32_view(kv->k, kv->v), n_heads, n_kv_heads, head_dim, max_seq, kv->window,
                          scale, pos0, ntok, last_pos, cap);
    } else if (kv->kh && kv->vh) {
        KvView v = { kv->kh, kv->vh, nullptr, nullptr, n_kv_heads };
        attention<KV_F16>(ao, att, q, v, n_heads, n_kv_heads, head_dim, max_seq, kv->window, scale, pos0, ntok,
                          last_pos, cap);
    } else if (kv->kq && kv->vq && kv->kd && kv->vd) {
        KvView v = { kv->kq, kv->vq, kv->kd, kv->vd, n_kv_heads };
        attention<KV_Q8>(ao, att, q, v, n_heads, n_kv_heads, head_dim, max_seq, kv->window, scale, pos0, ntok,
                         last_pos, cap);
    } else {
        kr_fail(ML_E_SHAPE, "attention: the cache view has no F32, F16 or Q8 rows", hipSuccess);
    }
}

extern "C" void krh_attention_q8_store(float *ao, float *att, const float *q, const ml_kv_layer *kv,
                                       const float *k_row, const float *v_row, int n_heads, int n_kv_heads,
                                       int head_dim, int max_seq, float scale, const int *pos) {
    if (!kv || !kv->kq || !kv->vq || !kv->kd || !kv->vd || !k_row || !v_row) {
        kr_fail(ML_E_SHAPE, "attention_q8_store: a Q8 cache view and the staging rows", hipSuccess);
        return;
    }
    KvView v = { kv->kq, kv->vq, kv->kd, kv->vd, n_kv_heads, k_row, v_row };
    attention<KV_Q8>(ao, att, q, v, n_heads, n_kv_heads, head_dim, max_seq, kv->window, scale, pos, 1, max_seq - 1);
}

extern "C" void krh_store_kv(int kv_type, void *kc, void *vc, float *kd, float *vd, const float *k, const float *v,
                             int n_kv_heads, int head_dim, const int *pos0, int ntok) {
    if (ntok <= 0 || n_kv_heads <= 0 || head_dim <= 0 || head_dim % 4 || !kc || !vc ||
        (kv_type == ML_Q8_0 && (!kd || !vd)) || (kv_type != ML_Q8_0 && kv_type != ML_F16)) {
        kr_fail(ML_E_SHAPE, "store_kv: an F16 or Q8 cache and its shape", hipSuccess);
        return;
    }
    const dim3 grid(n_kv_heads, 2, ntok);
    const int kv_dim = n_kv_heads * head_dim;
    KvOut o = { kc, vc, kd, vd, n_kv_heads };
    if (kv_type == ML_F16)
        hipLaunchKernelGGL(k_store_kv<KV_F16>, grid, dim3(64), 0, kr_stream(), o, k, v, kv_dim, head_dim, pos0);
    else
        hipLaunchKernelGGL(k_store_kv<KV_Q8>, grid, dim3(64), 0, kr_stream(), o, k, v, kv_dim, head_dim, pos0);
    kr_check_launch("store_kv");
}

