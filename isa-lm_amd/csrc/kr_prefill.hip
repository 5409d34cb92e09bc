// Batched prompt prefill on gfx950: the matrix products as int8 MFMA.
//
// Y[t][r] = sum over blocks b, in block order, of ((float)S * wd[r][b]) * xd[t][b]
// where S = the exact int32 dot of block b of weight row r with block b of
// token t's Q8_0 activation: the scalar kernel's float order for every token
// (kernels/scalar/k_scalar.c:4-37, ops/ops.c:51-73), so each token's result is
// bit-identical to the decode matvec's (model/transformer.c:381-384).
//
// One v_mfma_i32_32x32x32_i8 computes S for a 32-token x 32-row tile and one
// block (K = 32 = one Q8_0 block). Operand lanes (checked on the device):
// lane l supplies A[l % 32][16 (l / 32) .. +15] and B[16 (l / 32) .. +15][l % 32];
// result register r of lane l is C[8 (r / 4) + 4 (l / 32) + r % 4][l % 32].
// A = the tokens' activations, B = the weight rows, so each lane holds one
// weight row (one scale per block) and 16 tokens, whose scales come from the
// transposed activation scales xdT[b][t] through the workgroup's LDS tile. The
// per-block rescale and the ordered accumulation are 3 VALU operations per
// output and block (f32 scales: 4), which bound the kernel, not the MFMA.
#include <algorithm>
#include "kr_internal.h"
#include "kr_numerics.h"

namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));

struct MMat {
    const uint8_t *q;
    const void *d;
    int rows, cols, type, d16;
};

enum { MM_STORE = 0, MM_ADD = 1, MM_QKV = 2, MM_SWIGLU = 3 };

struct MmArgs {
    MMat w[3];
    int tile0[4];        // first workgroup of matrix i; tile0[nmat] = grid size
    int nmat;
    const int8_t *xq;    // [T][K] (rows up to the padded token count readable)
    const float *xdT;    // activation scale of block b of token t: xdT[b * xsb + t * xst]
    int ldx;             // T rounded up to MM_TT: xq's readable rows
    int xsb, xst;        // transposed [K / 32][ldx]: ldx and 1; token rows [T][K / 32]: 1 and K / 32
    int T, K;
    float *y[3];         // y[i][t * ldy[i] + r]
    int ldy[3];
    const float *bias[3];
    const float *rope_cos, *rope_sin;
    int head_dim, pos0;
    int form;            // MmForm
    int8_t *hq;          // MM_SWIGLU: h's Q8_0 quants [T][rows] and scales [rows / 32][ldx]
    float *hdT;
};

// the 16 signed quant bytes of elements 16h .. 16h + 15 of a Q4 block: byte p
// holds element p (low nibble) and p + 16 (high); nibble n is weight n - 8:
// (n | 0x80) - 8 never borrows across bytes, and ^ 0x80 then leaves n - 8 as
// a signed byte
__device__ __forceinline__ v4i q4_frag(const v4i v, int h) {
    const unsigned sh = 4u * (unsigned)h, M = 0x0F0F0F0Fu;
    v4i r;
#pragma unroll
    for (int i = 0; i < 4; i++)
        r[i] = (int)((((((unsigned)v[i] >> sh) & M) | 0x80808080u) - 0x08080808u) ^ 0x80808080u);
    return r;
}

// f16 scales: the MFMA's accumulator starts at the bits of the float
// M = 1.5 * 2^23, so a result register holds the bits of the float M + S
// exactly (|S| <= 32 * 128 * 127 < 2^22), and fl(S * wd) is one
// fma(M + S, wd, -M * wd): -M * wd is exact (3 times an 11-bit scale), so the
// fma's exact value is S * wd and it rounds once, as the product does. (S = 0
// gives +0 where the product has wd's sign; a sum that starts from +0 cannot
// tell.) That takes the conversion out: 3 VALU operations an output and block
// instead of 4. An infinite scale is the one value it does not hold for: the
// FAST loops collect the scales' largest magnitude, and a workgroup that met
// an infinity sums its tile again with the conversion. f32 scales (M * wd
// would round) always convert.
constexpr int MM_MAGIC = 0x4B400000;      // the bits of M
constexpr float MM_M = 12582912.0f;
__device__ __forceinline__ v16i mm_magic() {
    constexpr int m = MM_MAGIC;
    return v16i{ m, m, m, m, m, m, m, m, m, m, m, m, m, m, m, m };
}

constexpr int MM_TT = 128;   // tokens per workgroup

// The kernels of a launch, by the rows x tokens of a workgroup. 16 x 64 and
// 32 x 64: k_matmul_short;
// 64 x 128 and 128 x 128: k_matmul, or k_matmul_ring for short reductions.
// A SwiGLU pair takes half a tile's rows from each matrix.
enum MmForm { MF_16, MF_32, MF_64, MF_128, MF_RING_64, MF_RING_128, MF_FORMS };
__host__ __device__ constexpr int mf_rows(int f) {
    return f == MF_16 ? 16 : f == MF_32 ? 32 : f == MF_64 || f == MF_RING_64 ? 64 : 128;
}
__host__ __device__ constexpr int mf_tokens(int f) { return f <= MF_32 ? 64 : MM_TT; }

template <int D16> struct MmScale { using T = uint32_t; };
template <> struct MmScale<1> { using T = uint16_t; };

// Where matrix mi's sums go, read once before the epilogue (read in mm_emit,
// the compiler selected the argument's address and each of a lane's 16 to 64
// sums waited for its own scalar loads: 1 us of a 14336 x 64 product's 6.3
// with 100 tokens)
struct MmOut {
    float *y;
    const float *bias;
    int mi, rows, ldy;
};
__device__ __forceinline__ MmOut mm_out(const MmArgs &a, int mi, int rows) {
    MmOut o = { a.y[0], a.bias[0], mi, rows, a.ldy[0] };
    if (mi == 1) o = { a.y[1], a.bias[1], mi, rows, a.ldy[1] };
    if (mi == 2) o = { a.y[2], a.bias[2], mi, rows, a.ldy[2] };
    return o;
}

// The sum of row `row` and token t, stored as the launch asks; lanes 2 i and
// 2 i + 1 hold neighbouring rows of one token.
template <int EPI>
__device__ __forceinline__ void mm_emit(const MmArgs &a, const MmOut &out, int row, int t, float v) {
    const bool rin = row < out.rows;
    if (EPI == MM_QKV) {
        // bias (model/transformer.c:276-277), then RoPE on q and k
        // (k_scalar.c:79-94): rows 2i, 2i+1 sit in lanes 2i, 2i+1
        if (out.bias && rin) v = kr_fadd(v, out.bias[row]);
        const float o = __shfl_xor(v, 1);
        if (out.mi < 2) {
            const int hd = a.head_dim, j = row % hd, h2 = hd >> 1;
            const int pos = a.pos0 + (t < a.T ? t : 0);
            const float c = a.rope_cos[(size_t)pos * h2 + (j >> 1)];
            const float sn = a.rope_sin[(size_t)pos * h2 + (j >> 1)];
            v = (j & 1) == 0 ? kr_fsub(kr_fmul(v, c), kr_fmul(o, sn)) : kr_fadd(kr_fmul(o, sn), kr_fmul(v, c));
        }
    }
    if (rin && t < a.T) {
        float *p = out.y + (size_t)t * out.ldy + row;
        if (EPI == MM_ADD) *p = kr_fadd(*p, v);
        else *p = v;
    }
}

// The sums of a wave over 32 x 32 tiles: lane = one row (32 g + lane % 32),
// tokens 8 (r / 4) + 4 (lane / 32) + r % 4 of the wave's 32
template <int EPI, int NG>
__device__ __forceinline__ void mm_finish(const MmArgs &a, int mi, int rows, int rowl, int tokl,
                                          const float (&acc)[NG][16], int lane) {
    if constexpr (EPI == MM_SWIGLU) {
        // h = silu(w1 x) * (w3 x) (k_scalar.c:96-98), then its Q8_0 in blocks
        // of 32 rows (k_scalar.c:39-57): a block's 32 values are the 32 lanes
        // of a half-wave (the first NG / 2 groups: w1 rows; the rest: the same w3 rows)
#pragma unroll
        for (int g = 0; g < NG / 2; g++) {
            const int row = rowl + 32 * g + (lane & 31);
            const bool bin = rowl + 32 * g < rows;   // rows % 32 == 0: whole blocks in or out
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int t = tokl + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
                const float h1 = acc[g][r], h3 = acc[g + NG / 2][r];
                const float v = kr_fmul(kr_fdiv(h1, kr_fadd(1.0f, kr_expf(-h1))), h3);
                int8_t q;
                float d;
                kr_quant_block32(v, &q, &d);
                if (bin && t < a.T) {
                    a.hq[(size_t)t * rows + row] = q;
                    if ((lane & 31) == 0) a.hdT[(size_t)(row >> 5) * a.ldx + t] = d;
                }
            }
        }
    } else {
        const MmOut out = mm_out(a, mi, rows);
#pragma unroll
        for (int g = 0; g < NG; g++)
#pragma unroll
            for (int r = 0; r < 16; r++)
                mm_emit<EPI>(a, out, rowl + 32 * g + (lane & 31), tokl + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3),
                             acc[g][r]);
    }
}

// ---- 128- and 64-row tiles: MM_SB blocks a stage ----
//
// A stage is MM_SB = 4 blocks: 128 bytes of every weight and token row, so
// the 8 lanes that load a row's stage use whole cache lines at once. (One
// block a step, the 32 bytes of 32 rows a load instruction touched cost 4
// times the lines, and the L1 could not keep them until the next block.) Rows
// are 144 bytes apart in LDS: the 16-byte fragment reads of 16 consecutive
// rows then fall on distinct banks. Two stages alternate, one barrier each;
// the next stage's loads are in flight while a stage is summed.
constexpr int MM_SB = 4, MM_RC = 2 * MM_SB + 1;   // blocks a stage; 16-byte chunks a staged row (one of padding)

template <int NG, int D16>
struct MmStage {
    v4i w[32 * NG][MM_RC];
    v4i x[MM_TT][MM_RC];
    float xs[MM_SB][MM_TT];                    // token scales
    typename MmScale<D16>::T d[32 * NG][MM_SB];   // raw weight scales
};

// a thread's share of a stage in registers
template <int QT, int NG>
struct MmPre {
    v4i w[QT == ML_Q8_0 ? NG : NG / 2], x[4];
    uint32_t d[NG / 2];
    float xs[2];
};

// wave-uniform bases of the tile's operands at block 0 (w, d: of the first
// and, for a SwiGLU pair, the second half's matrix) and this thread's byte
// offsets from them
template <int NG>
struct MmTile {
    const uint8_t *w[2], *d[2], *xs, *x;
    uint32_t wo[NG], so[NG / 2], xo, xso, xstep;
    size_t xsb;
    int nb;
};

template <int QT, int D16, int NG, bool PAIR>
__device__ __forceinline__ MmTile<NG> mm_tile(const MmArgs &a, const MMat &W, const MMat &W2, int nb, int rowl,
                                              int tok0, int tid) {
    constexpr int BB = QT == ML_Q8_0 ? 32 : 16, SB = D16 ? 2 : 4;
    MmTile<NG> t;
    const size_t blk = (size_t)rowl * nb;
    t.w[0] = W.q + blk * BB;
    t.w[1] = (PAIR ? W2.q : W.q) + blk * BB;
    t.d[0] = (const uint8_t *)W.d + blk * SB;
    t.d[1] = (const uint8_t *)(PAIR ? W2.d : W.d) + blk * SB;
    if (PAIR && NG == 2 && __builtin_amdgcn_readfirstlane(tid >> 6) >= 2) {
        // a 64-row pair's second 32 rows in the loads that take 64 rows at once
        if (QT != ML_Q8_0) t.w[0] = t.w[1];
        t.d[0] = t.d[1];
    }
    // rows past the end re-read the last row (not stored)
    auto row = [&](int r) { return (uint32_t)(min(rowl + (PAIR ? r & (16 * NG - 1) : r), W.rows - 1) - rowl); };
#pragma unroll
    for (int u = 0; u < NG; u++)   // Q8: 8 threads a row; Q4: 4
        t.wo[u] = QT == ML_Q8_0 ? row((tid >> 3) + 32 * u) * nb * BB : row((tid >> 2) + 64 * (u & (NG / 2 - 1))) * nb * BB;
#pragma unroll
    for (int u = 0; u < NG / 2; u++) t.so[u] = row((tid >> 2) + 64 * u) * nb * SB;
    t.xs = (const uint8_t *)(a.xdT + (size_t)tok0 * a.xst);
    t.xso = (uint32_t)(min(tok0 + (tid & (MM_TT - 1)), a.T - 1) - tok0) * a.xst * 4;
    t.xsb = (size_t)a.xsb * 4;
    t.x = (const uint8_t *)a.xq + (size_t)tok0 * a.K;   // readable: the caller pads to ldx rows
    t.xo = (uint32_t)(tid >> 3) * a.K;
    t.xstep = 32u * a.K;
    t.nb = nb;
    return t;
}

// the stage at block b0; blocks past the last re-read the last (unused)
template <int QT, int D16, int NG, bool PAIR>
__device__ __forceinline__ void mm_load(MmPre<QT, NG> &R, const MmTile<NG> &t, int b0, int tid) {
    const int left = t.nb - b0;
    const uint32_t c8 = 16 * min(tid & 7, 2 * left - 1), c4 = min(tid & 3, left - 1);
    if constexpr (QT == ML_Q8_0) {
#pragma unroll
        for (int u = 0; u < NG; u++) R.w[u] = *(const v4i *)(t.w[PAIR && u >= NG / 2] + (size_t)b0 * 32 + (t.wo[u] + c8));
    } else {
#pragma unroll
        for (int u = 0; u < NG / 2; u++) R.w[u] = *(const v4i *)(t.w[PAIR && u] + (size_t)b0 * 16 + (t.wo[u] + 16 * c4));
    }
#pragma unroll
    for (int u = 0; u < 4; u++) R.x[u] = *(const v4i *)(t.x + (size_t)b0 * 32 + (size_t)u * t.xstep + (t.xo + c8));
#pragma unroll
    for (int u = 0; u < NG / 2; u++) {
        const uint8_t *d = t.d[PAIR && u] + (size_t)b0 * (D16 ? 2 : 4);
        R.d[u] = D16 ? (uint32_t)*(const uint16_t *)(d + (t.so[u] + 2 * c4)) : *(const uint32_t *)(d + (t.so[u] + 4 * c4));
    }
#pragma unroll
    for (int u = 0; u < 2; u++)
        R.xs[u] = *(const float *)(t.xs + (size_t)(b0 + min((tid >> 7) + 2 * u, left - 1)) * t.xsb + t.xso);
}

template <int QT, int D16, int NG>
__device__ __forceinline__ void mm_put(MmStage<NG, D16> &L, const MmPre<QT, NG> &R, int tid) {
    if constexpr (QT == ML_Q8_0) {
#pragma unroll
        for (int u = 0; u < NG; u++) L.w[(tid >> 3) + 32 * u][tid & 7] = R.w[u];
    } else {
#pragma unroll
        for (int u = 0; u < NG / 2; u++) {
            L.w[(tid >> 2) + 64 * u][2 * (tid & 3)] = q4_frag(R.w[u], 0);
            L.w[(tid >> 2) + 64 * u][2 * (tid & 3) + 1] = q4_frag(R.w[u], 1);
        }
    }
#pragma unroll
    for (int u = 0; u < 4; u++) L.x[(tid >> 3) + 32 * u][tid & 7] = R.x[u];
#pragma unroll
    for (int u = 0; u < NG / 2; u++) L.d[(tid >> 2) + 64 * u][tid & 3] = (typename MmScale<D16>::T)R.d[u];
#pragma unroll
    for (int u = 0; u < 2; u++) L.xs[(tid >> 7) + 2 * u][tid & (MM_TT - 1)] = R.xs[u];
}

// where a lane reads a block's operands in a stage; stepped from block to
// block, the row groups at constant offsets
template <int D16>
struct MmAt {
    const v4i *w, *x;
    const float4 *xs;
    const typename MmScale<D16>::T *d;
    __device__ __forceinline__ void next() {
        w += 2;
        x += 2;
        xs += MM_TT / 4;
        d += 1;
    }
};

// the next block of a stage for the wave's 32 tokens
template <int D16, int NG, bool FAST>
__device__ __forceinline__ void mm_block(float (&acc)[NG][16], float &mx, const v16i &s0, const MmAt<D16> &p) {
    const v4i xa = *p.x;
    v4i wb[NG];
    uint32_t wdr[NG];
#pragma unroll
    for (int g = 0; g < NG; g++) {
        wb[g] = p.w[32 * MM_RC * g];
        wdr[g] = p.d[32 * MM_SB * g];
    }
    float xd[16];
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const float4 v = p.xs[2 * q];   // tokens 8 q + 4 hf .. + 3
        xd[4 * q] = v.x;
        xd[4 * q + 1] = v.y;
        xd[4 * q + 2] = v.z;
        xd[4 * q + 3] = v.w;
    }
    v16i s = __builtin_amdgcn_mfma_i32_32x32x32_i8(xa, wb[0], s0, 0, 0, 0), sn = s;
#pragma unroll
    for (int g = 0; g < NG; g++) {
        float wd = D16 ? kr_h2f((uint16_t)wdr[g]) : __uint_as_float(wdr[g]);
        float c = 0.0f;
        if constexpr (FAST) {
            asm volatile("" : "+v"(wd));   // a register: no fma_mix from the half
            mx = fmaxf(mx, fabsf(wd));
            c = kr_fmul(-MM_M, wd);
        }
        __builtin_amdgcn_sched_barrier(0);
        if (g + 1 < NG) sn = __builtin_amdgcn_mfma_i32_32x32x32_i8(xa, wb[g + 1], s0, 0, 0, 0);
#pragma unroll
        for (int h = 0; h < 16; h += 8) {
            float t[8];
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int r = 0; r < 8; r++) t[r] = FAST ? __builtin_fmaf(__int_as_float(s[h + r]), wd, c) : kr_fmul((float)s[h + r], wd);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int r = 0; r < 8; r++) t[r] = kr_fmul(t[r], xd[h + r]);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int r = 0; r < 8; r++) acc[g][h + r] = kr_fadd(acc[g][h + r], t[r]);
        }
        __builtin_amdgcn_sched_barrier(0);
        s = sn;
    }
}

template <int QT, int D16, int NG, bool PAIR, bool FAST>
__device__ __forceinline__ float mm_sums(float (&acc)[NG][16], MmStage<NG, D16> *L, const MmTile<NG> &t, int tid) {
    const int wave = tid >> 6, lane = tid & 63, nb = t.nb;
    v16i s0 = FAST ? mm_magic() : v16i{};
    if constexpr (FAST) asm volatile("" : "+v"(s0));
    float mx = 0.0f;
#pragma unroll
    for (int g = 0; g < NG; g++)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[g][r] = 0.0f;
    MmPre<QT, NG> R;
    mm_load<QT, D16, NG, PAIR>(R, t, 0, tid);
    mm_put<QT, D16, NG>(L[0], R, tid);
    __syncthreads();
    int st = 0;
    for (int b0 = 0; b0 < nb; b0 += MM_SB) {
        const bool more = b0 + MM_SB < nb;
        mm_load<QT, D16, NG, PAIR>(R, t, more ? b0 + MM_SB : b0, tid);   // unconditional: past the end unused
        __builtin_amdgcn_sched_barrier(0);
        const int n = min(MM_SB, nb - b0);
        const int ln = lane & 31, hf = lane >> 5, tk = 32 * wave;
        MmAt<D16> p = { &L[st].w[ln][hf], &L[st].x[tk + ln][hf], (const float4 *)&L[st].xs[0][tk + 4 * hf],
                        &L[st].d[ln][0] };
#pragma unroll 1
        for (int blk = 0; blk < n; blk++) {
            mm_block<D16, NG, FAST>(acc, mx, s0, p);
            p.next();
        }
        st ^= 1;
        mm_put<QT, D16, NG>(L[st], R, tid);
        __syncthreads();
    }
    return mx;
}

// ---- 16-row tiles: short prompts ----
//
// When the grid of 64-row tiles leaves CUs idle, a workgroup takes 16 rows
// (RG groups of them) x 64 tokens, a wave 16 tokens of all its rows, one
// v_mfma_i32_16x16x32_i8 per row group and block: a lane holds one weight row
// and 4 tokens, so the sums' chains are a quarter as long as with the
// 32 x 32 form and a short batch still has rows / 16 workgroups. A stage is 8
// blocks (256 bytes of every row: whole cache lines), staged through two LDS
// buffers and loaded 2 stages ahead in a register ring. (4 stages ahead took all
// 256 VGPRs, spilled, and were 3 to 6% slower from 2048 to 4096 columns, 1% at
// 14336.)
constexpr int MS_SB = 8, MS_TT = 64;             // blocks a stage, tokens a workgroup
constexpr int MS_D = 2;                          // stages ahead (even)
constexpr int MS_RC = 2 * MS_SB + 1;             // 16-byte chunks a staged row (one of padding)

template <int RG, int D16>
struct MsStage {
    v4i w[16 * RG][MS_RC];
    v4i x[MS_TT][MS_RC];
    float xs[MS_SB][MS_TT];
    __align__(16) typename MmScale<D16>::T d[16 * RG][MS_SB];
};

template <int QT, int RG>
struct MsPre {
    static constexpr int NW = QT == ML_Q8_0 ? RG : (RG + 1) / 2, ND = (RG + 1) / 2;
    v4i w[NW], x[4];
    uint32_t d[ND];
    float xs[2];
};

template <int QT, int RG>
struct MsTile {
    const uint8_t *w, *d, *xs, *x;
    uint32_t wo[MsPre<QT, RG>::NW], so[MsPre<QT, RG>::ND], xo[4], xso;
    size_t xsb;
    int nb;
};

template <int QT, int D16, int RG>
__device__ __forceinline__ MsTile<QT, RG> ms_tile(const MmArgs &a, const MMat &W, int nb, int rowl, int tok0, int tid) {
    constexpr int BB = QT == ML_Q8_0 ? 32 : 16, SB = D16 ? 2 : 4;
    MsTile<QT, RG> t;
    const size_t blk = (size_t)rowl * nb;
    t.w = W.q + blk * BB;
    t.d = (const uint8_t *)W.d + blk * SB;
    // rows past the end re-read the last row, tokens past it the last token (not stored)
    auto row = [&](int r) { return (uint32_t)(min(rowl + (r & (16 * RG - 1)), W.rows - 1) - rowl); };
#pragma unroll
    for (int u = 0; u < MsPre<QT, RG>::NW; u++)   // Q8: 16 threads a row; Q4: 8
        t.wo[u] = row(QT == ML_Q8_0 ? (tid >> 4) + 16 * u : (tid >> 3) + 32 * u) * nb * BB;
#pragma unroll
    for (int u = 0; u < MsPre<QT, RG>::ND; u++) t.so[u] = row((tid >> 3) + 32 * u) * nb * SB;
    t.x = (const uint8_t *)a.xq + (size_t)tok0 * a.K;
#pragma unroll
    for (int u = 0; u < 4; u++) t.xo[u] = (uint32_t)(min(tok0 + (tid >> 4) + 16 * u, a.T - 1) - tok0) * a.K;
    t.xs = (const uint8_t *)(a.xdT + (size_t)tok0 * a.xst);
    t.xso = (uint32_t)(min(tok0 + (tid & (MS_TT - 1)), a.T - 1) - tok0) * a.xst * 4;
    t.xsb = (size_t)a.xsb * 4;
    t.nb = nb;
    return t;
}

// the stage at block b0 (one past the last: the last stage again); blocks past the last re-read the last (unused)
template <int QT, int D16, int RG>
__device__ __forceinline__ void ms_load(MsPre<QT, RG> &R, const MsTile<QT, RG> &t, int b, int tid) {
    const int b0 = min(b, (t.nb - 1) / MS_SB * MS_SB), left = t.nb - b0;
    const uint32_t c16 = 16 * min(tid & 15, 2 * left - 1), c8 = min(tid & 7, left - 1);
#pragma unroll
    for (int u = 0; u < MsPre<QT, RG>::NW; u++)
        R.w[u] = QT == ML_Q8_0 ? *(const v4i *)(t.w + (size_t)b0 * 32 + (t.wo[u] + c16))
                               : *(const v4i *)(t.w + (size_t)b0 * 16 + (t.wo[u] + 16 * c8));
#pragma unroll
    for (int u = 0; u < 4; u++) R.x[u] = *(const v4i *)(t.x + (size_t)b0 * 32 + (t.xo[u] + c16));
#pragma unroll
    for (int u = 0; u < MsPre<QT, RG>::ND; u++) {
        const uint8_t *d = t.d + (size_t)b0 * (D16 ? 2 : 4);
        R.d[u] = D16 ? (uint32_t)*(const uint16_t *)(d + (t.so[u] + 2 * c8)) : *(const uint32_t *)(d + (t.so[u] + 4 * c8));
    }
#pragma unroll
    for (int u = 0; u < 2; u++)
        R.xs[u] = *(const float *)(t.xs + (size_t)(b0 + min((tid >> 6) + 4 * u, left - 1)) * t.xsb + t.xso);
}

template <int QT, int D16, int RG>
__device__ __forceinline__ void ms_put(MsStage<RG, D16> &L, const MsPre<QT, RG> &R, int tid) {
#pragma unroll
    for (int u = 0; u < MsPre<QT, RG>::NW; u++) {
        if constexpr (QT == ML_Q8_0) {
            L.w[(tid >> 4) + 16 * u][tid & 15] = R.w[u];
        } else if ((tid >> 3) + 32 * u < 16 * RG) {   // RG 1: half of the threads
            L.w[(tid >> 3) + 32 * u][2 * (tid & 7)] = q4_frag(R.w[u], 0);
            L.w[(tid >> 3) + 32 * u][2 * (tid & 7) + 1] = q4_frag(R.w[u], 1);
        }
    }
#pragma unroll
    for (int u = 0; u < 4; u++) L.x[(tid >> 4) + 16 * u][tid & 15] = R.x[u];
#pragma unroll
    for (int u = 0; u < MsPre<QT, RG>::ND; u++)
        if ((tid >> 3) + 32 * u < 16 * RG) L.d[(tid >> 3) + 32 * u][tid & 7] = (typename MmScale<D16>::T)R.d[u];
#pragma unroll
    for (int u = 0; u < 2; u++) L.xs[(tid >> 6) + 4 * u][tid & (MS_TT - 1)] = R.xs[u];
}

// blocks b0 .. b0 + NB - 1 of a stage for the wave's 16 tokens: every read,
// then every MFMA, then the rescales, so that one wave a SIMD still overlaps
// the latencies
template <int D16, int RG, bool FAST, int NB>
__device__ __forceinline__ void ms_blocks(float (&acc)[RG][4], float &mx, const v4i &s0, const MsStage<RG, D16> &L,
                                          int b0, int wave, int lane) {
    const int ln = lane & 15, q = lane >> 4;
    const long *xp = (const long *)&L.x[16 * wave + ln][2 * b0] + q;
    const long *wp = (const long *)&L.w[ln][2 * b0] + q;
    const float4 *xv = (const float4 *)&L.xs[b0][16 * wave + 4 * q];
    float4 xd[NB];
    float wd[NB][RG], c[NB][RG];
    v4i s[NB][RG];
#pragma unroll
    for (int b = 0; b < NB; b++) {
        const long xa = xp[4 * b];
        xd[b] = xv[b * (MS_TT / 4)];
#pragma unroll
        for (int g = 0; g < RG; g++) {
            const uint32_t wdr = L.d[16 * g + ln][b0 + b];
            wd[b][g] = D16 ? kr_h2f((uint16_t)wdr) : __uint_as_float(wdr);
            s[b][g] = __builtin_amdgcn_mfma_i32_16x16x32_i8(xa, wp[2 * 16 * MS_RC * g + 4 * b], s0, 0, 0, 0);
        }
    }
#pragma unroll
    for (int b = 0; b < NB; b++)
#pragma unroll
        for (int g = 0; g < RG; g++) {
            if constexpr (FAST) {
                asm volatile("" : "+v"(wd[b][g]));   // a register: no fma_mix from the half
                mx = fmaxf(mx, fabsf(wd[b][g]));
                c[b][g] = kr_fmul(-MM_M, wd[b][g]);
            }
        }
#pragma unroll
    for (int b = 0; b < NB; b++) {
        const float x4[4] = { xd[b].x, xd[b].y, xd[b].z, xd[b].w };
#pragma unroll
        for (int g = 0; g < RG; g++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const float t = FAST ? __builtin_fmaf(__int_as_float(s[b][g][r]), wd[b][g], c[b][g])
                                     : kr_fmul((float)s[b][g][r], wd[b][g]);
                acc[g][r] = kr_fadd(acc[g][r], kr_fmul(t, x4[r]));
            }
    }
}

template <int D16, int RG, bool FAST>
__device__ __forceinline__ void ms_stage(float (&acc)[RG][4], float &mx, const v4i &s0, const MsStage<RG, D16> &L,
                                         int n, int wave, int lane) {
    constexpr int NB = 4;
    if (n >= MS_SB) {
#pragma unroll
        for (int b = 0; b < MS_SB; b += NB) ms_blocks<D16, RG, FAST, NB>(acc, mx, s0, L, b, wave, lane);
    } else {
#pragma unroll 1
        for (int b = 0; b < n; b++) ms_blocks<D16, RG, FAST, 1>(acc, mx, s0, L, b, wave, lane);
    }
}

template <int QT, int D16, int RG, bool FAST>
__device__ __forceinline__ float ms_sums(float (&acc)[RG][4], MsStage<RG, D16> *L, const MsTile<QT, RG> &t, bool live,
                                         int tid) {
    const int wave = tid >> 6, lane = tid & 63, nb = t.nb;
    constexpr int m = FAST ? MM_MAGIC : 0;
    v4i s0 = v4i{ m, m, m, m };
    if constexpr (FAST) asm volatile("" : "+v"(s0));
    float mx = 0.0f;
#pragma unroll
    for (int g = 0; g < RG; g++)
#pragma unroll
        for (int r = 0; r < 4; r++) acc[g][r] = 0.0f;
    MsPre<QT, RG> R[MS_D];   // stage k sits in R[k % MS_D] until it is put
#pragma unroll
    for (int k = 0; k < MS_D; k++) ms_load<QT, D16, RG>(R[k], t, k * MS_SB, tid);
    ms_put<QT, D16, RG>(L[0], R[0], tid);
    ms_load<QT, D16, RG>(R[0], t, MS_D * MS_SB, tid);
    __syncthreads();
    // step k: stage k is summed from buffer k % 2 while stage k + 1 goes into
    // the other (its last reader was step k - 1) and stage k + 1 + MS_D is
    // loaded; every wave reaches every barrier
    for (int b0 = 0; b0 < nb; b0 += MS_D * MS_SB) {
#pragma unroll
        for (int k = 0; k < MS_D; k++) {
            const int b = b0 + k * MS_SB, k1 = (k + 1) % MS_D;
            ms_put<QT, D16, RG>(L[(k + 1) & 1], R[k1], tid);
            ms_load<QT, D16, RG>(R[k1], t, b + (MS_D + 1) * MS_SB, tid);
            __builtin_amdgcn_sched_barrier(0);
            if (live) ms_stage<D16, RG, FAST>(acc, mx, s0, L[k & 1], nb - b, wave, lane);
            __syncthreads();
        }
    }
    return mx;
}

template <int EPI, int QT, int D16, int RG>
__global__ void __launch_bounds__(256, 2) k_matmul_short(const MmArgs a) {
    __shared__ MsStage<RG, D16> L[2];
    int mi = 0;
    while (mi + 1 < a.nmat && (int)blockIdx.x >= a.tile0[mi + 1]) mi++;
    const MMat W = mi == 0 ? a.w[0] : (mi == 1 ? a.w[1] : a.w[2]);
    const int ntt = (a.T + MS_TT - 1) / MS_TT;
    const int local = (int)blockIdx.x - a.tile0[mi];
    const int rt = local / ntt, tt = local - rt * ntt;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int rowl = rt * 16 * RG, tokl = tt * MS_TT + 16 * wave;
    const MsTile<QT, RG> t = ms_tile<QT, D16, RG>(a, W, a.K / KR_QK, rowl, tt * MS_TT, tid);
    const bool live = __builtin_amdgcn_readfirstlane(tokl) < a.T;
    float acc[RG][4];
    if constexpr (D16) {
        const float mx = ms_sums<QT, 1, RG, true>(acc, L, t, live, tid);
        if (__syncthreads_or(mx == __builtin_inff())) ms_sums<QT, 1, RG, false>(acc, L, t, live, tid);
    } else {
        ms_sums<QT, 0, RG, false>(acc, L, t, live, tid);
    }
    const MmOut out = mm_out(a, mi, W.rows);
#pragma unroll
    for (int g = 0; g < RG; g++)
#pragma unroll
        for (int r = 0; r < 4; r++)
            mm_emit<EPI>(a, out, rowl + 16 * g + (lane & 15), tokl + 4 * (lane >> 4) + r, acc[g][r]);
}

// Workgroup = 4 waves over a 32 NG-row x 128-token tile; wave w takes all the
// tile's rows (NG row groups) and tokens 32 w .. 32 w + 31, NG 32x32x32 MFMAs a
// block.
template <int EPI, int QT, int D16, int NG>
__global__ void __launch_bounds__(256, 2) k_matmul(const MmArgs a) {
    constexpr int TT = MM_TT;
    __shared__ MmStage<NG, D16> L[2];
    int mi = 0;
    while (mi + 1 < a.nmat && (int)blockIdx.x >= a.tile0[mi + 1]) mi++;
    const MMat W = mi == 0 ? a.w[0] : (mi == 1 ? a.w[1] : a.w[2]);
    const int ntt = (a.T + TT - 1) / TT;
    const int local = (int)blockIdx.x - a.tile0[mi];
    const int rt = local / ntt, tt = local - rt * ntt;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    constexpr bool PAIR = EPI == MM_SWIGLU;   // 16 NG rows of w1 and the same of w3
    const int rowl = rt * (PAIR ? 16 : 32) * NG, tokl = tt * TT + 32 * wave;
    const int nb = a.K / KR_QK;
    float acc[NG][16];
    const MmTile<NG> t = mm_tile<QT, D16, NG, PAIR>(a, W, a.w[1], nb, rowl, tt * TT, tid);
    if constexpr (D16) {
        // every wave of the workgroup sees the tile's rows: one vote for all
        const float mx = mm_sums<QT, 1, NG, PAIR, true>(acc, L, t, tid);
        if (__syncthreads_or(mx == __builtin_inff())) mm_sums<QT, 1, NG, PAIR, false>(acc, L, t, tid);
    } else {
        mm_sums<QT, 0, NG, PAIR, false>(acc, L, t, tid);
    }

    mm_finish<EPI, NG>(a, mi, W.rows, rowl, tokl, acc, lane);
}

// ---- 128- and 64-row tiles of a short reduction: one block a stage ----
//
// A reduction of few blocks never fills k_matmul's pipeline: its stages of 4
// blocks cost the first one's whole latency, and their 80 KB leave a CU two
// workgroups to overlap it (and the stores of the sums) with. Here a stage is one
// block in an LDS ring of 3: 12 KB and 146 VGPRs, 3 waves a SIMD. On the other
// side of the line its 32 bytes a row and load cost 4 times the cache lines.
// 128-row tiles, 14336 rows and 700 tokens: 288 columns 21.8 us against
// k_matmul's 26.5, 896 columns 47.0 against 48.0, 2048 columns 101 against 97.
struct MrX {
    v4i xa;              // the wave's 32 tokens
};

// Per thread and block, for the workgroup's tile: 16 quant bytes of weight
// row tid / 2 (half tid % 2, Q4 unpacked to n - 8), that row's raw scale, and
// the scale of the workgroup's token tid % 128.
struct MrW {
    v4i w;
    uint32_t d;
    float xs;
};

constexpr int MR_ST = 3;   // LDS ring stages of the weight tile

template <int NG>
struct MrLds {
    v4i w[MR_ST][32 * NG][2];     // [stage][row][half]
    uint32_t d[MR_ST][32 * NG];   // [stage][row] raw scale bits
    float xs[MR_ST][MM_TT];       // [stage][token] the tokens' scales
};

__device__ __forceinline__ void mr_load_x(MrX &f, const MmArgs &a, int b, int tokl, int lane) {
    const int t = tokl + (lane & 31);   // readable: the caller pads the activations to ldx rows
    f.xa = *(const v4i *)(a.xq + (size_t)t * a.K + (size_t)b * 32 + 16 * (lane >> 5));
}

// thread tid loads half tid % 2 of tile row (tid / 2) mod 32 NG (NG 2: the
// second half of the threads repeats a row's load, which keeps every load
// unconditional, and does not store it); xcol: the scales of this thread's token,
// clamped to the last. PAIR: the tile's first half are rows rowl.. of W,
// the second the same rows of W2 (SwiGLU's w1 and w3).
template <int QT, int D16, int NG, bool PAIR>
__device__ __forceinline__ void mr_load(MrW &R, const MMat &W, const MMat &W2, const float *xcol, int xsb, int nb,
                                        int b, int rowl, int tid) {
    const int tr = (tid >> 1) & (32 * NG - 1);
    const int r = min(rowl + (PAIR ? tr & (16 * NG - 1) : tr), W.rows - 1);   // rows past the end re-read the last (not stored)
    const size_t blk = (size_t)r * nb + b;
    const bool second = PAIR && tr >= 16 * NG;
    const uint8_t *wq = (second ? W2.q : W.q) + blk * (QT == ML_Q8_0 ? 32 : 16);
    const void *wd = second ? W2.d : W.d;
    R.w = QT == ML_Q8_0 ? *(const v4i *)(wq + 16 * (tid & 1)) : q4_frag(*(const v4i *)wq, tid & 1);
    R.d = D16 ? (uint32_t)((const uint16_t *)wd)[blk] : ((const uint32_t *)wd)[blk];
    R.xs = xcol[(size_t)b * xsb];
}

template <int NG>
__device__ __forceinline__ void mr_put(MrLds<NG> &L, int st, const MrW &R, int tid) {
    if (tid < MM_TT) L.xs[st][tid] = R.xs;
    if ((tid >> 1) >= 32 * NG) return;
    L.w[st][tid >> 1][tid & 1] = R.w;
    if ((tid & 1) == 0) L.d[st][tid >> 1] = R.d;
}

// Row group g + 1's MFMA is issued after the whole rescale of group g: an
// empty asm takes every rescaled value of group g as input and the MFMA's
// weight operand as in-out, so only one 16-register result set is live (left
// to itself the compiler holds NG of them: 183 VGPRs, 2 waves a SIMD).
template <int D16, int NG>
__device__ __forceinline__ void mr_step(float (&acc)[NG][16], const MrX &f, const MrLds<NG> &L, int st, int lane,
                                        int tokw) {
    const int ln = lane & 31, hf = lane >> 5;
    v4i wb[NG];
    uint32_t wdr[NG];
#pragma unroll
    for (int g = 0; g < NG; g++) {
        wb[g] = L.w[st][32 * g + ln][hf];
        wdr[g] = L.d[st][32 * g + ln];
    }
    float xd[16];
    const float4 *xv = (const float4 *)&L.xs[st][tokw + 4 * hf];
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const float4 v = xv[2 * q];   // tokens 8 q + 4 hf .. + 3
        xd[4 * q] = v.x;
        xd[4 * q + 1] = v.y;
        xd[4 * q + 2] = v.z;
        xd[4 * q + 3] = v.w;
    }
    v16i s = __builtin_amdgcn_mfma_i32_32x32x32_i8(f.xa, wb[0], v16i{}, 0, 0, 0);
#pragma unroll
    for (int g = 0; g < NG; g++) {
        const float wd = D16 ? kr_h2f((uint16_t)wdr[g]) : __uint_as_float(wdr[g]);
#pragma unroll
        for (int r = 0; r < 16; r++)
            acc[g][r] = kr_fadd(acc[g][r], kr_fmul(kr_fmul((float)s[r], wd), xd[r]));
        if (g + 1 < NG) {
            v4i w = wb[g + 1];
#pragma unroll
            for (int r = 0; r < 16; r++) asm volatile("" : "+v"(w) : "v"(acc[g][r]));
            s = __builtin_amdgcn_mfma_i32_32x32x32_i8(f.xa, w, v16i{}, 0, 0, 0);
        }
    }
}

// The workgroup's threads load each block's weight tile and its scales once
// (16 bytes and one scale per thread) into the LDS ring: block b + 1 is stored
// during step b into the stage step b - 2 read, and the barrier closing each
// step orders those stores before step b + 1 reads them.
template <int EPI, int QT, int D16, int NG>
__global__ void __launch_bounds__(256, 3) k_matmul_ring(const MmArgs a) {
    __shared__ MrLds<NG> L;
    int mi = 0;
    while (mi + 1 < a.nmat && (int)blockIdx.x >= a.tile0[mi + 1]) mi++;
    const MMat W = mi == 0 ? a.w[0] : (mi == 1 ? a.w[1] : a.w[2]);
    const int ntt = (a.T + MM_TT - 1) / MM_TT;
    const int local = (int)blockIdx.x - a.tile0[mi];
    const int rt = local / ntt, tt = local - rt * ntt;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    constexpr bool PAIR = EPI == MM_SWIGLU;   // 16 NG rows of w1 and the same of w3
    const int rowl = rt * (PAIR ? 16 : 32) * NG, tokl = tt * MM_TT + 32 * wave;
    const int nb = a.K / KR_QK;
    const float *xcol = a.xdT + (size_t)min(tt * MM_TT + (tid & (MM_TT - 1)), a.T - 1) * a.xst;
    float acc[NG][16];
#pragma unroll
    for (int g = 0; g < NG; g++)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[g][r] = 0.0f;
    // Loads are unconditional (block indices past the end re-read the last
    // block, unused): a load issued on only one path makes the wait-count
    // pass drain every in-flight load at the loop head, which would cancel
    // the prefetch. Only the odd tail's step is conditional; every thread
    // reaches every barrier.
    const int bl = nb - 1;
    MrW R;
    MrX x0, x1;
    auto load = [&](int b) { mr_load<QT, D16, NG, PAIR>(R, W, a.w[1], xcol, a.xsb, nb, min(b, bl), rowl, tid); };
    load(0);
    mr_put(L, 0, R, tid);
    load(1);
    mr_load_x(x0, a, 0, tokl, lane);
    mr_load_x(x1, a, min(1, bl), tokl, lane);
    __syncthreads();
    int st = 0;   // stage of block b
    for (int b = 0; b < nb; b += 2) {
        const int s1 = st == MR_ST - 1 ? 0 : st + 1, s2 = s1 == MR_ST - 1 ? 0 : s1 + 1;
        mr_put(L, s1, R, tid);
        load(b + 2);
        mr_step<D16, NG>(acc, x0, L, st, lane, 32 * wave);
        mr_load_x(x0, a, min(b + 2, bl), tokl, lane);
        __syncthreads();
        mr_put(L, s2, R, tid);
        load(b + 3);
        if (b + 1 < nb) mr_step<D16, NG>(acc, x1, L, s1, lane, 32 * wave);
        mr_load_x(x1, a, min(b + 3, bl), tokl, lane);
        __syncthreads();
        st = s2;
    }
    mm_finish<EPI, NG>(a, mi, W.rows, rowl, tokl, acc, lane);
}

template <int EPI>
void launch_mm(const MmArgs &a, const MMat &W) {
    const int grid = a.tile0[a.nmat];
    if (a.K % KR_QK || a.T <= 0 || grid <= 0 || a.ldx % MM_TT || a.T > a.ldx || a.xsb <= 0 || a.xst <= 0) {
        kr_fail(ML_E_SHAPE, "matmul shape", hipSuccess);
        return;
    }
    auto run = [&](auto qt, auto d16) {
        constexpr int QT = decltype(qt)::value, D16 = decltype(d16)::value;
        auto go = [&](auto kern) { hipLaunchKernelGGL(kern, dim3(grid), dim3(256), 0, kr_stream(), a); };
        if constexpr (EPI != MM_SWIGLU) {
            if (a.form == MF_16) return go(k_matmul_short<EPI, QT, D16, 1>);
            if (a.form == MF_32) return go(k_matmul_short<EPI, QT, D16, 2>);
        }
        if (a.form == MF_64) return go(k_matmul<EPI, QT, D16, 2>);
        if (a.form == MF_128) return go(k_matmul<EPI, QT, D16, 4>);
        if (a.form == MF_RING_64) return go(k_matmul_ring<EPI, QT, D16, 2>);
        go(k_matmul_ring<EPI, QT, D16, 4>);
    };
    using std::integral_constant;
    if (W.type == ML_Q8_0) {
        if (W.d16) run(integral_constant<int, ML_Q8_0>{}, integral_constant<int, 1>{});
        else run(integral_constant<int, ML_Q8_0>{}, integral_constant<int, 0>{});
    } else {
        if (W.d16) run(integral_constant<int, ML_Q4_0>{}, integral_constant<int, 1>{});
        else run(integral_constant<int, ML_Q4_0>{}, integral_constant<int, 0>{});
    }
    kr_check_launch("matmul");
}

MMat to_mmat(const krh_mat *m) {
    MMat k = { (const uint8_t *)m->q, m->d, m->rows, m->cols, m->type, m->d16 };
    return k;
}

// The form of a launch: the one with the least estimated time on this device,
//   rounds * (fixed + K / 32 * alone) + (n - rounds) * K / 32 * shared + n * tile   (us),
// n the workgroups of the fullest CU, which holds `resident` of them at a time:
// the first of a round takes `alone` a block of 32 columns, each of the others
// adds `shared`, and each stores its tile. Larger tiles load less per sum, smaller
// ones make more workgroups. The constants are fitted to the choice, over krh_matmul
// and krh_matmul_swiglu with every form timed at 11 heights from 288 to 14336
// rows, 7 reductions from 288 to 14336 columns and 19 batches from 2 to 2047
// tokens (Q8 and Q4, f16 and f32 scales): over those 3914 sizes it costs 0.2%
// more than the best form of each. Some of its lines (us, the call alone):
// 16-row tiles 13.3 and 32-row ones 10.6 (896 x 896, 700 tokens), 7.0 and 8.6 (64
// tokens); 64-row tiles 63 and 128-row ones 86 (14336 x 4096, 256 tokens), 122
// and 106 (511 tokens); SwiGLU 14336 x 288, 300 tokens: rings 35, k_matmul 47;
// 4864 x 2048, 511 tokens: 76 and 69.
struct MmCost {
    int resident;
    float fixed, alone, shared, tile;
};
constexpr MmCost MF_COST[MF_FORMS] = {
    { 3, 3.3f, 0.076f, 0.089f, 0.38f }, { 2, 4.0f, 0.18f, 0.06f, 0.026f }, { 2, 3.3f, 0.49f, 0.025f, 1.1f },
    { 2, 6.2f, 0.7f, 0.13f, 1.5f }, { 4, 6.3f, 0.53f, 0.2f, 0.15f }, { 3, 2.6f, 1.2f, 0.32f, 0.79f },
};
constexpr MmCost MF_PAIR_COST[MF_FORMS] = {
    {}, {}, { 2, 19.0f, 0.3f, 0.097f, 0.13f }, { 2, 29.0f, 0.47f, 0.21f, 2.0f },
    { 4, 14.0f, 0.62f, 0.23f, 0.56f }, { 3, 30.0f, 0.51f, 0.48f, 1.6f },
};

int mm_form(int nmat, const int *rows, int K, int T, bool pair) {
    const int cus = krh_device_cus() > 0 ? krh_device_cus() : 256;
    const float nb = (float)(K / KR_QK);
    int best = MF_64;
    float least = INFINITY;
    for (int f = pair ? MF_64 : MF_16; f < MF_FORMS; f++) {
        const int per = mf_rows(f) / (pair ? 2 : 1);
        long wgs = 0;
        for (int i = 0; i < nmat; i++) wgs += (long)((rows[i] + per - 1) / per) * ((T + mf_tokens(f) - 1) / mf_tokens(f));
        const MmCost &c = (pair ? MF_PAIR_COST : MF_COST)[f];
        const long nl = (wgs + cus - 1) / cus;
        const float n = (float)nl, rounds = (float)((nl + c.resident - 1) / c.resident);
        const float t = rounds * (c.fixed + nb * c.alone) + (n - rounds) * nb * c.shared + n * c.tile;
        if (t < least) {
            least = t;
            best = f;
        }
    }
    return best;
}

void mm_plan(MmArgs &a, int nmat, const int *rows, bool pair = false) {
    a.form = mm_form(nmat, rows, a.K, a.T, pair);
    const int per = mf_rows(a.form) / (pair ? 2 : 1), ntt = (a.T + mf_tokens(a.form) - 1) / mf_tokens(a.form);
    a.tile0[0] = 0;
    for (int i = 0; i < nmat; i++) a.tile0[i + 1] = a.tile0[i] + (rows[i] + per - 1) / per * ntt;
}

// ---- per-token work of a batched step ----

// h = silu(g) * u (k_scalar.c:96-98) for ntok rows of n, then Q8_0 of h
// into q [t][n] and the transposed scales dT[b * ldd + t].
__global__ void __launch_bounds__(256) k_silu_quant(int8_t *q, float *dT, int ldd, const float *g, const float *u,
                                                    int n) {
    const size_t t = blockIdx.y;
    const int i = blockIdx.x * 1024 + 4 * threadIdx.x;
    if (i >= n) return;   // n % 32 == 0
    const float4 gv = *(const float4 *)(g + t * n + i), uv = *(const float4 *)(u + t * n + i);
    float4 v;
    v.x = kr_fmul(kr_fdiv(gv.x, kr_fadd(1.0f, kr_expf(-gv.x))), uv.x);
    v.y = kr_fmul(kr_fdiv(gv.y, kr_fadd(1.0f, kr_expf(-gv.y))), uv.y);
    v.z = kr_fmul(kr_fdiv(gv.z, kr_fadd(1.0f, kr_expf(-gv.z))), uv.z);
    v.w = kr_fmul(kr_fdiv(gv.w, kr_fadd(1.0f, kr_expf(-gv.w))), uv.w);
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
    *(int *)(q + t * n + i) = packed;
    if ((i & 31) == 0) dT[(size_t)(i >> 5) * ldd + t] = dd;
}

__global__ void k_embed_batch(float *x, const MMat e, const int *tok, float scale) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x, t = blockIdx.y;
    if (i >= e.cols) return;
    const int nb = e.cols / KR_QK, row = tok[t], b = i / KR_QK, j = i % KR_QK;
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
    x[(size_t)t * e.cols + i] = o;
}

}  // namespace

// ---- C ABI ----

extern "C" int krh_matmul_form(int rows, int cols, int ntok, int swiglu) {
    return rows > 0 && cols > 0 && ntok > 0 ? mm_form(1, &rows, cols, ntok, swiglu != 0) : -1;
}

extern "C" void krh_matmul_swiglu(int8_t *hq, float *hdT, const krh_mat *w1, const krh_mat *w3, const int8_t *xq,
                                  const float *xdT, int ldx, int T) {
    if (!hq || !hdT || w1->rows != w3->rows || w1->cols != w3->cols || w1->type != w3->type || w1->d16 != w3->d16 ||
        w1->rows % KR_QK) {
        kr_fail(ML_E_SHAPE, "matmul_swiglu: w1 and w3 of one shape, type and scale width, rows % 32 == 0",
                hipSuccess);
        return;
    }
    MmArgs a = {};
    a.w[0] = to_mmat(w1);
    a.w[1] = to_mmat(w3);
    a.nmat = 1;
    a.xq = xq;
    a.xdT = xdT;
    a.ldx = ldx;
    a.xsb = ldx;
    a.xst = 1;
    a.T = T;
    a.K = w1->cols;
    a.hq = hq;
    a.hdT = hdT;
    mm_plan(a, 1, &w1->rows, true);
    launch_mm<MM_SWIGLU>(a, a.w[0]);
}

// one matrix over T tokens; the scales' strides say their layout
static void matmul_one(float *Y, int ldy, const krh_mat *W, const int8_t *xq, const float *xd, int ldx, int T,
                       int accumulate, int xsb, int xst) {
    MmArgs a = {};
    a.w[0] = to_mmat(W);
    a.nmat = 1;
    a.xq = xq;
    a.xdT = xd;
    a.ldx = ldx;
    a.xsb = xsb;
    a.xst = xst;
    a.T = T;
    a.K = W->cols;
    a.y[0] = Y;
    a.ldy[0] = ldy;
    mm_plan(a, 1, &W->rows);
    if (accumulate) launch_mm<MM_ADD>(a, a.w[0]);
    else launch_mm<MM_STORE>(a, a.w[0]);
}

extern "C" void krh_matmul(float *Y, int ldy, const krh_mat *W, const int8_t *xq, const float *xdT, int ldx, int T,
                           int accumulate) {
    matmul_one(Y, ldy, W, xq, xdT, ldx, T, accumulate, ldx, 1);
}

extern "C" void krh_matmul_rows(float *Y, int ldy, const krh_mat *W, const int8_t *xq, const float *xd, int ldx,
                                int T, int accumulate) {
    matmul_one(Y, ldy, W, xq, xd, ldx, T, accumulate, 1, W->cols / KR_QK);
}

// k and v go to the F32 cache rows pos0 + t, or with stage set to the
// staging rows kc, vc [T][kv_dim] of an F16 / Q8 cache
static void matmul_qkv(float *q, float *kc, float *vc, const krh_mat *wq, const krh_mat *wk, const krh_mat *wv,
                       const float *bq, const float *bk, const float *bv, const int8_t *xq, const float *xdT, int ldx,
                       int T, const float *rope_cos, const float *rope_sin, int head_dim, int pos0, bool stage) {
    if (wq->cols != wk->cols || wq->cols != wv->cols || wk->rows != wv->rows || head_dim % 2 || wq->type != wk->type ||
        wq->d16 != wk->d16 || wv->d16 != wq->d16) {
        kr_fail(ML_E_SHAPE, "matmul qkv shapes", hipSuccess);
        return;
    }
    MmArgs a = {};
    a.w[0] = to_mmat(wq);
    a.w[1] = to_mmat(wk);
    a.w[2] = to_mmat(wv);
    a.xq = xq;
    a.xdT = xdT;
    a.ldx = ldx;
    a.xsb = ldx;
    a.xst = 1;
    a.T = T;
    a.K = wq->cols;
    // q rows [t][q_dim]; k and v straight into the cache rows pos0 + t
    a.y[0] = q;
    a.ldy[0] = wq->rows;
    a.y[1] = kc + (stage ? 0 : (size_t)pos0 * wk->rows);
    a.ldy[1] = wk->rows;
    a.y[2] = vc + (stage ? 0 : (size_t)pos0 * wv->rows);
    a.ldy[2] = wv->rows;
    a.bias[0] = bq;
    a.bias[1] = bk;
    a.bias[2] = bv;
    a.rope_cos = rope_cos;
    a.rope_sin = rope_sin;
    a.head_dim = head_dim;
    a.pos0 = pos0;
    const int rows[3] = { wq->rows, wk->rows, wv->rows };
    mm_plan(a, 3, rows);
    if (wv->type == wq->type) {
        a.nmat = 3;
        launch_mm<MM_QKV>(a, a.w[0]);
        return;
    }
    MmArgs b = a;   // q and k
    b.nmat = 2;
    launch_mm<MM_QKV>(b, b.w[0]);
    MmArgs c = a;   // v alone, as matrix 2 of the same epilogue
    c.tile0[0] = c.tile0[1] = c.tile0[2] = 0;
    c.tile0[3] = a.tile0[3] - a.tile0[2];
    c.w[0] = c.w[1] = c.w[2];
    c.nmat = 3;
    launch_mm<MM_QKV>(c, c.w[2]);
}

extern "C" void krh_matmul_qkv(float *q, float *kc, float *vc, const krh_mat *wq, const krh_mat *wk,
                               const krh_mat *wv, const float *bq, const float *bk, const float *bv, const int8_t *xq,
                               const float *xdT, int ldx, int T, const float *rope_cos, const float *rope_sin,
                               int head_dim, int pos0) {
    matmul_qkv(q, kc, vc, wq, wk, wv, bq, bk, bv, xq, xdT, ldx, T, rope_cos, rope_sin, head_dim, pos0, false);
}

extern "C" void krh_matmul_qkv_stage(float *q, float *k, float *v, const krh_mat *wq, const krh_mat *wk,
                                     const krh_mat *wv, const float *bq, const float *bk, const float *bv,
                                     const int8_t *xq, const float *xdT, int ldx, int T, const float *rope_cos,
                                     const float *rope_sin, int head_dim, int pos0) {
    matmul_qkv(q, k, v, wq, wk, wv, bq, bk, bv, xq, xdT, ldx, T, rope_cos, rope_sin, head_dim, pos0, true);
}

extern "C" void krh_silu_quant(int8_t *q, float *dT, int ldd, const float *g, const float *u, int n, int ntok) {
    if (n % KR_QK || ntok <= 0) { kr_fail(ML_E_SHAPE, "silu_quant shape", hipSuccess); return; }
    hipLaunchKernelGGL(k_silu_quant, dim3((n + 1023) / 1024, ntok), dim3(256), 0, kr_stream(), q, dT, ldd, g, u, n);
    kr_check_launch("silu_quant");
}

extern "C" void krh_embed_batch(float *x, const krh_mat *emb, const int *tok, int ntok, float embed_scale) {
    hipLaunchKernelGGL(k_embed_batch, dim3((emb->cols + 255) / 256, ntok), dim3(256), 0, kr_stream(), x, to_mmat(emb),
                       tok, embed_scale);
    kr_check_launch("embed_batch");
}
