// attn.hip -- causal multi-head attention on the bf16 matrix cores, in fp32 (gfx950).
//
// Forward (train.c:339-370 attention_forward; gpu_kernels.cu:403-432 attn_fwd):
// per (batch, head) and query i, p_ij = softmax_j<=i(scale * q_i . k_j) and
// att_i = sum_j p_ij v_j, with the probabilities optionally stored for the
// backward ([B*H][T][T], zero above the diagonal as gpu_kernels.cu:279 does).
//
// Every product is fp32 by fp32: an operand element is the sum of three bf16
// (each the rounding of what the ones before it leave, 24 bits and their signs
// together, over fp32's whole range), and of the nine products the six that
// reach 2^-24 of the result are summed in fp32 accumulators, smallest first.
// The f32 MFMA does the same work at 1/16 of the bf16 rate, so six bf16
// products take 3/8 of its time; what is left is mostly the splitting (5.5
// VALU operations per element) and the softmax. An infinity or NaN has no such
// split and gives NaN: rows whose results are not finite are computed again
// from the operands with fp32 fma, one lane per row.
//
// Measured, f32 matrix cores -> these kernels: 4 x 16 heads of 64 over 1024
// tokens: forward with probabilities 155 -> 103 us, one pass 87 -> 63, backward
// 239 -> 197 (dS no longer stored); 1 x 16 x 64 over 1500 one pass 112 -> 62,
// 2 x 6 x 128 over 500 forward and backward 305 -> 203, 1 x 16 x 32 over 256
// one pass 13.3 -> 11.9. The matrix cores are busy 40% of that: a SIMD's two waves
// overlap their matrix and VALU phases only in part. Tried on the way: the four
// waves of one group alone, two workgroups per CU (84 us instead of 62 for the
// 1500 tokens); the next block's scores between the softmax's operations in one
// wave (spills at 64-wide heads); wave priorities (no change).
//
// One launch, no score matrix in HBM: a workgroup owns 128 queries of one head,
// as two groups of four waves (32 queries per wave) that each stream every other
// 32-key block of K and V through LDS, split as they are stored, and add what
// they have at the end. A causal grid is as long as its heaviest workgroup's
// chain of key blocks, so both waves of a SIMD work on that one chain, heaviest
// workgroups first. Each wave keeps its queries' Q in
// registers and computes the transposed score block S^T = K_blk . Q^T with
// v_mfma_f32_32x32x16_bf16, so a lane holds 16 scores of ONE query (its column)
// and a row reduction is 16 lane-local values plus one exchange with lane^32.
// O^T = V^T . P^T takes P^T as the register layout S^T left behind (B operand:
// the MFMA's k is permuted to the order in which a lane holds its keys, and V^T
// is stored in LDS in that order).
#include "internal.h"

#include <math.h>

namespace pcl {

typedef float v4f __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef float v2f __attribute__((ext_vector_type(2)));
typedef __bf16 v2bf __attribute__((ext_vector_type(2)));
typedef unsigned v2u __attribute__((ext_vector_type(2)));
typedef unsigned v4u __attribute__((ext_vector_type(4)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));

constexpr int AT_QB = 128;  // queries per workgroup (4 waves x 32)
constexpr int AT_G = 2;     // groups of waves, each taking every AT_G-th block
constexpr int AT_KB = 32;   // keys per block

// Two floats as three words of two bf16, h + m + l = (x, y).
__device__ __forceinline__ void at_split2(float x, float y, unsigned (&p)[3]) {
#pragma unroll
    for (int q = 0; q < 3; q++) {
        p[q] = __builtin_bit_cast(unsigned, __builtin_convertvector(v2f{x, y}, v2bf));
        if (q < 2) x -= __uint_as_float(p[q] << 16), y -= __uint_as_float(p[q] & 0xffff0000u);
    }
}
// Eight floats as three bf16 vectors.
__device__ __forceinline__ void at_split(const float (&a)[8], v4u (&p)[3]) {
#pragma unroll
    for (int e = 0; e < 4; e++) {
        unsigned w[3];
        at_split2(a[2 * e], a[2 * e + 1], w);
#pragma unroll
        for (int q = 0; q < 3; q++) p[q][e] = w[q];
    }
}

// The six products of two split operands, smallest first.
__device__ __forceinline__ v16f at_mfma(const v4u (&a)[3], const v4u (&b)[3], v16f c) {
    constexpr int I[6] = {2, 0, 1, 1, 0, 0}, J[6] = {0, 2, 1, 0, 1, 0};
#pragma unroll
    for (int x = 0; x < 6; x++)
        c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8bf, a[I[x]]), __builtin_bit_cast(v8bf, b[J[x]]),
                                                    c, 0, 0, 0);
    return c;
}
// The end of a chain of matrix instructions: 16 wait states before c is read
// (11 are needed). The compiler counts them itself, but here has once placed
// them behind the first reads, where two copies of a chain met at a branch.
__device__ __forceinline__ void at_settle(v16f (&c)[1]) { asm volatile("s_nop 15" : "+v"(c[0])); }
__device__ __forceinline__ void at_settle(v16f (&c)[2]) { asm volatile("s_nop 15" : "+v"(c[0]), "+v"(c[1])); }
__device__ __forceinline__ void at_settle(v16f (&c)[4]) {
    asm volatile("s_nop 15" : "+v"(c[0]), "+v"(c[1]), "+v"(c[2]), "+v"(c[3]));
}

// key offset (within the block) of accumulator element v for lane half lg
__device__ __forceinline__ constexpr int at_key(int v, int lg) { return (v >> 2) * 8 + lg * 4 + (v & 3); }

// A 32-row block of an operand in LDS, three planes of bf16. Row form (the
// score products' A operand, k along the head): rows of DH + 8, so that the 16
// rows that 16 lanes read as 16-byte pieces start in 16 different 16-byte bank
// groups. Column form (the accumulations' A operand, k along the rows): DH rows
// of 32 + 8, row d's elements in the order in which a lane half takes its
// keys (key 16u + 8h + 4lg + e at 16u + 8lg + 4h + e), the same bank groups.
template <int DH>
struct AtTile {
    static constexpr int RS = DH + 8, CS = AT_KB + 8;
    static constexpr int ROW = AT_KB * RS, COL = DH * CS;  // one plane
    static constexpr int BUFS = DH > 64 ? 1 : 2;           // blocks in LDS per group
    // waves per SIMD: one workgroup per CU, two with 32-wide heads (128 registers)
    static constexpr int WAVES = DH > 32 ? 2 : 4;
};

// A 32 x DH block of rows [r0, r0 + 32) of a (rows x ld) operand as this
// thread's (of NT) pieces: 8 consecutive elements of a row, or 4 x 4 elements.
// Rows >= T read row T-1 again: their scores are masked and their weights zero
// (ZERO: they are read as zeros).
template <int DH, int NT>
struct AtRows {
    static constexpr int N = (4 * DH + NT - 1) / NT;
    __device__ __forceinline__ static void load(v4f (&r)[2 * N], const float *X, long ld, long row0, int r0, int T,
                                                int t) {
#pragma unroll
        for (int u = 0; u < N; u++) {
            const int i = u * NT + t, rr = i / (DH / 8) % AT_KB, c = i % (DH / 8) * 8;
            const v4f *s = reinterpret_cast<const v4f *>(X + (row0 + min(r0 + rr, T - 1)) * ld + c);
            r[2 * u] = s[0], r[2 * u + 1] = s[1];
        }
    }
    __device__ __forceinline__ static void store(__bf16 *lds, const v4f (&r)[2 * N], int t) {
#pragma unroll
        for (int u = 0; u < N; u++) {
            const int i = u * NT + t, rr = i / (DH / 8), c = i % (DH / 8) * 8;
            if (4 * DH % NT != 0 && i >= 4 * DH) break;
            float a[8];
#pragma unroll
            for (int e = 0; e < 8; e++) a[e] = r[2 * u + e / 4][e % 4];
            v4u p[3];
            at_split(a, p);
#pragma unroll
            for (int q = 0; q < 3; q++)
                *reinterpret_cast<v4u *>(lds + q * AtTile<DH>::ROW + rr * AtTile<DH>::RS + c) = p[q];
        }
    }
};
template <int DH, int NT>
struct AtCols {
    static constexpr int N = (2 * DH + NT - 1) / NT;
    template <bool ZERO = false>
    __device__ __forceinline__ static void load(v4f (&r)[4 * N], const float *X, long ld, long row0, int r0, int T,
                                                int t) {
#pragma unroll
        for (int u = 0; u < N; u++) {
            const int i = u * NT + t, kg = i % (AT_KB / 4), c = i / (AT_KB / 4) % (DH / 4) * 4;
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const int rr = r0 + 4 * kg + k;
                r[4 * u + k] = *reinterpret_cast<const v4f *>(X + (row0 + min(rr, T - 1)) * ld + c);
            }
        }
        if (ZERO && r0 + AT_KB > T) {
#pragma unroll
            for (int u = 0; u < 4 * N; u++)
                if (r0 + (u / 4 * NT + t) % (AT_KB / 4) * 4 + u % 4 >= T) r[u] = v4f{0.f, 0.f, 0.f, 0.f};
        }
    }
    // column form, and with BOTH the row form at `rows` too
    template <bool BOTH = false>
    __device__ __forceinline__ static void store(__bf16 *cols, const v4f (&r)[4 * N], int t, __bf16 *rows = nullptr) {
#pragma unroll
        for (int u = 0; u < N; u++) {
            const int i = u * NT + t, kg = i % (AT_KB / 4), c = i / (AT_KB / 4) * 4;
            if (2 * DH % NT != 0 && i >= 2 * DH) break;
            unsigned w[4][2][3];  // [row][pair][plane]
#pragma unroll
            for (int k = 0; k < 4; k++) {
#pragma unroll
                for (int e = 0; e < 2; e++) at_split2(r[4 * u + k][2 * e], r[4 * u + k][2 * e + 1], w[k][e]);
                if constexpr (BOTH)
#pragma unroll
                    for (int q = 0; q < 3; q++)
                        *reinterpret_cast<v2u *>(rows + q * AtTile<DH>::ROW + (4 * kg + k) * AtTile<DH>::RS + c) =
                            v2u{w[k][0][q], w[k][1][q]};
            }
            const int at = (kg >> 2) * 16 + (kg & 1) * 8 + (kg >> 1 & 1) * 4;
#pragma unroll
            for (int d = 0; d < 4; d++)
#pragma unroll
                for (int q = 0; q < 3; q++) {
                    const int sel = d % 2 ? 0x07060302 : 0x05040100;  // high or low halves
                    *reinterpret_cast<v2u *>(cols + q * AtTile<DH>::COL + (c + d) * AtTile<DH>::CS + at) =
                        v2u{__builtin_amdgcn_perm(w[1][d / 2][q], w[0][d / 2][q], sel),
                            __builtin_amdgcn_perm(w[3][d / 2][q], w[2][d / 2][q], sel)};
                }
        }
    }
};

// This lane's row of an operand in registers (B operand of the score
// products): elements 16u + 8lg .. + 7, times mul.
template <int DH>
__device__ __forceinline__ void at_own_row(v4u (&f)[DH / 16][3], const float *row, int lg, float mul) {
#pragma unroll
    for (int u = 0; u < DH / 16; u++) {
        const v4f *s = reinterpret_cast<const v4f *>(row + 16 * u + 8 * lg);
        const v4f x = s[0] * mul, y = s[1] * mul;
        const float a[8] = {x[0], x[1], x[2], x[3], y[0], y[1], y[2], y[3]};
        at_split(a, f[u]);
    }
}

// S^T block (rows of the tile x own rows) of this wave.
template <int DH>
__device__ __forceinline__ v16f at_scores(const __bf16 *rows, const v4u (&own)[DH / 16][3], int r32, int lg) {
    v16f s[1];
#pragma unroll
    for (int v = 0; v < 16; v++) s[0][v] = 0.f;
    const __bf16 *x = rows + r32 * AtTile<DH>::RS + 8 * lg;
#pragma unroll
    for (int u = 0; u < DH / 16; u++) {
        v4u a[3];
#pragma unroll
        for (int q = 0; q < 3; q++) a[q] = *reinterpret_cast<const v4u *>(x + q * AtTile<DH>::ROW + 16 * u);
        s[0] = at_mfma(a, own[u], s[0]);
    }
    at_settle(s);
    return s[0];
}

// acc[nb] += X^T . W^T over one 32-row block: A = the block's column form, B =
// w (this lane's 16 weights, in the score layout's order).
template <int DH>
__device__ __forceinline__ void at_accum(v16f (&acc)[DH / 32], const __bf16 *cols, const float (&w)[16], int r32,
                                         int lg) {
    const __bf16 *x = cols + r32 * AtTile<DH>::CS + 8 * lg;
#pragma unroll
    for (int u = 0; u < 2; u++) {
        float h[8];
#pragma unroll
        for (int e = 0; e < 8; e++) h[e] = w[8 * u + e];
        v4u b[3];
        at_split(h, b);
#pragma unroll
        for (int nb = 0; nb < DH / 32; nb++) {
            v4u a[3];
#pragma unroll
            for (int q = 0; q < 3; q++)
                a[q] = *reinterpret_cast<const v4u *>(x + q * AtTile<DH>::COL + nb * 32 * AtTile<DH>::CS + 16 * u);
            acc[nb] = at_mfma(a, b, acc[nb]);
        }
    }
    at_settle(acc);
}

// max(v, the value of lane ^ 32) through v_permlane32_swap (a VALU exchange
// of the wave's halves, no LDS crossbar round trip)
__device__ __forceinline__ float at_max_halves(float v) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ bool at_finite(float x) { return fabsf(x) < INFINITY; }

// The online-softmax step of one key block in the log2 domain: the wave's Q
// fragments carry scale * log2(e), so s is already the exponent base 2 and
// p = 2^(s - m). Only a block holding keys past a query of the wave or past T
// (the diagonal block, the tail) is masked. The running maximum m moves only
// when a row's block maximum exceeds it by more than AT_LAZY (then the row's
// O^T and l are rescaled by 2^(m_old - m_new)); otherwise p = 2^(s - m) stays
// below 2^AT_LAZY. O / l and m + log2(l) do not depend on which m was used.
// The caller guarantees a visible key in every block it passes (so m is
// finite after the first).
constexpr float AT_LAZY = 8.f;
constexpr float AT_LOG2E = 1.44269504088896341f, AT_LN2 = 0.693147180559945309f;

// x = the block's scores with keys j > qi or j >= T set to -inf (MASK; keys k0 +
// at_key(v, lg)); returns max x.
template <bool MASK>
__device__ __forceinline__ float at_mask(const v16f &s, int k0, int qi, int T, int lg, float (&x)[16]) {
    const int lim = min(qi, T - 1) - k0;
#pragma unroll
    for (int v = 0; v < 16; v++) x[v] = !MASK || at_key(v, lg) <= lim ? s[v] : -INFINITY;
    float bm = x[0];
#pragma unroll
    for (int v = 1; v < 16; v++) bm = fmaxf(bm, x[v]);
    return bm;
}

// x = the block's masked scores; m moved, l and oacc rescaled where it moves.
template <int DH, bool MASK>
__device__ __forceinline__ void at_online(const v16f &s, int k0, int qi, int T, int lg, float &m, float &l,
                                          v16f (&oacc)[DH / 32], float (&x)[16]) {
    const float bm = at_mask<MASK>(s, k0, qi, T, lg, x);
    const float mn = fmaxf(m, at_max_halves(bm));  // lanes i and i ^ 32 agree
    const bool grow = mn > m + AT_LAZY;
    if (__any(grow)) {
        const float mu = grow ? mn : m;
        const float alpha = __builtin_amdgcn_exp2f(m - mu);  // 1 where m stays, 0 on the first block
        l *= alpha;
#pragma unroll
        for (int nb = 0; nb < DH / 32; nb++)
#pragma unroll
            for (int v = 0; v < 16; v++) oacc[nb][v] *= alpha;
        m = mu;
    }
}

// The two operands a group streams, one by each half of it: waves 0-1 the
// row-form one (scores), waves 2-3 the column-form one (accumulation). lds: the
// group's ELEMS; tid: within the group.
template <int DH>
struct AtPair {
    static constexpr int NR = 2 * AtRows<DH, 128>::N, NC = 4 * AtCols<DH, 128>::N;
    static constexpr int ROWS = 3 * AtTile<DH>::ROW, COLS = 3 * AtTile<DH>::COL;
    static constexpr int BUFS = AtTile<DH>::BUFS, ELEMS = BUFS * (ROWS + COLS);
    v4f r[NR > NC ? NR : NC];
    const float *X;
    __bf16 *lds;
    long ld, row0;
    int T, t;
    bool first;
    __device__ __forceinline__ AtPair(const float *rows, const float *cols, long ld_, long row0_, int T_, int tid,
                                      __bf16 *lds_)
        : X(tid < 128 ? rows : cols), lds(lds_), ld(ld_), row0(row0_), T(T_), t(tid & 127),
          first(__builtin_amdgcn_readfirstlane(tid) < 128) {}
    __device__ __forceinline__ __bf16 *rows(int block) const { return lds + block / AT_G % BUFS * ROWS; }
    __device__ __forceinline__ __bf16 *cols(int block) const { return lds + BUFS * ROWS + block / AT_G % BUFS * COLS; }
    __device__ __forceinline__ void load(int block) {
        if (first) AtRows<DH, 128>::load(*reinterpret_cast<v4f(*)[NR]>(&r), X, ld, row0, block * AT_KB, T, t);
        else AtCols<DH, 128>::load(*reinterpret_cast<v4f(*)[NC]>(&r), X, ld, row0, block * AT_KB, T, t);
    }
    __device__ __forceinline__ void store(int block) {
        if (first) AtRows<DH, 128>::store(rows(block), *reinterpret_cast<v4f(*)[NR]>(&r), t);
        else AtCols<DH, 128>::store(cols(block), *reinterpret_cast<v4f(*)[NC]>(&r), t);
    }
};

// Blocks g, g + AT_G, .. <= last through LDS: body(block) between barriers, which
// both groups cross as often; load(block) to registers, store(block) from there
// to LDS. With two blocks in LDS group 0 stores the next block after the body and
// group 1 before it: the groups share the barriers, so without that they would be
// in the same phase, both on the matrix cores or both splitting and storing.
// With one block both store it between two barriers, and EARLY load it before
// the body (else, without registers for that, there too).
template <int BUFS, bool EARLY, typename L, typename S, typename F>
__device__ __forceinline__ void at_stream(int g, int last, L &&load, S &&store, F &&body) {
    if (g <= last) {
        load(g);
        store(g);
    }
    if (BUFS > 1 && g == 1 && g + AT_G <= last) load(g + AT_G);
    __syncthreads();
    for (int kb = g; kb - g <= last; kb += AT_G) {
        const bool more = kb + AT_G <= last;
        if (BUFS > 1 && more) {
            if (g == 0) {
                load(kb + AT_G);
            } else {
                store(kb + AT_G);
                if (kb + 2 * AT_G <= last) load(kb + 2 * AT_G);
            }
        }
        if (BUFS == 1 && EARLY && more) load(kb + AT_G);
        if (kb <= last) body(kb);
        if (BUFS == 1) {
            __syncthreads();
            if (!EARLY && more) load(kb + AT_G);
        }
        if (more && (BUFS == 1 || g == 0)) store(kb + AT_G);
        __syncthreads();
    }
}
template <int DH, typename F>
__device__ __forceinline__ void at_stream(AtPair<DH> &x, int g, int last, F &&body) {
    at_stream<AtPair<DH>::BUFS, false>(
        g, last, [&](int kb) { x.load(kb); }, [&](int kb) { x.store(kb); },
        [&](int kb) { body(kb, x.rows(kb), x.cols(kb)); });
}

// Group 1's accumulators through LDS, to be added to group 0's (same slot).
template <int N>
__device__ __forceinline__ float *at_slot(float *x, int slot, int lane) {
    return x + slot * (N * 16 * 64) + lane;
}
template <int N>
__device__ __forceinline__ void at_give(float *x, const v16f (&acc)[N]) {
#pragma unroll
    for (int nb = 0; nb < N; nb++)
#pragma unroll
        for (int v = 0; v < 16; v++) x[(nb * 16 + v) * 64] = acc[nb][v];
}
template <int N>
__device__ __forceinline__ void at_take(const float *x, v16f (&acc)[N], float mine, float theirs) {
#pragma unroll
    for (int nb = 0; nb < N; nb++)
#pragma unroll
        for (int v = 0; v < 16; v++) acc[nb][v] = acc[nb][v] * mine + x[(nb * 16 + v) * 64] * theirs;
}

// One row with fp32 fma (a row whose split product is not finite): att at the
// head's columns [d0, d0 + dn), lse, and the probabilities when prow is set.
template <int DH>
__device__ __noinline__ void at_row_f32(const float *q, const float *K, const float *V, long ld, int n, float qsc,
                                        int d0, int dn, float *o, float *lse, float *prow) {
    auto score = [&](int j) {
        float s = 0.f;
        for (int d = 0; d < DH; d++) s = fmaf(q[d] * qsc, K[j * ld + d], s);
        return s;
    };
    float m = -INFINITY, l = 0.f;
    for (int j = 0; j < n; j++) m = fmaxf(m, score(j));
    for (int j = 0; j < n; j++) l += __builtin_amdgcn_exp2f(score(j) - m);
    const float inv = 1.f / l;
    if (lse) *lse = (m + __log2f(l)) * AT_LN2;
    for (int d = 0; d < dn; d += 4) {
        v4f a = {0.f, 0.f, 0.f, 0.f};
        for (int j = 0; j < n; j++) {
            const float p = __builtin_amdgcn_exp2f(score(j) - m) * inv;
            if (prow && d == 0) prow[j] = p;
            for (int e = 0; e < 4; e++) a[e] = fmaf(p, V[j * ld + d0 + d + e], a[e]);
        }
        for (int e = 0; e < 4; e++) o[d0 + d + e] = a[e];
    }
}

// The query block of a workgroup, heaviest first (causal work grows with it),
// and this wave's slice of it: group 1 hands its slices out in reverse, so the
// two waves that share a SIMD sum to about the same work.
struct AtQuery {
    int g, slot, lane, r32, lg, gtid, bh, hc, q0w, qi, kb_last, kbw;
    long row0;
    __device__ __forceinline__ AtQuery(int T, int H, int BH, int DH) {
        const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
        g = wave >> 2, slot = g ? 7 - wave : wave;
        lane = tid & 63, r32 = lane & 31, lg = lane >> 5, gtid = tid & 255;
        const int nqb = (T + AT_QB - 1) / AT_QB;
        bh = (int)(blockIdx.x % BH);
        row0 = (long)(bh / H) * T;  // first token row of this sequence
        hc = bh % H * DH;           // first column of this head
        const int q0 = (nqb - 1 - (int)(blockIdx.x / BH)) * AT_QB;
        q0w = q0 + slot * 32;
        qi = q0w + r32;                                     // this lane's query
        kb_last = min(T - 1, q0 + AT_QB - 1) / AT_KB;       // last key block of the workgroup
        kbw = q0w < T ? min(T - 1, q0w + 31) / AT_KB : -1;  // and of this wave
    }
};

template <int DH>
__global__ __launch_bounds__(256 * AT_G, AtTile<DH>::WAVES) void attn_fwd_kernel(const float *__restrict__ Q, const float *__restrict__ K,
                                                          const float *__restrict__ V, long ld,
                                                          float *__restrict__ O, long ldo, float *__restrict__ P,
                                                          int T, int H, int BH, float scale) {
    using TL = AtTile<DH>;
    __shared__ __attribute__((aligned(16))) __bf16 shared[AT_G * AtPair<DH>::ELEMS];
    const AtQuery a(T, H, BH, DH);
    const int lane = a.lane, r32 = a.r32, lg = a.lg, tid = a.gtid;
    __bf16 *lds = shared + a.g * AtPair<DH>::ELEMS;
    float *slot = at_slot<DH / 32>(reinterpret_cast<float *>(shared), a.slot, lane);
    const int qi = a.qi, q0w = a.q0w, kb_last = a.kb_last, kbw = a.kbw;

    // Q carries scale * log2(e): scores come out in log2 units and
    // p = 2^(s - m) / l = 2^(s - (m + log2 l))
    v4u qf[DH / 16][3];
    const float *qrow = Q + (a.row0 + min(qi, T - 1)) * ld + a.hc;
    at_own_row<DH>(qf, qrow, lg, scale * AT_LOG2E);

    // ---- pass 1: row maximum and exp-sum over keys j <= i (this lane's half)
    float m = -INFINITY, l = 0.f;
    {
        auto Kb = [&](int kb) { return lds + kb / AT_G % 2 * 3 * TL::ROW; };
        v4f kr[2 * AtRows<DH, 256>::N];
        at_stream<2, false>(
            a.g, kb_last, [&](int kb) { AtRows<DH, 256>::load(kr, K + a.hc, ld, a.row0, kb * AT_KB, T, tid); },
            [&](int kb) { AtRows<DH, 256>::store(Kb(kb), kr, tid); },
            [&](int kb) {
                if (kb > kbw) return;
                const v16f s = at_scores<DH>(Kb(kb), qf, r32, lg);
                float x[16], mn;
                if (kb < kbw) mn = at_mask<false>(s, kb * AT_KB, qi, T, lg, x);
                else mn = at_mask<true>(s, kb * AT_KB, qi, T, lg, x);
                mn = fmaxf(m, mn);
                // this lane half may not have seen a key yet: everything is 2^-inf then
                const float mf = mn == -INFINITY ? 0.f : mn;
                float acc = 0.f;
#pragma unroll
                for (int v = 0; v < 16; v++) acc += __builtin_amdgcn_exp2f(x[v] - mf);
                l = l * __builtin_amdgcn_exp2f(m - mf) + acc;
                m = mn;
            });
    }
    // combine the two key halves of each query (lanes c and c + 32) and the two
    // groups
    {
        auto merge = [&](float mo, float lo) {
            const float mx = fmaxf(m, mo);
            l = (m == -INFINITY ? 0.f : l * __builtin_amdgcn_exp2f(m - mx)) +
                (mo == -INFINITY ? 0.f : lo * __builtin_amdgcn_exp2f(mo - mx));
            m = mx;
        };
        merge(__shfl_xor(m, 32), __shfl_xor(l, 32));
        float *x = reinterpret_cast<float *>(shared) + a.slot * 64 + lane;
        x[a.g * 512] = m, x[a.g * 512 + 256] = l;
        __syncthreads();
        const float mo = x[(1 - a.g) * 512], lo = x[(1 - a.g) * 512 + 256];
        __syncthreads();
        merge(mo, lo);
        m = m + __log2f(l);  // p = 2^(s - m) from here on
    }

    // ---- pass 2: normalised probabilities, stored if asked, and O^T += V^T P^T
    v16f oacc[DH / 32];
#pragma unroll
    for (int nb = 0; nb < DH / 32; nb++)
#pragma unroll
        for (int v = 0; v < 16; v++) oacc[nb][v] = 0.f;
    const bool store_p = P != nullptr && qi < T;
    float *prow = store_p ? P + ((long)a.bh * T + qi) * T : nullptr;
    const bool vec_p = (T & 3) == 0 && (reinterpret_cast<uintptr_t>(P) & 15) == 0;
    AtPair<DH> kv(K + a.hc, V + a.hc, ld, a.row0, T, tid, lds);
    at_stream<DH>(kv, a.g, kb_last, [&](int kb, const __bf16 *rows, const __bf16 *cols) {
        if (kb > kbw) return;
        const v16f s = at_scores<DH>(rows, qf, r32, lg);
        float p[16];
        if (kb < kbw) at_mask<false>(s, kb * AT_KB, qi, T, lg, p);
        else at_mask<true>(s, kb * AT_KB, qi, T, lg, p);
#pragma unroll
        for (int v = 0; v < 16; v++) p[v] = __builtin_amdgcn_exp2f(p[v] - m);  // 2^-inf = 0
        // elements 4g .. 4g+3 are keys 8g + 4lg + 0..3: one 16-byte store each
        if (store_p && vec_p && (kb + 1) * AT_KB <= T) {  // a whole block inside T
            float *pr = prow + kb * AT_KB + 4 * lg;
#pragma unroll
            for (int g4 = 0; g4 < 4; g4++)
                *reinterpret_cast<v4f *>(pr + 8 * g4) = v4f{p[4 * g4], p[4 * g4 + 1], p[4 * g4 + 2], p[4 * g4 + 3]};
        } else if (store_p) {
#pragma unroll
            for (int v = 0; v < 16; v++) {
                const int j = kb * AT_KB + at_key(v, lg);
                if (j < T) prow[j] = p[v];
            }
        }
        at_accum<DH>(oacc, cols, p, r32, lg);
    });

    if (a.g == 1) at_give(slot, oacc);
    __syncthreads();
    // att: O^T element v of block nb is (d = 32 nb + key-layout row v, query qi)
    bool bad = !at_finite(m);
    if (a.g == 0 && qi < T) {
        at_take(slot, oacc, 1.f, 1.f);
        float *orow = O + (a.row0 + qi) * ldo + a.hc;
#pragma unroll
        for (int nb = 0; nb < DH / 32; nb++)
#pragma unroll
            for (int v = 0; v < 16; v++) {
                orow[nb * 32 + at_key(v, lg)] = oacc[nb][v];
                bad |= !at_finite(oacc[nb][v]);
            }
        bad = bad | (__shfl_xor((int)bad, 32) != 0);  // both halves of the row
        if (bad)
            at_row_f32<DH>(qrow, K + a.row0 * ld + a.hc, V + a.row0 * ld + a.hc, ld, qi + 1, scale * AT_LOG2E,
                           lg * (DH / 2), DH / 2, orow, nullptr, lg == 0 ? prow : nullptr);
    }
    // probabilities right of this wave's last key block are zero (the future)
    if (P != nullptr && q0w < T) {
        const int c0 = (kbw + 1) * AT_KB;
        for (int rr = a.g; rr < 32 && q0w + rr < T; rr += AT_G) {
            float *zr = P + ((long)a.bh * T + q0w + rr) * T;
            for (int c = c0 + lane; c < T; c += 64) zr[c] = 0.f;
        }
    }
}

// One pass with a running maximum, for callers that need no probabilities:
// per key block the two lanes of a query agree on the block maximum (one
// exchange) and add 2^(s - m) . v (at_online: base 2, scale folded into Q,
// masking and rescaling only where a block needs them). Scores are computed
// once; att = O / l, and the row's natural log-sum-exp ln2 (m + log2 l) is
// stored when lse is given (p_ij = exp(scale q_i.k_j - lse_i)).
template <int DH>
__global__ __launch_bounds__(256 * AT_G, AtTile<DH>::WAVES) void attn_fwd_online_kernel(const float *__restrict__ Q,
                                                                 const float *__restrict__ K,
                                                                 const float *__restrict__ V, long ld,
                                                                 float *__restrict__ O, long ldo,
                                                                 float *__restrict__ lse, int T, int H,
                                                                 int BH, float scale) {
    __shared__ __attribute__((aligned(16))) __bf16 shared[AT_G * AtPair<DH>::ELEMS];
    const AtQuery a(T, H, BH, DH);
    const int lane = a.lane, r32 = a.r32, lg = a.lg, tid = a.gtid;
    __bf16 *lds = shared + a.g * AtPair<DH>::ELEMS;
    float *slot = at_slot<DH / 32>(reinterpret_cast<float *>(shared), a.slot, lane);
    const int qi = a.qi;
    v4u qf[DH / 16][3];
    const float *qrow = Q + (a.row0 + min(qi, T - 1)) * ld + a.hc;
    at_own_row<DH>(qf, qrow, lg, scale * AT_LOG2E);  // scores in log2 units

    v16f oacc[DH / 32];
#pragma unroll
    for (int nb = 0; nb < DH / 32; nb++)
#pragma unroll
        for (int v = 0; v < 16; v++) oacc[nb][v] = 0.f;
    float m = -INFINITY, l = 0.f;
    AtPair<DH> kv(K + a.hc, V + a.hc, ld, a.row0, T, tid, lds);
    at_stream<DH>(kv, a.g, a.kb_last, [&](int kb, const __bf16 *rows, const __bf16 *cols) {
        if (kb > a.kbw) return;
        const v16f s = at_scores<DH>(rows, qf, r32, lg);
        float p[16];
        if (kb < a.kbw) at_online<DH, false>(s, kb * AT_KB, qi, T, lg, m, l, oacc, p);
        else at_online<DH, true>(s, kb * AT_KB, qi, T, lg, m, l, oacc, p);
        float ps = 0.f;
#pragma unroll
        for (int v = 0; v < 16; v++) {
            p[v] = __builtin_amdgcn_exp2f(p[v] - m);
            ps += p[v];
        }
        l += ps;
        at_accum<DH>(oacc, cols, p, r32, lg);
    });
    l += __shfl_xor(l, 32);  // the two key halves share m
    float *ml = reinterpret_cast<float *>(shared) + 4 * (DH / 32) * 16 * 64 + a.slot * 64 + lane;
    if (a.g == 1) at_give(slot, oacc), ml[0] = m, ml[256] = l;
    __syncthreads();
    if (a.g == 0 && qi < T) {
        const float mo = ml[0], mx = fmaxf(m, mo);  // group 1 may have seen no key
        const float mine = __builtin_amdgcn_exp2f(m - mx), theirs = mo == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(mo - mx);
        l = l * mine + ml[256] * theirs;
        m = mx;
        at_take(slot, oacc, mine, theirs);
        const float inv = 1.f / l;
        float *orow = O + (a.row0 + qi) * ldo + a.hc;
        bool bad = !at_finite(m) || !at_finite(l);
#pragma unroll
        for (int nb = 0; nb < DH / 32; nb++)
#pragma unroll
            for (int v = 0; v < 16; v++) {
                const float o = oacc[nb][v] * inv;
                orow[nb * 32 + at_key(v, lg)] = o;
                bad |= !at_finite(o);
            }
        float *lp = lse && lg == 0 ? lse + (long)a.bh * T + qi : nullptr;
        if (lp) *lp = (m + __log2f(l)) * AT_LN2;
        bad = bad | (__shfl_xor((int)bad, 32) != 0);
        if (bad)
            at_row_f32<DH>(qrow, K + a.row0 * ld + a.hc, V + a.row0 * ld + a.hc, ld, qi + 1, scale * AT_LOG2E,
                           lg * (DH / 2), DH / 2, orow, lp, nullptr);
    }
}

// ---------------------------------------------------------------- backward
// train.c:374-407 attention_backward / gpu_kernels.cu:437-486 attn_bwd, from
// the forward's stored probabilities P:
//   dP_ij = dO_i . v_j,  D_i = sum_j P_ij dP_ij,  dS_ij = P_ij (dP_ij - D_i) scale
//   dQ_i = sum_j dS_ij k_j,  dK_j = sum_i dS_ij q_i,  dV_j = sum_i P_ij dO_i
// Kernel A (per 128 queries of one head, like the forward): dP^T = V_blk .
// dO^T in the score layout (lane = query, 16 keys), pass 1 sums D_i, pass 2
// forms dS and accumulates dQ^T = K^T dS^T with dS^T as the register B operand.
// Kernel B (per 128 keys): dV^T = dO^T P and dK^T = Q^T dS over the query
// blocks at or after the keys (causal), with dO and Q blocks in LDS (A
// operand) and P rows read straight from HBM as the B operand (32 consecutive
// keys per lane half: one 128-byte row piece).
// dS goes through HBM ([B*H][T][T]: kernel A stores it in 16-byte pieces) only
// where the caller keeps it or the heads are 128 wide, whose kernel B has no
// registers for more; otherwise kernel A leaves D, and kernel B forms dP = dO .
// V^T again: a third product on the matrix cores for a write and a read of T^2
// floats.

// Row i of kernel A with fp32 fma, as at_row_f32; D is given or, without the
// forward's output, summed here.
template <int DH>
__device__ __noinline__ void at_dq_row_f32(const float *dO, const float *K, const float *V, long ld, const float *P,
                                           int n, float scale, float D, bool sum_d, float *Dout, float *dS, int d0,
                                           float *dQ, int accumulate) {
    auto dp = [&](int j) {
        float s = 0.f;
        for (int d = 0; d < DH; d++) s = fmaf(dO[d], V[j * ld + d], s);
        return s;
    };
    if (sum_d) {
        D = 0.f;
        for (int j = 0; j < n; j++) D = fmaf(P[j], dp(j), D);
        if (Dout) *Dout = D;
    }
    for (int d = d0; d < d0 + DH / 2; d += 4) {
        v4f a = {0.f, 0.f, 0.f, 0.f};
        for (int j = 0; j < n; j++) {
            const float ds = P[j] * (dp(j) - D) * scale;
            if (dS && d == 0) dS[j] = ds;
            for (int e = 0; e < 4; e++) a[e] = fmaf(ds, K[j * ld + d + e], a[e]);
        }
        for (int e = 0; e < 4; e++) dQ[d + e] = accumulate ? dQ[d + e] + a[e] : a[e];
    }
}

template <int DH>
__global__ __launch_bounds__(256 * AT_G, 2) void attn_bwd_dq_kernel(
    const float *__restrict__ dO, long ldo, const float *__restrict__ K,
    const float *__restrict__ V, long ld, const float *__restrict__ P, float *__restrict__ dS,
    float *__restrict__ dQ, long ldg, int T, int H, int BH, float scale, int accumulate, int keep_ds,
    const float *__restrict__ Ofw, long ldfw) {
    using TL = AtTile<DH>;
    __shared__ __attribute__((aligned(16))) __bf16 shared[AT_G * AtPair<DH>::ELEMS];
    const AtQuery a(T, H, BH, DH);
    const int lane = a.lane, r32 = a.r32, lg = a.lg, tid = a.gtid;
    __bf16 *lds = shared + a.g * AtPair<DH>::ELEMS;
    float *slot = at_slot<DH / 32>(reinterpret_cast<float *>(shared), a.slot, lane);
    const int qi = a.qi, kb_last = a.kb_last, kbw = a.kbw;
    const bool vec_p = (T & 3) == 0 && (reinterpret_cast<uintptr_t>(P) & 15) == 0 &&
                       (reinterpret_cast<uintptr_t>(dS) & 15) == 0;

    v4u df[DH / 16][3];  // dO of this lane's query
    const float *drow = dO + (a.row0 + min(qi, T - 1)) * ldo + a.hc;
    at_own_row<DH>(df, drow, lg, 1.f);
    const long prow = ((long)a.bh * T + min(qi, T - 1)) * T;
    // P_ij for this lane's 16 keys of block kb (zero past T)
    auto load_p = [&](int kb, float (&x)[16]) {
        if (vec_p && (kb + 1) * AT_KB <= T) {  // a whole block inside T (wave-uniform)
            const float *xr = P + prow + kb * AT_KB + 4 * lg;
#pragma unroll
            for (int g4 = 0; g4 < 4; g4++) {
                const v4f t = *reinterpret_cast<const v4f *>(xr + 8 * g4);
#pragma unroll
                for (int e = 0; e < 4; e++) x[4 * g4 + e] = t[e];
            }
            return;
        }
#pragma unroll
        for (int v = 0; v < 16; v++) {
            const int j = kb * AT_KB + at_key(v, lg);
            x[v] = j < T ? P[prow + j] : 0.f;
        }
    };

    // ---- pass 1: D_i = sum_j P_ij dP_ij (this lane's half of the keys), or,
    // given the forward's output, D_i = dO_i . att_i (the same sum, since
    // att_i = sum_j P_ij v_j) from the lane's half of the row
    float Dsum = 0.f, pn[16];
    if (Ofw) {
        const float *orow = Ofw + (a.row0 + min(qi, T - 1)) * ldfw + a.hc + 8 * lg;
#pragma unroll
        for (int u = 0; u < DH / 16; u++)
#pragma unroll
            for (int h = 0; h < 8; h += 4) {
                const v4f o = *reinterpret_cast<const v4f *>(orow + 16 * u + h);
                const v4f g = *reinterpret_cast<const v4f *>(drow + 8 * lg + 16 * u + h);
#pragma unroll
                for (int e = 0; e < 4; e++) Dsum += g[e] * o[e];
            }
    } else {
        // P rows are fetched one key block ahead of their use
        auto Vb = [&](int kb) { return lds + kb / AT_G % 2 * 3 * TL::ROW; };
        v4f vr[2 * AtRows<DH, 256>::N];
        if (a.g <= kbw) load_p(a.g, pn);
        at_stream<2, false>(
            a.g, kb_last, [&](int kb) { AtRows<DH, 256>::load(vr, V + a.hc, ld, a.row0, kb * AT_KB, T, tid); },
            [&](int kb) { AtRows<DH, 256>::store(Vb(kb), vr, tid); },
            [&](int kb) {
                if (kb > kbw) return;
                float pv[16];
#pragma unroll
                for (int v = 0; v < 16; v++) pv[v] = pn[v];
                if (kb + AT_G <= kbw) load_p(kb + AT_G, pn);
                const v16f dp = at_scores<DH>(Vb(kb), df, r32, lg);
                const int lim = min(qi, T - 1) - kb * AT_KB;  // P is zero above the diagonal, dP may be anything
#pragma unroll
                for (int v = 0; v < 16; v++) Dsum += at_key(v, lg) <= lim ? pv[v] * dp[v] : 0.f;
            });
        float *x = reinterpret_cast<float *>(shared) + a.slot * 64 + lane;  // the other group's keys
        x[a.g * 256] = Dsum;
        __syncthreads();
        Dsum = a.g ? x[0] + Dsum : Dsum + x[256];
        __syncthreads();
    }
    Dsum += __shfl_xor(Dsum, 32);

    // ---- pass 2: dS (stored if kept) and dQ^T += K^T dS^T
    v16f qacc[DH / 32];
#pragma unroll
    for (int nb = 0; nb < DH / 32; nb++)
#pragma unroll
        for (int v = 0; v < 16; v++) qacc[nb][v] = 0.f;
    const bool live = qi < T;
    if (a.g <= kbw) load_p(a.g, pn);
    AtPair<DH> vk(V + a.hc, K + a.hc, ld, a.row0, T, tid, lds);
    at_stream<DH>(vk, a.g, kb_last, [&](int kb, const __bf16 *rows, const __bf16 *cols) {
        if (kb > kbw) return;
        float pv[16], ds[16];
#pragma unroll
        for (int v = 0; v < 16; v++) pv[v] = pn[v];
        if (kb + AT_G <= kbw) load_p(kb + AT_G, pn);
        const v16f dp = at_scores<DH>(rows, df, r32, lg);
#pragma unroll
        for (int v = 0; v < 16; v++) ds[v] = pv[v] * (dp[v] - Dsum) * scale;
        if (kb == kbw) {  // the diagonal block (wave-uniform)
            const int lim = min(qi, T - 1) - kb * AT_KB;
#pragma unroll
            for (int v = 0; v < 16; v++) ds[v] = at_key(v, lg) <= lim ? ds[v] : 0.f;
        }
        if (keep_ds && live && vec_p && (kb + 1) * AT_KB <= T) {
            float *sr = dS + prow + kb * AT_KB + 4 * lg;
#pragma unroll
            for (int g4 = 0; g4 < 4; g4++)
                *reinterpret_cast<v4f *>(sr + 8 * g4) = v4f{ds[4 * g4], ds[4 * g4 + 1], ds[4 * g4 + 2], ds[4 * g4 + 3]};
        } else if (keep_ds && live) {
#pragma unroll
            for (int v = 0; v < 16; v++) {
                const int j = kb * AT_KB + at_key(v, lg);
                if (j < T) dS[prow + j] = ds[v];
            }
        }
        at_accum<DH>(qacc, cols, ds, r32, lg);
    });
    if (a.g == 1) at_give(slot, qacc);
    __syncthreads();
    if (a.g == 0 && live) {
        at_take(slot, qacc, 1.f, 1.f);
        float *grow = dQ + (a.row0 + qi) * ldg + a.hc;
        float *Dout = !keep_ds && lg == 0 ? dS + (long)a.bh * T + qi : nullptr;
        if (Dout) *Dout = Dsum;
        bool bad = !at_finite(Dsum);
#pragma unroll
        for (int nb = 0; nb < DH / 32; nb++)
#pragma unroll
            for (int v = 0; v < 16; v++) bad |= !at_finite(qacc[nb][v]);
        bad = bad | (__shfl_xor((int)bad, 32) != 0);
        if (bad) {
            at_dq_row_f32<DH>(drow, K + a.row0 * ld + a.hc, V + a.row0 * ld + a.hc, ld, P + prow, qi + 1, scale, Dsum,
                              Ofw == nullptr, Dout, keep_ds && lg == 0 ? dS + prow : nullptr, lg * (DH / 2), grow,
                              accumulate);
        } else {
#pragma unroll
            for (int nb = 0; nb < DH / 32; nb++)
#pragma unroll
                for (int v = 0; v < 16; v++) {
                    float *o = grow + nb * 32 + at_key(v, lg);
                    *o = accumulate ? *o + qacc[nb][v] : qacc[nb][v];
                }
        }
    }
}

// Key j of kernel B with fp32 fma; dS is the stored one or, without (DS NULL),
// formed from D.
template <int DH>
__device__ __noinline__ void at_dkv_row_f32(const float *dO, long ldo, const float *Q, const float *vrow, long ld,
                                            const float *P, const float *DS, const float *D, int j, int T,
                                            float scale, int d0, float *dK, float *dV, int accumulate) {
    for (int d = d0; d < d0 + DH / 2; d += 4) {
        v4f a = {0.f, 0.f, 0.f, 0.f}, b = a;
        for (int i = j; i < T; i++) {
            const float p = P[(long)i * T + j];
            float ds;
            if (DS) {
                ds = DS[(long)i * T + j];
            } else {
                float dp = 0.f;
                for (int e = 0; e < DH; e++) dp = fmaf(dO[i * ldo + e], vrow[e], dp);
                ds = p * (dp - D[i]) * scale;
            }
            for (int e = 0; e < 4; e++) {
                a[e] = fmaf(p, dO[i * ldo + d + e], a[e]);
                b[e] = fmaf(ds, Q[i * ld + d + e], b[e]);
            }
        }
        for (int e = 0; e < 4; e++) {
            dV[d + e] = accumulate ? dV[d + e] + a[e] : a[e];
            dK[d + e] = accumulate ? dK[d + e] + b[e] : b[e];
        }
    }
}

// DSMEM: dS comes from memory (written by kernel A), else D does and dP is
// formed here.
template <int DH, bool DSMEM>
__global__ __launch_bounds__(256 * AT_G, 2) void attn_bwd_dkv_kernel(
    const float *__restrict__ dO, long ldo, const float *__restrict__ Q, const float *__restrict__ V, long ld,
    const float *__restrict__ P, const float *__restrict__ dS, float *__restrict__ dK,
    float *__restrict__ dV, long ldg, int T, int H, int BH, float scale, int accumulate) {
    using TL = AtTile<DH>;
    constexpr int COLS = 3 * TL::COL, ROWS = DSMEM ? 0 : 3 * TL::ROW, STAGE = 2 * COLS + ROWS;
    constexpr int BUFS = AT_G * 2 * STAGE * 2 <= 128 * 1024 ? 2 : 1;
    constexpr int NC = 4 * AtCols<DH, 128>::N;
    __shared__ __attribute__((aligned(16))) __bf16 shared[AT_G * BUFS * STAGE];
    __shared__ __attribute__((aligned(16))) float Dl_all[AT_G][BUFS][AT_KB];
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), g = wave >> 2, slot = g ? 7 - wave : wave;
    const int tid = threadIdx.x & 255, lane = tid & 63, r32 = lane & 31, lg = lane >> 5;
    __bf16 *lds = shared + g * BUFS * STAGE;
    auto &Dl = Dl_all[g];
    // key block k needs the query blocks from k on: work falls with k
    const int bh = (int)(blockIdx.x % BH), kblk = (int)(blockIdx.x / BH);
    const long row0 = (long)(bh / H) * T;
    const int hc = bh % H * DH;
    const int k0 = kblk * AT_QB, k0w = k0 + slot * 32;
    const int kj = k0w + r32;  // this lane's key (its output column)
    const int qb_first = k0 / AT_KB, qb_last = (T - 1) / AT_KB;
    const int qbw = k0w / AT_KB;  // this wave's first query block
    const int kcol = min(kj, T - 1);
    const float *vrow = V + (row0 + kcol) * ld + hc;
    v4u vf[DSMEM ? 1 : DH / 16][3];
    if constexpr (!DSMEM) at_own_row<DH>(vf, vrow, lg, 1.f);

    v16f vacc[DH / 32], kacc[DH / 32];
#pragma unroll
    for (int nb = 0; nb < DH / 32; nb++)
#pragma unroll
        for (int v = 0; v < 16; v++) vacc[nb][v] = 0.f, kacc[nb][v] = 0.f;
    const float *Pbh = P + (long)bh * T * T, *Sbh = dS + (long)bh * T * T, *Dbh = dS + (long)bh * T;

    // P (and dS) of queries qb*32 + at_key(v, lg), key kj, fetched one query
    // block ahead of their use. Rows past T read row T-1 and keys past T key
    // T-1: finite values that meet zero dO / Q rows in LDS or land in output
    // columns that are not stored. A block inside T addresses its rows as a
    // uniform base plus the lane's 32-bit offset.
    float pn[16], sn[DSMEM ? 16 : 1];
    const unsigned lane_off = (unsigned)(4 * lg * T + kcol);
    auto load_ps = [&](int qb) {
        const bool whole = (qb + 1) * AT_KB <= T;
        const float *pr = Pbh + (long)qb * AT_KB * T, *sr = Sbh + (long)qb * AT_KB * T;
#pragma unroll
        for (int v = 0; v < 16; v++) {
            if (whole) {
                const long ro = (long)at_key(v, 0) * T;
                pn[v] = (pr + ro)[lane_off];
                if constexpr (DSMEM) sn[v] = (sr + ro)[lane_off];
            } else {
                const long o = (long)min(qb * AT_KB + at_key(v, lg), T - 1) * T + kcol;
                pn[v] = Pbh[o];
                if constexpr (DSMEM) sn[v] = Sbh[o];
            }
        }
    };
    // waves 0-1 stream dO (column form, and row form for dP), waves 2-3 Q
    v4f xr[NC];
    float dn = 0.f;
    const bool first = (wave & 3) < 2;
    auto load = [&](int qb) {
        AtCols<DH, 128>::template load<true>(xr, first ? dO + hc : Q + hc, first ? ldo : ld, row0, qb * AT_KB, T, tid & 127);
        if (!DSMEM && tid < AT_KB) dn = Dbh[min(qb * AT_KB + tid, T - 1)];
    };
    auto store = [&](int buf) {
        __bf16 *st = lds + buf * STAGE;
        if (first && !DSMEM) AtCols<DH, 128>::template store<true>(st, xr, tid & 127, st + 2 * COLS);
        else AtCols<DH, 128>::store(first ? st : st + COLS, xr, tid & 127);
        if (!DSMEM && tid < AT_KB) Dl[buf][tid] = dn;
    };
    const int p0 = max(qbw, qb_first) + ((qbw ^ (qb_first + g)) & 1);  // this wave's first block that is its group's
    if (k0w < T && p0 <= qb_last) load_ps(p0);
    at_stream<BUFS, DH <= 64>(
        g, qb_last - qb_first, [&](int i) { load(qb_first + i); }, [&](int i) { store(i / AT_G % BUFS); },
        [&](int i) {
            const int qb = qb_first + i, buf = i / AT_G % BUFS;
            if (k0w >= T || qb < qbw) return;
            const __bf16 *st = lds + buf * STAGE;
            float pv[16], sv[16];
#pragma unroll
            for (int v = 0; v < 16; v++) {
                pv[v] = pn[v];
                if constexpr (DSMEM) sv[v] = sn[v];
            }
            if (qb + AT_G <= qb_last) load_ps(qb + AT_G);
            if (qb == qbw) {  // the diagonal block: queries before the key take nothing
#pragma unroll
                for (int v = 0; v < 16; v++)
                    if (qb * AT_KB + at_key(v, lg) < kj) {
                        pv[v] = 0.f;
                        if constexpr (DSMEM) sv[v] = 0.f;
                    }
            }
            if constexpr (!DSMEM) {
                const v16f dp = at_scores<DH>(st + 2 * COLS, vf, r32, lg);
#pragma unroll
                for (int g = 0; g < 4; g++) {
                    const v4f D4 = *reinterpret_cast<const v4f *>(&Dl[buf][8 * g + 4 * lg]);
#pragma unroll
                    for (int e = 0; e < 4; e++) sv[4 * g + e] = pv[4 * g + e] * (dp[4 * g + e] - D4[e]) * scale;
                }
            }
            at_accum<DH>(vacc, st, pv, r32, lg);
            at_accum<DH>(kacc, st + COLS, sv, r32, lg);
        });
    float *x = at_slot<DH / 32>(reinterpret_cast<float *>(shared), slot, lane);
    if (g == 1) at_give(x, vacc);
    __syncthreads();
    if (g == 0) at_take(x, vacc, 1.f, 1.f);
    __syncthreads();
    if (g == 1) at_give(x, kacc);
    __syncthreads();
    if (g == 0) at_take(x, kacc, 1.f, 1.f);
    if (g == 0 && kj < T) {
        float *vout = dV + (row0 + kj) * ldg + hc, *kout = dK + (row0 + kj) * ldg + hc;
        bool bad = false;
#pragma unroll
        for (int nb = 0; nb < DH / 32; nb++)
#pragma unroll
            for (int v = 0; v < 16; v++) bad |= !at_finite(vacc[nb][v]) || !at_finite(kacc[nb][v]);
        bad = bad | (__shfl_xor((int)bad, 32) != 0);
        if (bad) {
            at_dkv_row_f32<DH>(dO + row0 * ldo + hc, ldo, Q + row0 * ld + hc, vrow, ld, Pbh, DSMEM ? Sbh : nullptr,
                               Dbh, kj, T, scale, lg * (DH / 2), kout, vout, accumulate);
        } else {
#pragma unroll
            for (int nb = 0; nb < DH / 32; nb++)
#pragma unroll
                for (int v = 0; v < 16; v++) {
                    const int d = nb * 32 + at_key(v, lg);
                    vout[d] = accumulate ? vout[d] + vacc[nb][v] : vacc[nb][v];
                    kout[d] = accumulate ? kout[d] + kacc[nb][v] : kacc[nb][v];
                }
        }
    }
}

hipError_t launch_attn_bwd(const float *dO, long ldo, const float *Q, const float *K,
                           const float *V, long ld, const float *P, float *dS, float *dQ,
                           float *dK, float *dV, long ldg, int B, int T, int H, int dh,
                           float scale, int flags, hipStream_t stream, const float *Ofw,
                           long ldfw) {
    const int BH = B * H, nb = (T + AT_QB - 1) / AT_QB;
    if (BH == 0 || T == 0) return hipSuccess;
    const dim3 grid((unsigned)((long)nb * BH)), block(256 * AT_G);
    const int accumulate = flags & ATTN_ACCUMULATE, keep = dh > 64 || (flags & ATTN_KEEP_DS);
#define PCL_ATTN_BWD(D)                                                                                      \
    hipLaunchKernelGGL(attn_bwd_dq_kernel<D>, grid, block, 0, stream, dO, ldo, K, V, ld, P, dS, dQ, ldg, T, H, \
                       BH, scale, accumulate, keep, Ofw, ldfw);                                              \
    if (keep)                                                                                                \
        hipLaunchKernelGGL((attn_bwd_dkv_kernel<D, true>), grid, block, 0, stream, dO, ldo, Q, V, ld, P, dS, \
                           dK, dV, ldg, T, H, BH, scale, accumulate);                                        \
    else if constexpr (D <= 64)                                                                              \
        hipLaunchKernelGGL((attn_bwd_dkv_kernel<D, false>), grid, block, 0, stream, dO, ldo, Q, V, ld, P, dS, \
                           dK, dV, ldg, T, H, BH, scale, accumulate)
    switch (dh) {
        case 32: PCL_ATTN_BWD(32); break;
        case 64: PCL_ATTN_BWD(64); break;
        case 128: PCL_ATTN_BWD(128); break;
        default: return hipErrorInvalidValue;
    }
#undef PCL_ATTN_BWD
    return hipGetLastError();
}

hipError_t launch_attn_fwd(const float *Q, const float *K, const float *V, long ld, float *O,
                           long ldo, float *P, int B, int T, int H, int dh, float scale,
                           hipStream_t stream, float *lse) {
    const int BH = B * H, nqb = (T + AT_QB - 1) / AT_QB;
    if (BH == 0 || T == 0) return hipSuccess;
    const dim3 grid((unsigned)((long)nqb * BH)), block(256 * AT_G);
    if (P == nullptr) {  // no probabilities: one pass
        switch (dh) {
            case 32:
                hipLaunchKernelGGL((attn_fwd_online_kernel<32>), grid, block, 0, stream, Q, K, V, ld, O, ldo, lse, T, H, BH, scale);
                break;
            case 64:
                hipLaunchKernelGGL((attn_fwd_online_kernel<64>), grid, block, 0, stream, Q, K, V, ld, O, ldo, lse, T, H, BH, scale);
                break;
            case 128:
                hipLaunchKernelGGL((attn_fwd_online_kernel<128>), grid, block, 0, stream, Q, K, V, ld, O, ldo, lse, T, H, BH, scale);
                break;
            default:
                return hipErrorInvalidValue;
        }
        return hipGetLastError();
    }
    if (lse) return hipErrorInvalidValue;
    switch (dh) {
        case 32:
            hipLaunchKernelGGL(attn_fwd_kernel<32>, grid, block, 0, stream, Q, K, V, ld, O, ldo, P, T, H, BH, scale);
            break;
        case 64:
            hipLaunchKernelGGL(attn_fwd_kernel<64>, grid, block, 0, stream, Q, K, V, ld, O, ldo, P, T, H, BH, scale);
            break;
        case 128:
            hipLaunchKernelGGL(attn_fwd_kernel<128>, grid, block, 0, stream, Q, K, V, ld, O, ldo, P, T, H, BH, scale);
            break;
        default:
            return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

}  // namespace pcl
