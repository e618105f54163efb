// sgemm_split.hip -- large FP32 GEMMs on the f16 matrix cores.
//
// The f32 MFMA runs at 1/16 of the f16 one, so above a size (chosen in pcl_sgemm)
// a product is taken as three f16 products that together keep the fp32
// operands' precision. Row m of op(A) is scaled by the power of two that puts
// its largest magnitude in [2^14, 2^15) and each element written as
//   a = hi + lo,  hi = f16(a), lo = f16(a - hi),
// likewise column n of op(B); then
//   C[m,n] = 2^(ea[m] + eb[n]) * sum_k (ah*bh + ah*bl + al*bh),
// every f16 product exact and all sums in fp32 accumulators.
//
// Error. The 11-bit hi and lo hold 22 bits and a sign, so hi + lo is within one
// fp32 ulp of a wherever |a| >= 2^-17 of its row's maximum, and within 2^-39 of
// that maximum below; al*bl, left out, is below 2^-22 |a b|. These are
// independent of k and average out along it, while the rounding of the
// accumulators grows with the number of additions: one MFMA adds 32 k here
// and 4 in the f32 form.
//
// Rows or columns that hold an infinity or a NaN have no such scale: their
// exponent carries SPLIT_NONFINITE, and the epilogue computes the outputs they
// touch from the original operands with fp32 fma, so the result is the IEEE
// one.
//
// Two kinds of kernel. The split pass reads each operand and writes it as K-
// contiguous units of 8 rows x 32 k (1 KB: 8 rows of 128 bytes, each four
// groups of 8 hi then 8 lo, 16-byte chunk c of row r at c ^ ((r >> 1) & 7)),
// the order in which the GEMM's LDS stages want them: any layout, stride or
// alignment of the operand ends here, and one GEMM DMA instruction reads 1 KB
// of consecutive memory. The GEMM kernel streams the units through an LDS ring.
#include "internal.h"
#include "sgemm_common.h"
#include "split_units.h"

namespace pcl {

// One operand to split: element (row, k) at X[row * ld + k] (kcontig) or X[k * ld + row].
struct SplitJob {
    const float *X;
    long ld;
    int rows, kcontig, vec;  // vec: 16-byte aligned rows
    int8_t *P;
    int *ex;
    unsigned *part;  // not kcontig: partial maxima, [ceil(K / SPLIT_KC)][rows]
    int blocks;      // of split_pass1_kernel
};

// Four floats of a run that ends at `n`, zeros past it.
__device__ __forceinline__ v4f split_load4(const float *x, int i, int n, bool vec) {
    if (vec && i + 4 <= n) return *reinterpret_cast<const v4f *>(x + i);
    v4f v;
#pragma unroll
    for (int e = 0; e < 4; e++) v[e] = i + e < n ? x[i + e] : 0.f;
    return v;
}

// Operand with consecutive k: NT threads per row, each G groups of 8 k in
// registers, so the operand is read once (rows of up to 8 NT G floats; MULTI:
// longer rows, read twice).
template <int NT, int G, bool MULTI>
__device__ __forceinline__ void split_rows(const SplitJob &j, int block, int K, unsigned (*wmax)[64]) {
    constexpr int RPB = NT < 256 ? 256 / NT : 1;
    const int t = threadIdx.x % NT, row = block * RPB + threadIdx.x / NT;
    const int nk = split_units(K), Kp = nk * SPLIT_BK;
    const bool in = row < j.rows;  // rows up to the last unit's are written as zeros
    const float *x = j.X + (long)(in ? row : 0) * j.ld;
    float a[G][8];
    auto load = [&](int k0) {
#pragma unroll
        for (int g = 0; g < G; g++)
#pragma unroll
            for (int h = 0; h < 8; h += 4) {
                const v4f v = split_load4(x, k0 + (g * NT + t) * 8 + h, in ? K : 0, j.vec);
#pragma unroll
                for (int e = 0; e < 4; e++) a[g][h + e] = v[e];
            }
    };
    unsigned mx = 0;
    const int steps = MULTI ? (K + NT * G * 8 - 1) / (NT * G * 8) : 1;
    for (int s = 0; s < steps; s++) {
        load(s * NT * G * 8);
#pragma unroll
        for (int g = 0; g < G; g++)
#pragma unroll
            for (int e = 0; e < 8; e++) mx = max(mx, split_mag(a[g][e]));
    }
    for (int o = 32; o > 0; o >>= 1) mx = max(mx, (unsigned)__shfl_xor((int)mx, o));
    if constexpr (NT > 64) {
        if ((threadIdx.x & 63) == 0) wmax[0][threadIdx.x >> 6] = mx;
        __syncthreads();
#pragma unroll
        for (int w = 0; w < NT / 64; w++) mx = max(mx, wmax[0][w]);
    }
    int shift;
    const bool finite = split_shift(mx, shift);
    if (t == 0 && in) j.ex[row] = finite ? -shift : SPLIT_NONFINITE;
    if (row >= (j.rows + 7) / 8 * 8) return;
    for (int s = 0; s < steps; s++) {
        if (MULTI) load(s * NT * G * 8);
#pragma unroll
        for (int g = 0; g < G; g++) {
            const int k = s * NT * G * 8 + (g * NT + t) * 8;
            if (k < Kp) split_store(j.P, nk, row, k, a[g], shift, finite);
        }
    }
}

// Operand with consecutive rows: largest |x| of 64 rows over SPLIT_KC k.
constexpr int SPLIT_KC = 128;
template <int THREADS>
__device__ __forceinline__ void split_colmax(const SplitJob &j, int block, int K, unsigned (*red)[64]) {
    const int nrb = (j.rows + 63) / 64;
    const int c = (threadIdx.x & 15) * 4, kr = threadIdx.x >> 4;
    const int r0 = block % nrb * 64, k0 = block / nrb * SPLIT_KC;
    unsigned mx[4] = {0, 0, 0, 0};
#pragma unroll
    for (int k = 0; k < SPLIT_KC; k += THREADS / 16) {
        const int kk = k0 + k + kr;
        const v4f v = split_load4(j.X + (long)min(kk, K - 1) * j.ld, r0 + c, kk < K ? j.rows : 0, j.vec);
#pragma unroll
        for (int e = 0; e < 4; e++) mx[e] = max(mx[e], split_mag(v[e]));
    }
#pragma unroll
    for (int e = 0; e < 4; e++) red[kr][c + e] = mx[e];
    __syncthreads();
    if (threadIdx.x < 64 && r0 + (int)threadIdx.x < j.rows) {
        unsigned m = 0;
#pragma unroll
        for (int r = 0; r < THREADS / 16; r++) m = max(m, red[r][threadIdx.x]);
        j.part[(long)(block / nrb) * j.rows + r0 + threadIdx.x] = m;
    }
}

// First pass over both operands: K-contiguous ones are split, the others' row
// maxima taken.
template <int NT, int G, bool MULTI>
__global__ __launch_bounds__(NT < 256 ? 256 : NT) void split_pass1_kernel(SplitJob a, SplitJob b, int K) {
    constexpr int THREADS = NT < 256 ? 256 : NT;
    __shared__ unsigned red[THREADS / 16][64];
    const bool second = (int)blockIdx.x >= a.blocks;
    const SplitJob &j = second ? b : a;
    const int block = second ? blockIdx.x - a.blocks : blockIdx.x;
    if (j.kcontig) split_rows<NT, G, MULTI>(j, block, K, red);
    else split_colmax<THREADS>(j, block, K, red);
}

// Second pass, operands with consecutive rows: 64 rows x 64 k per block through
// LDS, the rows' scales from the partial maxima. A quarter-wave's stores fill
// whole 128-byte unit rows.
__global__ __launch_bounds__(256) void split_pass2_kernel(SplitJob a, SplitJob b, int K, int blocks_a) {
    __shared__ float tile[64][66];  // [k][row]
    __shared__ unsigned red[4][64];
    __shared__ int sh[64];
    const bool second = (int)blockIdx.x >= blocks_a;
    const SplitJob &j = second ? b : a;
    const int block = second ? blockIdx.x - blocks_a : blockIdx.x;
    const int nrb = (j.rows + 63) / 64, nk = split_units(K), nparts = (K + SPLIT_KC - 1) / SPLIT_KC;
    const int tid = threadIdx.x, r0 = block % nrb * 64, k0 = block / nrb * 64;
    const int c = (tid & 15) * 4, kr = tid >> 4;
    v4f v[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int k = k0 + i * 16 + kr;
        v[i] = split_load4(j.X + (long)min(k, K - 1) * j.ld, r0 + c, k < K ? j.rows : 0, j.vec);
    }
    {
        const int r = min(r0 + (tid & 63), j.rows - 1);
        unsigned m = 0;
#pragma unroll 8
        for (int p = tid >> 6; p < nparts; p += 4) m = max(m, j.part[(long)p * j.rows + r]);
        red[tid >> 6][tid & 63] = m;
    }
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
        for (int e = 0; e < 4; e++) tile[i * 16 + kr][c + e] = v[i][e];
    __syncthreads();
    if (tid < 64) {
        int s;
        const bool finite = split_shift(max(max(red[0][tid], red[1][tid]), max(red[2][tid], red[3][tid])), s);
        sh[tid] = finite ? s : SPLIT_NONFINITE;
        if (k0 == 0 && r0 + tid < j.rows) j.ex[r0 + tid] = finite ? -s : SPLIT_NONFINITE;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 2; i++) {
        const int r = tid >> 2, k = i * 32 + (tid & 3) * 8;
        if (r0 + r >= (j.rows + 7) / 8 * 8 || k0 + k >= nk * SPLIT_BK) continue;
        float x[8];
#pragma unroll
        for (int e = 0; e < 8; e++) x[e] = tile[k + e][r];
        split_store(j.P, nk, r0 + r, k0 + k, x, sh[r], sh[r] != SPLIT_NONFINITE);
    }
}

// ---- the product of two split operands ----
struct SplitGemmArgs {
    const int8_t *Ap, *Bp;  // units of op(A)'s rows and op(B)'s columns
    const int *ea, *eb;
    const float *A, *B;  // the originals, for rows and columns that are not finite
    long sam, sak, sbn, sbk;
    const float *bias;
    float *C;
    long ldc;
    int M, N, K, accumulate, kchunk;  // kchunk: k per blockIdx.y, a multiple of SPLIT_BK
    const float *aux_in;
    float *aux_out;
    long ld_aux;
};

// BM x BN tile, WM x WN waves per K group, KG groups of waves that each take
// every KG-th unit of K (their sums added through LDS at the end). A wave's tile
// is TM x TN blocks of 16x16; its A fragments are taken in APH phases of TMP
// blocks, so 128-row wave tiles fit their registers.
template <int BM, int BN, int STAGES, int KG, int WM, int WN, int APH, int OCC, int EPI>
__global__ __launch_bounds__(64 * KG * WM * WN, OCC * KG * WM * WN / 4) void sgemm_split_kernel(SplitGemmArgs p) {
    constexpr int NW = KG * WM * WN, WTM = BM / WM, WTN = BN / WN, TM = WTM / 16, TN = WTN / 16, TMP = TM / APH;
    constexpr int SUB = (BM + BN) * 128, STAGE = KG * SUB, LOADS = STAGE / SPLIT_UNIT / NW;
    static_assert(LOADS * NW * SPLIT_UNIT == STAGE && (STAGES - 1) * LOADS <= 63, "DMA split and vmcnt range");
    static_assert(STAGES * STAGE <= 160 * 1024 / OCC, "OCC workgroups per CU");
    static_assert(TM % (APH * KG) == 0 && (APH == 1 || APH % 2 == 0) && KG <= SPLIT_KUNITS, "phases and groups");
    __shared__ __attribute__((aligned(1024))) int8_t lds[STAGES * STAGE];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int kg = wave / (WM * WN), wm = wave / WN % WM, wn = wave % WN, r16 = lane & 15, q = lane >> 4;
    const int M = p.M, N = p.N;
    const int nbm = (M + BM - 1) / BM, nbn = (N + BN - 1) / BN;
    int bm, bn;
    tile_coords(xcd_remap(blockIdx.x, nbm * nbn), nbm, nbn, 8, bm, bn);
    const int m0 = bm * BM, n0 = bn * BN;
    const int nkt = split_units(p.K);  // units along K
    const int kt0 = blockIdx.y * (p.kchunk / SPLIT_BK);
    const int nk = min(nkt - kt0, p.kchunk / SPLIT_BK) / KG;  // stages

    // this wave's DMA instructions of a stage: unit u of the KG (A, B) tiles
    const int8_t *src[LOADS];
#pragma unroll
    for (int l = 0; l < LOADS; l++) {
        const int u = (l * NW + wave) % (SUB / SPLIT_UNIT), sub = (l * NW + wave) / (SUB / SPLIT_UNIT);
        const bool isa = u < BM / 8;
        const int g = isa ? min(m0 / 8 + u, (M + 7) / 8 - 1) : min(n0 / 8 + u - BM / 8, (N + 7) / 8 - 1);
        src[l] = (isa ? p.Ap : p.Bp) + ((long)g * nkt + kt0 + sub) * SPLIT_UNIT;
    }
    const unsigned voff = lane * 16;
    auto dma1 = [&](auto Lx, int t) {
        constexpr int l = decltype(Lx)::value;
        const int8_t *b = src[l] + (long)min(t, nk - 1) * (KG * SPLIT_UNIT);
        asm("" : "+s"(b));  // a uniform base: the lane's offset stays one 32-bit register
        __builtin_amdgcn_global_load_lds(
            (const void *)(b + voff),
            (__attribute__((address_space(3))) void *)(lds + (t % STAGES) * STAGE + (l * NW + wave) * SPLIT_UNIT), 16,
            0, 0);
    };
    const unsigned lds0 = (unsigned)(uintptr_t)(const __attribute__((address_space(3))) void *)lds + kg * SUB;
    const unsigned swz = ((2 * q) ^ (r16 >> 1)) << 4;
    const unsigned a_addr = lds0 + (wm * WTM + r16) * 128 + swz, b_addr = lds0 + BM * 128 + (wn * WTN + r16) * 128 + swz;
    v4f fa[2][TMP][2], fb[2][TN][2];  // [slot][block][hi, lo]
    auto read_a = [&](auto SL, auto PH, auto R, unsigned st) {
        constexpr int sl = decltype(SL)::value, ph = decltype(PH)::value, r = decltype(R)::value, part = r & 1;
        sd_read128<(ph * TMP + (r >> 1)) * 2048>(fa[sl][r >> 1][part], st + (part ? a_addr ^ 16 : a_addr));
    };
    auto read_b = [&](auto SL, auto R, unsigned st) {
        constexpr int sl = decltype(SL)::value, r = decltype(R)::value, part = r & 1;
        sd_read128<(r >> 1) * 2048>(fb[sl][r >> 1][part], st + (part ? b_addr ^ 16 : b_addr));
    };
    auto fence_a = [&](auto SL) {
        constexpr int sl = decltype(SL)::value;
#pragma unroll
        for (int i = 0; i < TMP; i++) sd_fence(fa[sl][i][0]), sd_fence(fa[sl][i][1]);
    };
    auto fence_b = [&](auto SL) {
        constexpr int sl = decltype(SL)::value;
#pragma unroll
        for (int j = 0; j < TN; j++) sd_fence(fb[sl][j][0]), sd_fence(fb[sl][j][1]);
    };
    v4f acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) acc[i][j] = v4f{0.f, 0.f, 0.f, 0.f};
    // MFMA x of a phase: block (i, j) of term lo*hi, hi*lo, hi*hi
    constexpr int NMF = 3 * TMP * TN;
    auto mfma1 = [&](auto AS, auto BS, auto PH, auto X) {
        constexpr int as = decltype(AS)::value, bs = decltype(BS)::value, ph = decltype(PH)::value;
        constexpr int x = decltype(X)::value, term = x / (TMP * TN), i = x % (TMP * TN) / TN, j = x % TN;
        acc[ph * TMP + i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
            __builtin_bit_cast(v8h, fa[as][i][term == 0]), __builtin_bit_cast(v8h, fb[bs][j][term == 1]),
            acc[ph * TMP + i][j], 0, 0, 0);
    };
    // `items` LDS reads and DMAs spread evenly between the MFMAs of a phase
    auto mix = [&](auto ITEMS, auto AS, auto BS, auto PH, auto &&item) {
        constexpr int n = decltype(ITEMS)::value;
        static_for<0, n>([&](auto G) {
            constexpr int g = decltype(G)::value;
            __builtin_amdgcn_sched_barrier(0);
            item(G);
            __builtin_amdgcn_sched_barrier(0);
            static_for<g * NMF / n, (g + 1) * NMF / n>([&](auto X) { mfma1(AS, BS, PH, X); });
        });
        __builtin_amdgcn_sched_barrier(0);
    };

    // A phase starts when this wave's fragments of it, read during the phase
    // before, have landed. All but a stage's last read the next phase's A
    // fragments; the last waits for this wave's DMA of the next stage, crosses
    // the stage's one barrier (every wave has read this stage, every DMA of
    // the next has landed), and reads the next stage's first fragments and
    // refills this one.
    static_for<0, STAGES>([&](auto T) { static_for<0, LOADS>([&](auto Lx) { dma1(Lx, decltype(T)::value); }); });
    __builtin_amdgcn_s_waitcnt(sd_waitcnt_vm((STAGES - 1) * LOADS));
    __builtin_amdgcn_s_barrier();
    static_for<0, 2 * TN>([&](auto R) { read_b(IC<0>{}, R, 0); });
    static_for<0, 2 * TMP>([&](auto R) { read_a(IC<0>{}, IC<0>{}, R, 0); });
    auto stage = [&](auto SL, int kt) {
        constexpr int bs = decltype(SL)::value;
        const unsigned st = (kt % STAGES) * STAGE, sn = ((kt + 1) % STAGES) * STAGE;
        static_for<0, APH>([&](auto PH) {
            constexpr int ph = decltype(PH)::value, as = APH == 1 ? bs : ph & 1;
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            fence_a(IC<as>{});
            if constexpr (ph == 0) fence_b(SL);
            if constexpr (ph + 1 < APH) {
                mix(IC<2 * TMP>{}, IC<as>{}, SL, PH, [&](auto G) { read_a(IC<as ^ 1>{}, IC<ph + 1>{}, G, st); });
            } else {
                __builtin_amdgcn_s_waitcnt(sd_waitcnt_vm((STAGES - 2) * LOADS));
                __builtin_amdgcn_s_barrier();
                mix(IC<2 * TN + 2 * TMP + LOADS>{}, IC<as>{}, SL, PH, [&](auto G) {
                    constexpr int g = decltype(G)::value;
                    if constexpr (g < 2 * TN) read_b(IC<bs ^ 1>{}, G, sn);
                    else if constexpr (g < 2 * TN + 2 * TMP) read_a(IC<as ^ 1>{}, IC<0>{}, IC<g - 2 * TN>{}, sn);
                    else dma1(IC<g - 2 * TN - 2 * TMP>{}, kt + STAGES);
                });
            }
        });
    };
    int kt = 0;
    for (; kt + 1 < nk; kt += 2) {
        stage(IC<0>{}, kt);
        stage(IC<1>{}, kt + 1);
    }
    if (kt < nk) stage(IC<0>{}, kt);
    // no DMA or fragment read in flight past the loop
    __builtin_amdgcn_s_waitcnt(sd_waitcnt_vm(0));
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    fence_a(IC<0>{}), fence_a(IC<1>{}), fence_b(IC<0>{}), fence_b(IC<1>{});

    // Two K groups: group g keeps blocks [g TM/2, (g+1) TM/2) of rows and adds the
    // other group's sums of them.
    constexpr int TE = TM / KG;  // block rows of the epilogue
    if constexpr (KG == 2) {
        static_assert(BM * BN * 4 <= STAGES * STAGE, "exchange");
        __builtin_amdgcn_s_barrier();  // every wave is done with the ring
        v4f *x = reinterpret_cast<v4f *>(lds) + (wm * WN + wn) * 64 + lane;
#pragma unroll
        for (int i = 0; i < TE; i++)
#pragma unroll
            for (int j = 0; j < TN; j++)
                x[(((1 - kg) * TE + i) * TN + j) * (WM * WN * 64)] = kg ? acc[i][j] : acc[TE + i][j];
        __syncthreads();
#pragma unroll
        for (int i = 0; i < TE; i++)
#pragma unroll
            for (int j = 0; j < TN; j++) {
                const v4f o = x[((kg * TE + i) * TN + j) * (WM * WN * 64)], me = kg ? acc[TE + i][j] : acc[i][j];
                acc[i][j] = kg ? o + me : me + o;
            }
    }

    // Epilogue: scale, bias, the fused operation. Outputs of rows or columns that
    // are not finite are left to the loop after it.
    constexpr bool AUX = EPI == EPI_RESID || EPI == EPI_GELU_BWD;
    float *C = p.C + (long)blockIdx.y * M * p.ldc;
    const int row0 = m0 + wm * WTM + (KG == 2 ? kg * TE * 16 : 0) + 4 * q, col0 = n0 + wn * WTN + r16;
    float bv[TN];
    int cj[TN], en[TN];
    bool bad = false;
#pragma unroll
    for (int j = 0; j < TN; j++) {
        cj[j] = min(col0 + j * 16, N - 1);
        bv[j] = p.bias ? p.bias[cj[j]] : 0.f;
        en[j] = p.eb[cj[j]];
        bad |= en[j] == SPLIT_NONFINITE;
    }
    auto finish = [&](float v, float old, int row, int col) {
        if constexpr (EPI == EPI_GELU) {
            if (p.aux_out) p.aux_out[(long)row * p.ld_aux + col] = v;
            v = gelu_f(v);
        } else if constexpr (EPI == EPI_RESID) {
            v = old + v;
        } else if constexpr (EPI == EPI_GELU_BWD) {
            v = v * gelu_grad(old);
        } else if (p.accumulate) {
            v = old + v;
        }
        C[(long)row * p.ldc + col] = v;
    };
    auto old_of = [&](int row, int col) {
        return AUX ? p.aux_in[(long)row * p.ld_aux + col] : p.accumulate ? C[(long)row * p.ldc + col] : 0.f;
    };
#pragma unroll
    for (int i = 0; i < TE; i++) {
        float old[4][TN];
        int em[4];
#pragma unroll
        for (int v = 0; v < 4; v++) {
            const int row = min(row0 + i * 16 + v, M - 1);
            em[v] = p.ea[row];
            bad |= em[v] == SPLIT_NONFINITE;
#pragma unroll
            for (int j = 0; j < TN; j++) old[v][j] = old_of(row, cj[j]);
        }
#pragma unroll
        for (int v = 0; v < 4; v++)
#pragma unroll
            for (int j = 0; j < TN; j++) {
                const int e = em[v] + en[j];
                if (row0 + i * 16 + v < M && col0 + j * 16 < N && e < SPLIT_NONFINITE / 2)
                    finish(ldexpf(acc[i][j][v], e) + bv[j], old[v][j], row0 + i * 16 + v, cj[j]);
            }
    }
    if (!__any(bad)) return;
    const int kbeg = blockIdx.y * p.kchunk, kend = min(p.K, kbeg + p.kchunk);
    for (int x = 0; x < TE * 4 * TN; x++) {
        const int row = row0 + x / (4 * TN) * 16 + x / TN % 4, col = col0 + x % TN * 16;
        if (row >= M || col >= N || (p.ea[row] != SPLIT_NONFINITE && p.eb[col] != SPLIT_NONFINITE)) continue;
        float s = 0.f;
        for (int k = kbeg; k < kend; k++)
            s = fmaf(p.A[(long)row * p.sam + (long)k * p.sak], p.B[(long)k * p.sbk + (long)col * p.sbn], s);
        finish(s + (p.bias ? p.bias[col] : 0.f), old_of(row, col), row, col);
    }
}

// ------------------------------------------------------------------ host ----
static size_t up256(size_t x) { return (x + 255) / 256 * 256; }

// Scratch of one call: the two operands' units, exponents, and partial maxima.
struct SplitLayout {
    size_t a, b, ea, eb, pa, pb, bytes;
    SplitLayout(int M, int N, int K) {
        const size_t nk = split_units(K), nc = (K + SPLIT_KC - 1) / SPLIT_KC;
        a = 0;
        b = a + up256((size_t)((M + 7) / 8) * nk * SPLIT_UNIT);
        ea = b + up256((size_t)((N + 7) / 8) * nk * SPLIT_UNIT);
        eb = ea + up256((size_t)M * 4);
        pa = eb + up256((size_t)N * 4);
        pb = pa + up256(nc * M * 4);
        bytes = pb + up256(nc * N * 4);
    }
};

template <int NT, int G, bool MULTI = false>
static void pass1_launch(SplitJob &a, SplitJob &b, int K, hipStream_t s) {
    constexpr int RPB = NT < 256 ? 256 / NT : 1;
    for (SplitJob *j : {&a, &b})
        j->blocks = j->kcontig ? ((j->rows + 7) / 8 * 8 + RPB - 1) / RPB
                               : ((j->rows + 63) / 64) * ((K + SPLIT_KC - 1) / SPLIT_KC);
    hipLaunchKernelGGL((split_pass1_kernel<NT, G, MULTI>), dim3((unsigned)(a.blocks + b.blocks)),
                       dim3(NT < 256 ? 256 : NT), 0, s, a, b, K);
}

static hipError_t split_operands(SplitJob a, SplitJob b, int K, hipStream_t s) {
    if (K <= 512) pass1_launch<64, 1>(a, b, K, s);
    else if (K <= 1024) pass1_launch<64, 2>(a, b, K, s);
    else if (K <= 4096) pass1_launch<256, 2>(a, b, K, s);
    else if (K <= 8192) pass1_launch<256, 4>(a, b, K, s);
    else if (K <= 65536) pass1_launch<1024, 8>(a, b, K, s);
    else pass1_launch<1024, 4, true>(a, b, K, s);
    auto blocks2 = [&](const SplitJob &j) { return j.kcontig ? 0 : ((j.rows + 63) / 64) * ((K + 63) / 64); };
    const int n = blocks2(a) + blocks2(b);
    if (n) hipLaunchKernelGGL(split_pass2_kernel, dim3((unsigned)n), dim3(256), 0, s, a, b, K, blocks2(a));
    return hipGetLastError();
}

enum SplitCfg {
    SPLIT_256x256,
    SPLIT_256x192,
    SPLIT_256x128,
    SPLIT_128x128,      // two workgroups per CU
    SPLIT_128x128_KG2,  // one, of two K groups
    SPLIT_64x128_KG2,
    SPLIT_CFGS
};

// Tiles (in the order of SplitCfg) and what they were measured at, in us: one
// round of tiles over the chip takes edge + unit per 32 k. A K split also
// writes and reads its partial products, at about the copy rate.
struct SplitTile {
    int bm, bn, per_round;
    float edge, unit;
};
static const SplitTile SPLIT_TILES[] = {{256, 256, 256, 10.f, 2.2f},  {256, 192, 256, 8.f, 1.85f},
                                        {256, 128, 256, 6.f, 1.13f},  {128, 128, 512, 5.f, 1.28f},
                                        {128, 128, 256, 5.f, 0.73f},  {64, 128, 256, 4.f, 0.42f}};
constexpr double SPLIT_CUT_US = 4, SPLIT_CUT_GAIN = 0.9;  // a second launch, and the share of the time it has to save

constexpr int SPLIT_STEP = SPLIT_BK * SPLIT_KUNITS;  // a K split's granularity
static double split_us(const SplitTile &t, long tiles, int chunk) {
    return (double)((tiles + t.per_round - 1) / t.per_round) * (t.edge + t.unit * SPLIT_KUNITS * chunk);
}

// The best tile and K split of one launch, and its time in us.
static double plan_part(int M, int N, int K, SgemmF16Part &p) {
    const int steps = (K + SPLIT_STEP - 1) / SPLIT_STEP;
    double best = 1e30;
    for (int c = 0; c < SPLIT_CFGS; c++)
        for (int z = 1; z <= 16 && z * 4 <= steps + 3; z++) {
            const SplitTile &t = SPLIT_TILES[c];
            const int chunk = (steps + z - 1) / z;
            double us = split_us(t, (long)((M + t.bm - 1) / t.bm) * ((N + t.bn - 1) / t.bn) * z, chunk);
            if (z > 1) us += 4 + (2 * z + 1) * 1e-6 * M * N;
            if (us < best) best = us, p.cfg = c, p.splits = z, p.kchunk = chunk * SPLIT_STEP;
        }
    p.splits = (K + p.kchunk - 1) / p.kchunk;
    return best;
}

SgemmF16Plan plan_sgemm_f16(int M, int N, int K) {
    SgemmF16Plan p;
    // Short sums: below 96 terms the two forms' errors meet (measured 1.1e-7 of
    // the result at K = 69, both). Narrow outputs leave most of a tile idle.
    if (K < 96 || M < 128 || N < 128) return p;
    const double whole = plan_part(M, N, K, p.main);
    // Several rounds of tiles of which the last is mostly idle: the rows or
    // columns past the whole rounds (at most an eighth) become a launch of their
    // own, over smaller tiles and K splits that fill the chip, where that is
    // expected to save a tenth of the time, with tiles no smaller than before.
    // 50257 x 1024 x 4096 1373 -> 1208 us (6.2 rounds of 256x128 -> 3 of 256x256),
    // 2253 x 7717 x 799 127 -> 107, 4096 x 4097 x 700 105 -> 85, 4143 x 4187 x 155
    // 51 -> 48, eight other shapes 4-17% less. Not for a single round that does
    // not fill the chip: its tiles run at a higher clock (3521 x 2622 x 1995 125 us
    // whole and 132 cut, 3006 x 2706 x 1877 114 both ways). Nor from 256x256 to
    // smaller tiles, which read more (4883 x 5197 x 2006 307 us whole and 314 cut).
    const SplitTile &t0 = SPLIT_TILES[p.main.cfg];
    const long tiles0 = (long)((M + t0.bm - 1) / t0.bm) * ((N + t0.bn - 1) / t0.bn);
    double best = whole * SPLIT_CUT_GAIN;
    const int steps = (K + SPLIT_STEP - 1) / SPLIT_STEP;
    int cut_cfg = -1;
    for (int c = 0; c <= p.main.cfg && p.main.splits == 1 && tiles0 > t0.per_round; c++)
        for (int cols = 0; cols < 2; cols++) {
            const SplitTile &t = SPLIT_TILES[c];
            const long nm = (M + t.bm - 1) / t.bm, nn = (N + t.bn - 1) / t.bn, rounds = nm * nn / t.per_round;
            const long keep = rounds * t.per_round / (cols ? nm : nn);  // whole rows or columns of tiles
            const long cut = keep * (cols ? t.bn : t.bm), len = cols ? N : M;
            if (cut >= len || cut < len - len / 8) continue;
            SgemmF16Part rest;
            const double us = split_us(t, keep * (cols ? nm : nn), steps) + SPLIT_CUT_US +
                              (cols ? plan_part(M, N - (int)cut, K, rest) : plan_part(M - (int)cut, N, K, rest));
            if (us < best) {
                best = us, p.rest = rest;
                p.cut_m = cols ? 0 : (int)cut, p.cut_n = cols ? (int)cut : 0;
                cut_cfg = c;
            }
        }
    if (cut_cfg >= 0) p.main = {cut_cfg, 1, steps * SPLIT_STEP};
    const size_t rm = M - p.cut_m, rn = N - p.cut_n;  // of the rest
    const bool cut = p.cut_m || p.cut_n;
    const int splits = cut ? p.rest.splits : p.main.splits;  // a cut plan's main launch is not split
    if (splits > 1) p.part_bytes = (size_t)splits * rm * rn * sizeof(float);
    p.op_bytes = SplitLayout(M, N, K).bytes;
    return p;
}

template <int BM, int BN, int STAGES, int KG, int WM, int WN, int APH, int OCC>
static void gemm_launch(int epi, int splits, const SplitGemmArgs &a, hipStream_t s) {
    const dim3 grid((unsigned)(((a.M + BM - 1) / BM) * ((a.N + BN - 1) / BN)), (unsigned)splits), block(64 * KG * WM * WN);
    if (epi == EPI_GELU)
        hipLaunchKernelGGL((sgemm_split_kernel<BM, BN, STAGES, KG, WM, WN, APH, OCC, EPI_GELU>), grid, block, 0, s, a);
    else if (epi == EPI_RESID)
        hipLaunchKernelGGL((sgemm_split_kernel<BM, BN, STAGES, KG, WM, WN, APH, OCC, EPI_RESID>), grid, block, 0, s, a);
    else if (epi == EPI_GELU_BWD)
        hipLaunchKernelGGL((sgemm_split_kernel<BM, BN, STAGES, KG, WM, WN, APH, OCC, EPI_GELU_BWD>), grid, block, 0, s, a);
    else
        hipLaunchKernelGGL((sgemm_split_kernel<BM, BN, STAGES, KG, WM, WN, APH, OCC, EPI_NONE>), grid, block, 0, s, a);
}

hipError_t launch_sgemm_f16(const SgemmF16Plan &p, bool a_kcontig, bool b_kcontig, int M, int N, int K, const float *A,
                            long lda, const float *B, long ldb, const float *bias, int accumulate, float *C, long ldc,
                            const Workspace &ws, hipStream_t s, int epi, const float *aux_in, float *aux_out,
                            long ld_aux) {
    const SplitLayout L(M, N, K);
    int8_t *o = static_cast<int8_t *>(ws.operands);
    int *ea = reinterpret_cast<int *>(o + L.ea), *eb = reinterpret_cast<int *>(o + L.eb);
    auto job = [&](const float *X, long ld, int rows, bool kc, size_t P, int *ex, size_t part) {
        return SplitJob{X, ld, rows, kc, (reinterpret_cast<uintptr_t>(X) & 15) == 0 && ld % 4 == 0, o + P, ex,
                        reinterpret_cast<unsigned *>(o + part), 0};
    };
    hipError_t e = hipSuccess;
    const bool ce = p.ce.logits != nullptr;  // splits op(A) itself
    if (ce) e = launch_cross_entropy_split(p.ce, M, K, o + L.a, ea, s);
    if (e != hipSuccess) return e;
    e = split_operands(job(A, lda, ce ? 0 : M, a_kcontig, L.a, ea, L.pa), job(B, ldb, N, b_kcontig, L.b, eb, L.pb), K, s);
    if (e != hipSuccess) return e;
    const long sam = a_kcontig ? lda : 1, sak = a_kcontig ? 1 : lda, sbn = b_kcontig ? ldb : 1, sbk = b_kcontig ? 1 : ldb;
    // rows [m0, m0 + rows) and columns [n0, n0 + cols), m0 and n0 multiples of 8
    auto part = [&](const SgemmF16Part &q, int m0, int rows, int n0, int cols) {
        const bool split = q.splits > 1;
        const long unit = (long)split_units(K) * (SPLIT_UNIT / 8), at = (long)m0 * ld_aux + n0;
        float *c = C + (long)m0 * ldc + n0;
        const float *bi = bias ? bias + n0 : nullptr, *in = aux_in ? aux_in + at : nullptr;
        float *out = aux_out ? aux_out + at : nullptr;
        SplitGemmArgs a{o + L.a + m0 * unit, o + L.b + n0 * unit, ea + m0, eb + n0, A + m0 * sam, B + n0 * sbn, sam, sak,
                        sbn, sbk, split ? nullptr : bi, split ? static_cast<float *>(ws.buf) : c, split ? cols : ldc,
                        rows, cols, K, split ? 0 : accumulate, q.kchunk, in, out, ld_aux};
        const int ge = split ? EPI_NONE : epi;
        if (q.cfg == SPLIT_256x256) gemm_launch<256, 256, 2, 1, 2, 4, 4, 1>(ge, q.splits, a, s);
        else if (q.cfg == SPLIT_256x128) gemm_launch<256, 128, 3, 1, 4, 2, 1, 1>(ge, q.splits, a, s);
        else if (q.cfg == SPLIT_128x128) gemm_launch<128, 128, 2, 1, 2, 2, 1, 2>(ge, q.splits, a, s);
        else if (q.cfg == SPLIT_128x128_KG2) gemm_launch<128, 128, 2, 2, 2, 2, 1, 1>(ge, q.splits, a, s);
        else if (q.cfg == SPLIT_256x192) gemm_launch<256, 192, 2, 1, 4, 2, 2, 1>(ge, q.splits, a, s);
        else gemm_launch<64, 128, 3, 2, 1, 4, 1, 1>(ge, q.splits, a, s);
        const hipError_t g = hipGetLastError();
        if (g != hipSuccess || !split) return g;
        return launch_splitk_reduce(static_cast<const float *>(ws.buf), q.splits, rows, cols, bi, c, ldc, accumulate, epi,
                                    in, out, ld_aux, s);
    };
    if (p.cut_m) {
        e = part(p.main, 0, p.cut_m, 0, N);
        return e != hipSuccess ? e : part(p.rest, p.cut_m, M - p.cut_m, 0, N);
    }
    if (p.cut_n) {
        e = part(p.main, 0, M, 0, p.cut_n);
        return e != hipSuccess ? e : part(p.rest, 0, M, p.cut_n, N - p.cut_n);
    }
    return part(p.main, 0, M, 0, N);
}

}  // namespace pcl
