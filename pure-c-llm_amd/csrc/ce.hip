// ce.hip -- softmax cross-entropy over rows of logits (train.c:449-465,
// gpu_kernels.cu:518-547): per row m with target t,
//   p[v] = expf(l[v] - max) * (1 / sum_v expf(l[v] - max)),
//   loss_m = -log((double)p[t] + 1e-30),  dl[v] = (p[v] - [v == t]) / M.
//
// One workgroup per row. Rows whose logits and dlogits share their alignment
// and that fit a workgroup's registers (ce_row_regs_kernel) are read once, with
// one exponential per element; others take two passes over the row in HBM
// (ce_rows_kernel): the first keeps a running (max, sum) per thread (the sum
// rescaled whenever the max grows), the second writes dl. dl may alias the
// logits (each element is read before the same thread overwrites it). Row losses go to a double array; a second kernel
// adds their mean, summed in a fixed order, into *loss. Columns [V, pad) of dl
// are written as zeros so a padded dl can feed K-padded products.
#include "internal.h"
#include "split_units.h"

namespace pcl {
namespace {

constexpr int CE_NT = 512;  // 8 waves per row

// (m, s) += x: s holds sum exp(x_i - m). NaN logits propagate into s; -inf
// logits add nothing.
__device__ __forceinline__ void ce_push(float &m, float &s, float x) {
    const float d = x - m;
    if (d > 0.f) {
        s = s * expf(-d) + 1.f;
        m = x;
    } else if (x != -INFINITY) {
        s += expf(d);
    }
}

__device__ __forceinline__ void ce_merge(float &m, float &s, float m2, float s2) {
    if (s2 == 0.f) return;
    if (s == 0.f) {
        m = m2, s = s2;
        return;
    }
    if (m2 > m) {
        s = s * expf(m - m2) + s2;
        m = m2;
    } else {
        s += s2 * expf(m2 - m);
    }
}

__global__ __launch_bounds__(CE_NT) void ce_rows_kernel(const float *logits, long ld,
                                                        const int *__restrict__ targets, float *dl,
                                                        long ldd, int V, int pad, float rows,
                                                        double *__restrict__ row_loss) {
    typedef float v4f_t __attribute__((ext_vector_type(4)));
    __shared__ float sm_m[CE_NT / 64], sm_s[CE_NT / 64];
    const int tid = threadIdx.x, row = blockIdx.x;
    const float *x = logits + (long)row * ld;
    float *o = dl + (long)row * ldd;
    // Rows are read (and written) as 16-byte vectors between a scalar head (up
    // to the first 16-byte boundary) and a scalar tail, when the dlogits row
    // has the same alignment as the logits row; otherwise element by element.
    const bool vec = ((reinterpret_cast<uintptr_t>(x) ^ reinterpret_cast<uintptr_t>(o)) & 15) == 0;
    const int head = vec ? min(V, (int)((16 - (reinterpret_cast<uintptr_t>(x) & 15)) & 15) / 4) : V;
    const int nv = vec ? (V - head) / 4 : 0;
    const int tail0 = head + 4 * nv;
    const v4f_t *x4 = reinterpret_cast<const v4f_t *>(x + head);
    float m = -INFINITY, s = 0.f;
    if (vec) {
        if (tid < head) ce_push(m, s, x[tid]);
        int c = tid;
        for (; c + CE_NT < nv; c += 2 * CE_NT) {
            const v4f_t a = x4[c], b = x4[c + CE_NT];
            ce_push(m, s, a[0]), ce_push(m, s, a[1]), ce_push(m, s, a[2]), ce_push(m, s, a[3]);
            ce_push(m, s, b[0]), ce_push(m, s, b[1]), ce_push(m, s, b[2]), ce_push(m, s, b[3]);
        }
        for (; c < nv; c += CE_NT) {
            const v4f_t a = x4[c];
            ce_push(m, s, a[0]), ce_push(m, s, a[1]), ce_push(m, s, a[2]), ce_push(m, s, a[3]);
        }
        for (int v = tail0 + tid; v < V; v += CE_NT) ce_push(m, s, x[v]);
    } else {
        int v = tid;
        for (; v + 3 * CE_NT < V; v += 4 * CE_NT) {
            const float x0 = x[v], x1 = x[v + CE_NT], x2 = x[v + 2 * CE_NT], x3 = x[v + 3 * CE_NT];
            ce_push(m, s, x0);
            ce_push(m, s, x1);
            ce_push(m, s, x2);
            ce_push(m, s, x3);
        }
        for (; v < V; v += CE_NT) ce_push(m, s, x[v]);
    }
#pragma unroll
    for (int sh = 32; sh > 0; sh >>= 1) {
        const float m2 = __shfl_xor(m, sh), s2 = __shfl_xor(s, sh);
        ce_merge(m, s, m2, s2);
    }
    if ((tid & 63) == 0) sm_m[tid >> 6] = m, sm_s[tid >> 6] = s;
    __syncthreads();
    m = sm_m[0], s = sm_s[0];
#pragma unroll
    for (int w = 1; w < CE_NT / 64; w++) ce_merge(m, s, sm_m[w], sm_s[w]);
    const float inv = 1.0f / s;
    const int t = targets[row];
    if (tid == 0 && (t < 0 || t >= V)) row_loss[row] = __longlong_as_double(0x7ff8000000000000LL);
    // p = expf(x - m) * inv; dl = (p - [v == t]) / rows; the target's loss term
    auto one = [&](int v, float xv) {
        const float p = expf(xv - m) * inv;
        if (v == t) row_loss[row] = -log((double)p + 1e-30);
        return (p - (v == t ? 1.0f : 0.0f)) / rows;
    };
    if (vec) {
        if (tid < head) o[tid] = one(tid, x[tid]);
        v4f_t *o4 = reinterpret_cast<v4f_t *>(o + head);
        for (int c = tid; c < nv; c += CE_NT) {
            const v4f_t a = x4[c];
            const int v0 = head + 4 * c;
            o4[c] = v4f_t{one(v0, a[0]), one(v0 + 1, a[1]), one(v0 + 2, a[2]), one(v0 + 3, a[3])};
        }
        for (int v = tail0 + tid; v < V; v += CE_NT) o[v] = one(v, x[v]);
        for (int v = V + tid; v < pad; v += CE_NT) o[v] = 0.f;
        return;
    }
    int v = tid;
    for (; v + 3 * CE_NT < V; v += 4 * CE_NT) {
        float p[4];
#pragma unroll
        for (int u = 0; u < 4; u++) p[u] = expf(x[v + u * CE_NT] - m) * inv;
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const int vv = v + u * CE_NT;
            if (vv == t) row_loss[row] = -log((double)p[u] + 1e-30);
            o[vv] = (p[u] - (vv == t ? 1.0f : 0.0f)) / rows;
        }
    }
    for (; v < V; v += CE_NT) {
        const float p = expf(x[v] - m) * inv;
        if (v == t) row_loss[row] = -log((double)p + 1e-30);
        o[v] = (p - (v == t ? 1.0f : 0.0f)) / rows;
    }
    for (v = V + tid; v < pad; v += CE_NT) o[v] = 0.f;
}

// f over the block's values, the same on every thread.
template <typename T, typename F>
__device__ __forceinline__ T ce_block(T v, T *red, F f) {
#pragma unroll
    for (int sh = 32; sh > 0; sh >>= 1) v = f(v, (T)__shfl_xor(v, sh));
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    v = red[0];
#pragma unroll
    for (int w = 1; w < CE_NT / 64; w++) v = f(v, red[w]);
    return v;
}

// The same rows held in registers between the passes: NV 16-byte pieces per
// thread. Bound by HBM, one read and one write of the row; two workgroups per CU
// at the largest NV (128 registers), so one row's loads run under the other's
// stores. The row has a scalar head up to its first 16-byte boundary
// and a scalar tail, together at most 6 elements, one more per thread. POW2: rows
// is a power of two, and dividing by it is multiplying by its reciprocal, exactly.
// 4096 rows of 50257: 319 us, 5.2 TB/s (a copy reaches 6.2); the two-pass
// kernel, with its second read and two exponentials per element, took 165 us more.
//
// SPLIT: the gradient's rows are also written in the two-f16 form that d_lnf's
// product takes (bit for bit what its split pass would make of dl), while they
// are in registers, instead of that pass's read and write. A thread's pieces
// then lie in pairs, eight consecutive entries, and the up to seven entries past
// the last eight are the scalar ones. The same rows: 531 us, 4.7 TB/s, against
// 319 and 339 for the two; head with cross-entropy 4161 -> 4035 us.
template <int NV, bool POW2, bool SPLIT>
__global__ __launch_bounds__(CE_NT, 4) void ce_row_regs_kernel(const float *logits, long ld,
                                                               const int *__restrict__ targets, float *dl,
                                                               long ldd, int V, int pad, float rows,
                                                               double *__restrict__ row_loss, int M, int8_t *units,
                                                               int *ex) {
    typedef float v4f_t __attribute__((ext_vector_type(4)));
    __shared__ float red[2][CE_NT / 64];
    __shared__ unsigned redu[CE_NT / 64];
    __shared__ float ends[8];  // SPLIT: the entries past the last whole eight
    const int tid = threadIdx.x, row = blockIdx.x;
    const float *x = logits + (long)row * ld;
    float *o = dl + (long)row * ldd;
    // this thread's piece i: lane0 + the first entry of piece i
    auto first = [](int i) { return SPLIT ? (i >> 1) * 2 * CE_NT + (i & 1) : i * CE_NT; };
    const int lane0 = SPLIT ? 2 * tid : tid;
    const int nk = split_units(V);
    if (SPLIT && row >= M) {  // rows up to the last unit's are zeros
        const float zero[8] = {};
        for (int k = 8 * tid; k < pad; k += 8 * CE_NT) split_store(units, nk, row, k, zero, 0, true);
        return;
    }
    const int head = SPLIT ? 0 : min(V, (int)((16 - (reinterpret_cast<uintptr_t>(x) & 15)) & 15) / 4);
    const int nv = SPLIT ? V / 8 * 2 : (V - head) / 4, tail = V - head - 4 * nv;
    auto has = [&](int i) { return first(SPLIT ? i & ~1 : i) + lane0 < nv; };  // a pair lies in the row whole
    const int ve = tid < head ? tid : tid < head + tail ? 4 * nv + tid : -1;  // this thread's scalar element
    const v4f_t *x4 = reinterpret_cast<const v4f_t *>(x + head);
    v4f_t a[NV];
#pragma unroll
    for (int i = 0; i < NV; i++) {
        a[i] = v4f_t{-INFINITY, -INFINITY, -INFINITY, -INFINITY};
        if (has(i)) a[i] = (x4 + first(i))[lane0];
    }
    float ae = ve >= 0 ? x[ve] : -INFINITY;
    const int t = targets[row];
    float m = ae;  // a NaN is dropped here and reaches the sum
#pragma unroll
    for (int i = 0; i < NV; i++) m = fmaxf(fmaxf(m, fmaxf(a[i][0], a[i][1])), fmaxf(a[i][2], a[i][3]));
    m = ce_block(m, red[0], [](float u, float v) { return fmaxf(u, v); });
    float s = ae = expf(ae - m);
#pragma unroll
    for (int i = 0; i < NV; i++) {
        __builtin_amdgcn_sched_barrier(0);  // one piece's temporaries at a time
#pragma unroll
        for (int e = 0; e < 4; e++) a[i][e] = expf(a[i][e] - m);
        s += (a[i][0] + a[i][1]) + (a[i][2] + a[i][3]);
    }
    if (m == INFINITY) {  // counts the infinite logits (each has exp(inf - inf) in its register)
        s = 0.f;
        for (int v = tid; v < V; v += CE_NT) s += x[v] == m ? 1.f : x[v] == x[v] ? 0.f : x[v];
    }
    s = ce_block(s, red[1], [](float u, float v) { return u + v; });
    if (m == INFINITY && s > 1.f) s = __builtin_nanf("");  // two of them: no finite element
    const float inv = 1.0f / s;
    if (tid == 0 && (t < 0 || t >= V)) row_loss[row] = __longlong_as_double(0x7ff8000000000000LL);
    const float r = 1.0f / rows;
    float pt = -1.f;  // p[t] on the thread that holds it
    auto one = [&](bool target, float ev) {
        const float p = ev * inv, d = p - (target ? 1.0f : 0.0f);
        pt = target ? p : pt;
        return POW2 ? d * r : d / rows;
    };
    if (ve >= 0) o[ve] = one(ve == t, ae);
    const int t0 = t - head - 4 * lane0;  // the target, from this thread's first piece
    unsigned mag = 0;
    if (SPLIT && tid < 8) {
        const float d = ve >= 0 ? one(ve == t, ae) : 0.f;
        ends[tid] = d, mag = split_mag(d);
    }
    v4f_t *o4 = reinterpret_cast<v4f_t *>(o + head);
#pragma unroll
    for (int i = 0; i < NV; i++) {
        __builtin_amdgcn_sched_barrier(0);
        const int v = 4 * first(i);
        if (has(i)) {
            a[i] = v4f_t{one(v == t0, a[i][0]), one(v + 1 == t0, a[i][1]), one(v + 2 == t0, a[i][2]),
                         one(v + 3 == t0, a[i][3])};
            (o4 + first(i))[lane0] = a[i];
#pragma unroll
            for (int e = 0; SPLIT && e < 4; e++) mag = max(mag, split_mag(a[i][e]));
        }
    }
    if constexpr (SPLIT) {
        mag = ce_block(mag, redu, [](unsigned u, unsigned v) { return max(u, v); });
        int shift;
        const bool finite = split_shift(mag, shift);
        if (tid < (pad - 4 * nv) / 8) {
            float d[8];
#pragma unroll
            for (int e = 0; e < 8; e++) d[e] = tid == 0 ? ends[e] : 0.f;
            split_store(units, nk, row, 4 * nv + 8 * tid, d, shift, finite);
        }
        if (tid == 0) ex[row] = finite ? -shift : SPLIT_NONFINITE;
        // the addresses of split_store, with the lane's part in 32 bits
        int8_t *base = units + (long)(row >> 3) * nk * SPLIT_UNIT + (row & 7) * 128;
        const unsigned lane = (8 * tid / SPLIT_BK) * SPLIT_UNIT, c = (tid & 3) * 2, key = row >> 1 & 7;
        const unsigned at_hi = lane + ((c ^ key) << 4), at_lo = lane + (((c + 1) ^ key) << 4);
#pragma unroll
        for (int i = 0; i < NV; i += 2) {
            __builtin_amdgcn_sched_barrier(0);
            v8h hi, lo;
#pragma unroll
            for (int e = 0; e < 8; e++) {
                _Float16 h, l;
                split_value(a[i + e / 4][e % 4], shift, finite, h, l);
                hi[e] = h, lo[e] = l;
            }
            if (has(i)) {
                int8_t *u = base + (long)(i >> 1) * (8 * CE_NT / SPLIT_BK) * SPLIT_UNIT;
                *reinterpret_cast<v8h *>(u + at_hi) = hi;
                *reinterpret_cast<v8h *>(u + at_lo) = lo;
            }
        }
    }
    if (!(pt < 0.f)) row_loss[row] = -log((double)pt + 1e-30);
    for (int v = V + tid; v < pad; v += CE_NT) o[v] = 0.f;
}

// *loss += (float)(sum_m row_loss[m] / rows), the sum in a fixed order.
__global__ __launch_bounds__(256) void ce_loss_kernel(const double *__restrict__ row_loss, int M,
                                                      double rows, float *__restrict__ loss) {
    __shared__ double red[4];
    double a = 0.0;
    for (int i = threadIdx.x; i < M; i += 256) a += row_loss[i];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) a += __shfl_xor(a, o);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = a;
    __syncthreads();
    if (threadIdx.x == 0) loss[0] += (float)((((red[0] + red[1]) + red[2]) + red[3]) / rows);
}

}  // namespace

hipError_t launch_cross_entropy(const float *logits, long ld, const int *targets, float *dl,
                                long ldd, int M, int V, int pad, int rows, double *row_loss,
                                hipStream_t s) {
    if (M <= 0) return hipSuccess;
    // every logits row at its dlogits row's offset from a 16-byte boundary
    const bool same = ((reinterpret_cast<uintptr_t>(logits) ^ reinterpret_cast<uintptr_t>(dl)) & 15) == 0 &&
                      (ld - ldd) % 4 == 0;
    // 25 pieces fill the 128 registers that two workgroups per CU leave a thread
    const int pieces = (V + 4 * CE_NT - 1) / (4 * CE_NT);  // 16-byte pieces per thread
    if (!same || pieces > 25) {
        hipLaunchKernelGGL(ce_rows_kernel, dim3((unsigned)M), dim3(CE_NT), 0, s, logits, ld, targets, dl, ldd, V, pad,
                           (float)rows, row_loss);
        return hipGetLastError();
    }
    auto launch = [&](auto general, auto pow2) {
        hipLaunchKernelGGL(rows & (rows - 1) ? general : pow2, dim3((unsigned)M), dim3(CE_NT), 0, s, logits, ld, targets,
                           dl, ldd, V, pad, (float)rows, row_loss, M, nullptr, nullptr);
    };
    if (pieces <= 1) launch(ce_row_regs_kernel<1, false, false>, ce_row_regs_kernel<1, true, false>);
    else if (pieces <= 4) launch(ce_row_regs_kernel<4, false, false>, ce_row_regs_kernel<4, true, false>);
    else if (pieces <= 8) launch(ce_row_regs_kernel<8, false, false>, ce_row_regs_kernel<8, true, false>);
    else if (pieces <= 16) launch(ce_row_regs_kernel<16, false, false>, ce_row_regs_kernel<16, true, false>);
    else launch(ce_row_regs_kernel<25, false, false>, ce_row_regs_kernel<25, true, false>);
    return hipGetLastError();
}

hipError_t launch_cross_entropy_split(const CeRows &c, int M, int V, int8_t *units, int *ex, hipStream_t s) {
    if (M <= 0) return hipSuccess;
    static_assert(CE_SPLIT_PAD == 26 * 4 * CE_NT, "pieces of the largest kernel");
    if (c.pad > CE_SPLIT_PAD || c.pad != split_units(V) * SPLIT_BK || (reinterpret_cast<uintptr_t>(c.logits) & 15))
        return hipErrorInvalidValue;
    const int pieces = (c.pad + 4 * CE_NT - 1) / (4 * CE_NT);
    auto launch = [&](auto general, auto pow2) {
        hipLaunchKernelGGL(c.rows & (c.rows - 1) ? general : pow2, dim3((unsigned)(M + 7) / 8 * 8), dim3(CE_NT), 0, s,
                           c.logits, (long)c.pad, c.targets, c.logits, (long)c.pad, V, c.pad, (float)c.rows, c.row_loss,
                           M, units, ex);
    };
    if (pieces <= 8) launch(ce_row_regs_kernel<8, false, true>, ce_row_regs_kernel<8, true, true>);
    else if (pieces <= 16) launch(ce_row_regs_kernel<16, false, true>, ce_row_regs_kernel<16, true, true>);
    else launch(ce_row_regs_kernel<26, false, true>, ce_row_regs_kernel<26, true, true>);
    return hipGetLastError();
}

hipError_t launch_ce_loss(const double *row_loss, int M, int rows, float *loss, hipStream_t s) {
    if (M <= 0) return hipSuccess;
    hipLaunchKernelGGL(ce_loss_kernel, dim3(1), dim3(256), 0, s, row_loss, M, (double)rows, loss);
    return hipGetLastError();
}

}  // namespace pcl
