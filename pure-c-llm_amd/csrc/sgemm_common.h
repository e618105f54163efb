// sgemm_common.h -- what the FP32 GEMM kernels share: vector types, the fused
// epilogues' elementwise functions, and the LDS reads and waits written out
// where LDS DMA is in flight (the compiler would wait for all of it).
#pragma once

#include "internal.h"

namespace pcl {

typedef float v4f __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));

// ---------------------------------------------------------------------------
// Epilogues (train.c:314-333 and gpu_kernels.cu:228-243 tanh-GELU, the
// residual adds of train.c:522/527): applied to v = acc + bias.
constexpr float GELU_C = 0.7978845608028654f;  // sqrt(2/pi)
__device__ __forceinline__ float gelu_f(float x) {
    return 0.5f * x * (1.0f + tanhf(GELU_C * (x + 0.044715f * x * x * x)));
}
__device__ __forceinline__ float gelu_grad(float x) {
    const float t = tanhf(GELU_C * (x + 0.044715f * x * x * x));
    const float dudx = GELU_C * (1.0f + 3.0f * 0.044715f * x * x);
    return 0.5f * (1.0f + t) + 0.5f * x * (1.0f - t * t) * dudx;
}
// EPI_GELU: aux_out (if set) <- v, C <- gelu(v); EPI_RESID: C <- aux_in + v;
// EPI_GELU_BWD: C <- v * gelu'(aux_in)
template <int EPI>
__device__ __forceinline__ float apply_epi(float v, const float *aux_in, float *aux_out, long ai) {
    if constexpr (EPI == EPI_GELU) {
        if (aux_out) aux_out[ai] = v;
        return gelu_f(v);
    } else if constexpr (EPI == EPI_RESID) {
        return aux_in[ai] + v;
    } else if constexpr (EPI == EPI_GELU_BWD) {
        return v * gelu_grad(aux_in[ai]);
    }
    return v;
}

template <int OFF>
__device__ __forceinline__ void sd_read128(v4f &r, unsigned addr) {
    static_assert(OFF >= 0 && OFF < 65536, "ds_read offset field");
    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(r) : "v"(addr), "i"(OFF));
}
template <int OFF>
__device__ __forceinline__ void sd_read32(float &r, unsigned addr) {
    static_assert(OFF >= 0 && OFF < 65536, "ds_read offset field");
    asm volatile("ds_read_b32 %0, %1 offset:%2" : "=v"(r) : "v"(addr), "i"(OFF));
}
__device__ __forceinline__ void sd_fence(v4f &r) { asm volatile("" : "+v"(r)); }
__device__ __forceinline__ void sd_fence(float &r) { asm volatile("" : "+v"(r)); }
constexpr int sd_waitcnt_vm(int n) { return (n & 15) | (((n >> 4) & 3) << 14) | (7 << 4) | (15 << 8); }

// The second pass of a K split (sgemm.hip): C = (accumulate ? C : 0) + the partial
// products P[splits][M][N] added in split order + bias, then the epilogue.
hipError_t launch_splitk_reduce(const float *P, int splits, int M, int N, const float *bias, float *C, long ldc,
                                int accumulate, int epi, const float *aux_in, float *aux_out, long ld_aux,
                                hipStream_t stream);
// launch_sgemm's contract on the f16 matrix cores (sgemm_split.hip), any operand
// layout and alignment; ws.operands holds plan.op_bytes.
hipError_t launch_sgemm_f16(const SgemmF16Plan &plan, bool a_kcontig, bool b_kcontig, int M, int N, int K,
                            const float *A, long lda, const float *B, long ldb, const float *bias, int accumulate,
                            float *C, long ldc, const Workspace &ws, hipStream_t stream, int epi, const float *aux_in,
                            float *aux_out, long ld_aux);

}  // namespace pcl
