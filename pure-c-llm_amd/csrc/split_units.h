// split_units.h -- the two-f16 form of an FP32 operand (sgemm_split.hip has the
// arithmetic), for the kernels that write it.
#pragma once
#include "internal.h"

namespace pcl {

typedef _Float16 v8h __attribute__((ext_vector_type(8)));

constexpr int SPLIT_BK = 32;                // k per unit
constexpr int SPLIT_KUNITS = 2;             // operands are padded to this many units of k
constexpr int SPLIT_UNIT = 1024;            // bytes of 8 rows x 32 k
constexpr int SPLIT_NONFINITE = 1 << 28;    // exponent of a row with inf or NaN

__host__ __device__ constexpr int split_units(int K) {
    return (K + SPLIT_BK * SPLIT_KUNITS - 1) / (SPLIT_BK * SPLIT_KUNITS) * SPLIT_KUNITS;
}

// A row's scale from the bits of its largest |a|: shift to add to the exponents
// of its elements, or none if it is not finite.
__device__ __forceinline__ bool split_shift(unsigned amax, int &shift) {
    if (amax >= 0x7f800000u) return shift = 0, false;
    if (amax == 0) return shift = 0, true;
    const int e = amax >= 0x00800000u ? (int)(amax >> 23) - 127 : -118 - __clz((int)amax);
    return shift = 14 - e, true;
}

__device__ __forceinline__ void split_value(float a, int shift, bool finite, _Float16 &hi, _Float16 &lo) {
    const float x = finite ? ldexpf(a, shift) : 0.f;
    hi = (_Float16)x;
    lo = (_Float16)(x - (float)hi);
}

// Eight consecutive k of one row: hi and lo at the unit's two chunks.
__device__ __forceinline__ void split_store(int8_t *P, int nk, int row, int k, const float (&a)[8], int shift,
                                            bool finite) {
    v8h hi, lo;
#pragma unroll
    for (int e = 0; e < 8; e++) {
        _Float16 h, l;
        split_value(a[e], shift, finite, h, l);
        hi[e] = h, lo[e] = l;
    }
    int8_t *u = P + ((long)(row >> 3) * nk + (k >> 5)) * SPLIT_UNIT + (row & 7) * 128;
    const int c = (k >> 3 & 3) * 2, key = row >> 1 & 7;
    *reinterpret_cast<v8h *>(u + ((c ^ key) << 4)) = hi;
    *reinterpret_cast<v8h *>(u + (((c + 1) ^ key) << 4)) = lo;
}

__device__ __forceinline__ unsigned split_mag(float x) { return __float_as_uint(x) & 0x7fffffffu; }

}  // namespace pcl
