// block_ops.h -- small dense block helpers of the device code (row-major, BS =
// 2 or 3).
#pragma once

#include <hip/hip_runtime.h>

namespace omodels {

template <int BS, class S>
__device__ __forceinline__ void bMatmul(const S* A, const S* B, S* C)
{
#pragma unroll
    for (int i = 0; i < BS; ++i)
#pragma unroll
        for (int j = 0; j < BS; ++j) {
            S s = A[i * BS] * B[j];
#pragma unroll
            for (int k = 1; k < BS; ++k) s += A[i * BS + k] * B[k * BS + j];
            C[i * BS + j] = s;
        }
}

template <int BS, class S>
__device__ __forceinline__ bool bInvert(S* a)
{
    if (BS == 2) {
        S det = a[0] * a[3] - a[1] * a[2];
        if (!(det != S(0)) || !isfinite((double)det)) return false;
        S r = S(1) / det;
        S i00 = a[3] * r, i01 = -a[1] * r, i10 = -a[2] * r, i11 = a[0] * r;
        a[0] = i00; a[1] = i01; a[2] = i10; a[3] = i11;
        return true;
    } else {
        S c00 = a[4] * a[8] - a[5] * a[7];
        S c01 = a[5] * a[6] - a[3] * a[8];
        S c02 = a[3] * a[7] - a[4] * a[6];
        S det = a[0] * c00 + a[1] * c01 + a[2] * c02;
        if (!(det != S(0)) || !isfinite((double)det)) return false;
        S r = S(1) / det;
        S c10 = a[2] * a[7] - a[1] * a[8];
        S c11 = a[0] * a[8] - a[2] * a[6];
        S c12 = a[1] * a[6] - a[0] * a[7];
        S c20 = a[1] * a[5] - a[2] * a[4];
        S c21 = a[2] * a[3] - a[0] * a[5];
        S c22 = a[0] * a[4] - a[1] * a[3];
        a[0] = c00 * r; a[1] = c10 * r; a[2] = c20 * r;
        a[3] = c01 * r; a[4] = c11 * r; a[5] = c21 * r;
        a[6] = c02 * r; a[7] = c12 * r; a[8] = c22 * r;
        return true;
    }
}

}  // namespace omodels
