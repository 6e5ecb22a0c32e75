// What stays certain about an MSA column whose weights are known to within an error.
//
// After refinement rounds that subtract removed candidates, each weight of a column with
// candidates of its base differs from the sum over the kept candidates by at most
// `weightError`; the weight of a base without any is exactly 0.
#pragma once

#include <hip/hip_runtime.h>

// Most that the column's support (largest weight / sum) can be off; above 1 where the sum is too
// small for a bound. With the sum off by at most 4 e and the largest weight by e, the support is
// off by at most 3 e / (sum - 4 e), which 6 e / sum covers where sum > 8 e; the rest of the
// factor 24 and 1e-6 are for the rounding of both divisions and sums.
__host__ __device__ inline float supportError(float sum, float weightError){
    return sum > 24.0f * weightError ? 6.0f * weightError / sum + 1e-6f : 2.0f;
}

// Whether the largest of the weights (0 for bases without candidates) is the largest of the exact
// ones. `bases` of the four have candidates; a weight of 0 says nothing about that, a small one can
// vanish in the subtraction.
__host__ __device__ inline bool consensusCertain(float w0, float w1, float w2, float w3, int bases, float weightError){
    const float w01 = fmaxf(w0, w1), v01 = fminf(w0, w1);
    const float w23 = fmaxf(w2, w3), v23 = fminf(w2, w3);
    const float first = fmaxf(w01, w23), second = fmaxf(fminf(w01, w23), fmaxf(v01, v23));
    return bases == 1 ? first > 0.0f : first - second > 2.0f * weightError + 1e-6f;
}
