// hadamard.h -- the wave's Walsh-Hadamard butterflies of the TurboQuant rotation.
#pragma once

#include <hip/hip_runtime.h>

namespace imh_tq {

// Strides 1..32 of the unnormalised fast Walsh-Hadamard transform of a
// 64-element vector held one element per lane: at stride s the pair (j, j + s)
// becomes (x_j + x_{j+s}, x_j - x_{j+s}), strides in increasing order.
__device__ __forceinline__ float hadamard64(float x, int lane) {
#pragma unroll
    for (int step = 1; step < 64; step *= 2) {
        const float p = __shfl_xor(x, step);
        x = (lane & step) ? p - x : x + p;   // element j + step of the pair: x_j - x_{j+step}
    }
    return x;
}

}  // namespace imh_tq
