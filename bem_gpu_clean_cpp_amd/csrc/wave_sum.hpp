// Sums over the 64 lanes of a wave (device code).
#pragma once

#include <hip/hip_runtime.h>

namespace bem {

// Sums x[v] (V a power of two, at most 64) over the 64 lanes: afterwards lane
// l holds the total of x[v(l)] in x[0], v(l) = the V-value index whose bits are
// the high bits of l (bit H of the lane picks the upper half at each step).
template <int V>
__device__ __forceinline__ void reduce_scatter(double (&x)[V], int lane) {
    int mask = 32;
#pragma unroll
    for (int h = V / 2; h >= 1; h >>= 1) {
        const bool up = (lane & mask) != 0;
#pragma unroll
        for (int i = 0; i < h; i++) {
            // (selected as values: a select of the two addresses puts x in
            // scratch memory)
            const double lo = x[i], hi = x[i + h];
            const double send = up ? lo : hi, keep = up ? hi : lo;
            x[i] = keep + __shfl_xor(send, mask, 64);
        }
        mask >>= 1;
    }
    for (; mask >= 1; mask >>= 1) x[0] += __shfl_xor(x[0], mask, 64);
}

}  // namespace bem
