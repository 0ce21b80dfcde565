// wavesort.hpp -- bitonic sort of 64 R keys in the registers of one wavefront.
#pragma once
#include <hip/hip_runtime.h>

namespace blqh {

// v[0..R) of lane l are elements l R .. l R + R - 1; ascending over the wavefront on
// return.  Steps at distances below R stay in the lane, the others exchange with one
// other lane: 21 of the 45 steps for 512 keys, against a load and a store of
// LDS per key and step and a barrier per step.
template <int R, class K>
__device__ __forceinline__ void wave_sort(K (&v)[R]) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int k = 2; k <= 64 * R; k <<= 1) {
#pragma unroll
        for (int j = k >> 1; j > 0; j >>= 1) {
            if (j >= R) {
                // the lane keeps the smaller key if it is the lower of an ascending pair
                const bool keep_min = ((lane & (j / R)) == 0) == ((lane * R & k) == 0);
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    const K o = __shfl_xor(v[r], j / R, 64);
                    v[r] = keep_min == (o < v[r]) ? o : v[r];
                }
            } else {
#pragma unroll
                for (int r = 0; r < R; ++r)
                    if ((r & j) == 0) {
                        const bool up = ((lane * R + r) & k) == 0;
                        const K a = v[r], b = v[r | j];
                        const bool swap = (b < a) == up;
                        v[r] = swap ? b : a;
                        v[r | j] = swap ? a : b;
                    }
            }
        }
    }
}

// buf[0, 64 R) in LDS, read and written by this wavefront only
template <int R, class K>
__device__ __forceinline__ void sort_lds(K* buf) {
    const int at = (threadIdx.x & 63) * R;
    K v[R];
#pragma unroll
    for (int r = 0; r < R; ++r) v[r] = buf[at + r];
    wave_sort<R, K>(v);
#pragma unroll
    for (int r = 0; r < R; ++r) buf[at + r] = v[r];
}

}  // namespace blqh
