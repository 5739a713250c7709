// Sorting within one wavefront.
#pragma once
#include "common.hpp"

namespace feasm {

// Orders one wavefront's LDS accesses among themselves (LDS that no other
// wavefront uses needs no workgroup barrier).
__device__ __forceinline__ void wave_fence() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Ascending bitonic sort of 64 E values held by one wavefront in
// registers: lane l holds entries l + 64 m.  Partners less than 64 apart
// are exchanged with lane shuffles, partners 64 or more apart sit in two
// registers of the same lane.
template <int E, typename T>
__device__ __forceinline__ void wave_sort(T (&x)[E], int lane) {
#pragma unroll
    for (int k = 2; k <= 64 * E; k <<= 1)
#pragma unroll
        for (int j = k >> 1; j > 0; j >>= 1) {
            if (j >= 64) {
                const int jj = j >> 6;
#pragma unroll
                for (int m = 0; m < E; m++) {
                    const int mp = m ^ jj;
                    if (mp > m) {
                        const bool up = ((lane + 64 * m) & k) == 0;
                        T &a = x[m];
                        T &b = x[mp < E ? mp : m];
                        const T lo = min(a, b), hi = max(a, b);
                        a = up ? lo : hi;
                        b = up ? hi : lo;
                    }
                }
            } else {
#pragma unroll
                for (int m = 0; m < E; m++) {
                    const int i = lane + 64 * m;
                    const T y = lane_xor(x[m], j, lane);
                    const bool take_min = ((i & k) == 0) == ((i & j) == 0);
                    x[m] = take_min ? min(x[m], y) : max(x[m], y);
                }
            }
        }
}

}  // namespace feasm
