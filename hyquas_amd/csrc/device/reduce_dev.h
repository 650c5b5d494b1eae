// reduce_dev.h -- wave reductions shared by the readout kernels.
#pragma once

#include <hip/hip_runtime.h>

namespace hq {

// Sum over the 64 lanes of each of the N columns v[0..N) (N <= 64), N <= 64;
// called with M = 32, lane L returns column bitreverse6(L) (its low log2
// bits, where N is a power of two).  Every step folds pairs of columns into
// one, each half of the wave keeping one of the pair: about N shuffles instead
// of 6 N.
template <int N, int M>
__device__ __forceinline__ double wave_columns(double* v, int lane)
{
    if constexpr (M == 0) {
        return v[0];
    } else {
        const bool up = (lane & M) != 0;
#pragma unroll
        for (int i = 0; i < (N + 1) / 2; i++) {
            if (2 * i + 1 < N) {
                const double keep = up ? v[2 * i + 1] : v[2 * i];
                const double send = up ? v[2 * i] : v[2 * i + 1];
                v[i] = keep + __shfl_xor(send, M);
            } else {
                v[i] = v[2 * i] + __shfl_xor(v[2 * i], M);
            }
        }
        return wave_columns<(N + 1) / 2, M / 2>(v, lane);
    }
}

// Inclusive prefix sum over the 64 lanes.
__device__ __forceinline__ double wave_scan(double v, int lane)
{
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const double u = __shfl_up(v, o);
        if (lane >= o) v += u;
    }
    return v;
}

}  // namespace hq
