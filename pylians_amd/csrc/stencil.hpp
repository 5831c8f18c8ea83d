// Stencils and cell arithmetic shared by the cell-binned deposits (binned.hip, binned2d.hip).
#pragma once
#include <math.h>

#include "common.hpp"

namespace pyl {

// Lowest stencil cell (unwrapped) and the float64 1-D weights; the same arithmetic as the
// stencils of deposit.hip (MAS_library.pyx:151-157, 290, 393-399, 486-492).
template <int S> struct Axis;
template <> struct Axis<1> {
    static __device__ __forceinline__ double eval(double d, double* w) {
        w[0] = 1.0;
        return floor(d + 0.5);
    }
};
template <> struct Axis<2> {
    static __device__ __forceinline__ double eval(double d, double* w) {
        const double b = floor(d);
        const double u = d - b;
        w[0] = 1.0 - u;
        w[1] = u;
        return b;
    }
};
template <> struct Axis<3> {
    static __device__ __forceinline__ double eval(double d, double* w) {
        const double mn = floor(d - 1.5);
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            const double s = fabs(mn + (j + 1) - d);
            w[j] = s < 0.5 ? 0.75 - s * s : (s < 1.5 ? 0.5 * (1.5 - s) * (1.5 - s) : 0.0);
        }
        return mn + 1.0;
    }
};
template <> struct Axis<4> {
    static __device__ __forceinline__ double eval(double d, double* w) {
        const double mn = floor(d - 2.0);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const double s = fabs(mn + (j + 1) - d);
            w[j] = s < 1.0 ? (4.0 - 6.0 * s * s + 3.0 * s * s * s) / 6.0
                           : (s < 2.0 ? (2.0 - s) * (2.0 - s) * (2.0 - s) / 6.0 : 0.0);
        }
        return mn + 1.0;
    }
};

// The same stencils with the 1-D weights evaluated in float32 from the float64 cell fraction
// (CIC: u and 1 - u in float64, each rounded once; TSC/PCS: the distance |cell - d| and its
// distance to the stencil's outer edge in float64, each rounded once, then the polynomials in
// float32, so that no weight loses precision to cancellation); the lowest cell is the float64 one.
template <int S> struct Axis32;
template <> struct Axis32<1> {
    static __device__ __forceinline__ double eval(double d, float* w) {
        w[0] = 1.0f;
        return floor(d + 0.5);
    }
};
template <> struct Axis32<2> {
    static __device__ __forceinline__ double eval(double d, float* w) {
        const double b = floor(d);
        const double u = d - b;
        w[0] = (float)(1.0 - u);
        w[1] = (float)u;
        return b;
    }
};
template <> struct Axis32<3> {
    static __device__ __forceinline__ double eval(double d, float* w) {
        const double mn = floor(d - 1.5);
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            const double s = fabs(mn + (j + 1) - d);
            const float sf = (float)s, t = (float)(1.5 - s);   // distance to the outer edge, exact first
            w[j] = s < 0.5 ? 0.75f - sf * sf : (s < 1.5 ? 0.5f * t * t : 0.0f);
        }
        return mn + 1.0;
    }
};
template <> struct Axis32<4> {
    static __device__ __forceinline__ double eval(double d, float* w) {
        const double mn = floor(d - 2.0);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const double s = fabs(mn + (j + 1) - d);
            const float sf = (float)s, t = (float)(2.0 - s);
            w[j] = s < 1.0 ? (4.0f - 6.0f * sf * sf + 3.0f * sf * sf * sf) * (1.0f / 6.0f)
                           : (s < 2.0 ? t * t * t * (1.0f / 6.0f) : 0.0f);
        }
        return mn + 1.0;
    }
};

// periodic cell index of an integral float64 cell coordinate b (positions inside the box give
// 0 <= b < N directly, a stencil edge at most one box away; others reduce with a float64 floor)
__device__ __forceinline__ int wrapN(double b, int N) {
    // v_cvt_i32_f64 clamps out-of-range values to INT_MIN / INT_MAX and turns NaN into 0, so one
    // integer test takes every cell inside the grid (and NaN to cell 0, as below)
    int i;
    asm("v_cvt_i32_f64 %0, %1" : "=v"(i) : "v"(b));
    if ((unsigned)i < (unsigned)N) return i;
    const double n = (double)N;
    if (b < 0.0 && b >= -n) return (int)(b + n);
    if (b >= n && b < 2.0 * n) return (int)(b - n);
    int r = (int)(b - n * floor(b / n));
    if (r >= N) r -= N;
    if (r < 0) r += N;
    return (unsigned)r < (unsigned)N ? r : 0;   // non-finite input: stay inside the grid
}

// ceil(2^32 nt / N): c * tile_mul(N, nt) >> 32 = floor(c nt / N) for 0 <= c < N + 4 and N < 65536 (the
// rounding of the factor adds less than (N + 4) / 2^32 < 1 / N, the smallest distance below an integer)
inline unsigned tile_mul(int N, int nt) { return (unsigned)((((unsigned long long)nt << 32) + N - 1) / N); }

// exclusive sums of one value a thread over the workgroup (wsum: a word of LDS per wave; synchronises once)
__device__ __forceinline__ unsigned block_exscan(unsigned x, unsigned* wsum) {
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    unsigned v = x;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const unsigned u = __shfl_up(v, o, 64);
        if (lane >= o) v += u;
    }
    if (lane == 63) wsum[wv] = v;
    __syncthreads();
    unsigned run = v - x;
    for (int j = 0; j < wv; ++j) run += wsum[j];
    return run;
}

}  // namespace pyl
