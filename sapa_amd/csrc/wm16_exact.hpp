// The slow way of the dense-window kernels, for tiles that hold non-finite values.
//
// A dense product multiplies what lies outside a child's window by a weight of zero, and 0 * inf is NaN:
// one non-finite value would reach every child (cell) of the blocks whose windows hold it and, through
// pieces that run over a row's end, the other edge of the image.  Such a result is never finite, so the
// kernels look at their results (NonFinite), and a workgroup that has a non-finite one forms the results of that block again here, term by term over the cells (children) that the operator
// names: finite where they are finite, and infinite or NaN where the operator's are.
//
// Nothing here is fast: a block is 64 children (16 cells) whose terms all threads of a workgroup share,
// from global memory, with the weights in LDS.
#pragma once
#include "wm16_common.hpp"

namespace sapa {

namespace wm {

// whether a result among those shown to it is infinite or NaN: their largest magnitude (half an
// instruction per value)
struct NonFinite {
    float m = 0.f;
    __device__ __forceinline__ void see(f32x4 x) {
        m = __builtin_elementwise_maximum(__builtin_elementwise_maximum(m, __builtin_fabsf(x[0])), __builtin_fabsf(x[1]));
        m = __builtin_elementwise_maximum(__builtin_elementwise_maximum(m, __builtin_fabsf(x[2])), __builtin_fabsf(x[3]));
    }
    __device__ __forceinline__ bool any() const { return !(m < __builtin_inff()); }
};

// every wave's result stores and LDS accesses are done with (the results below overwrite some of the former)
__device__ __forceinline__ void settled() {
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
#endif
}

// one image of a tensor: channel c of pixel i at p[c * cs + i * ps]
template <typename T> struct Plane {
    T *p;
    long cs, ps;
    __device__ __forceinline__ float operator()(int c, long i) const { return (float)p[c * cs + i * ps]; }
    __device__ __forceinline__ void set(int c, long i, float v) const { p[c * cs + i * ps] = (T)v; }
};
template <bool CL, typename T>
__device__ __forceinline__ Plane<T> plane_of(T *t, long n, int channels, long pixels) {
    return Plane<T>{t + n * channels * pixels, CL ? 1 : pixels, CL ? channels : 1};
}

template <typename T>
__device__ __forceinline__ float dot(const Plane<const T> &a, long i, const Plane<const T> &b, long j, int channels) {
    float s = 0.f;
    for (int c = 0; c < channels; ++c) s = __builtin_fmaf(a(c, i), b(c, j), s);
    return s;
}

// The 8 x 8 children from child (cy0, cx0) on: outputs c_lo .. c_hi - 1.  lds: 64 K * K floats.
template <typename T, int K, int S, int NT>
__device__ __forceinline__ void exact_children(float *lds, Plane<const T> q, Plane<const T> key, Plane<const T> value,
                                               Plane<T> out, int d, int c_lo, int c_hi, int H, int W, int cy0, int cx0) {
    constexpr int KK = K * K, R = (K - 1) / 2;
    const int tid = threadIdx.x, child = tid % 64;
    const int cy = cy0 + child / 8, cx = cx0 + child % 8, y0 = cy / S - R, x0 = cx / S - R;
    const long at = (long)cy * S * W + cx;
    const bool in = cy < S * H && cx < S * W;
    auto cell = [&](int k) { return (u32)(y0 + k / K) < (u32)H && (u32)(x0 + k % K) < (u32)W ? (long)(y0 + k / K) * W + x0 + k % K : -1L; };
    if (in)
        for (int k = tid / 64; k < KK; k += NT / 64) {
            const long i = cell(k);
            lds[k * 64 + child] = i < 0 ? 0.f : dot<T>(q, at, key, i, d);
        }
    __syncthreads();
    if (in && tid < 64) {
        float m = -__builtin_inff(), sum = 0.f;
        for (int k = 0; k < KK; ++k) m = fmaxf(m, lds[k * 64 + child]);
        for (int k = 0; k < KK; ++k) {
            const float e = __builtin_amdgcn_exp2f(__builtin_fmaf(lds[k * 64 + child], LOG2E, -m * LOG2E));
            lds[k * 64 + child] = e;
            sum += e;
        }
        const float inv = 1.f / sum;
        for (int k = 0; k < KK; ++k) lds[k * 64 + child] *= inv;
    }
    __syncthreads();
    if (in)
        for (int c = c_lo + tid / 64; c < c_hi; c += NT / 64) {
            float s = 0.f;
            for (int k = 0; k < KK; ++k) {
                const long i = cell(k);
                if (i >= 0) s = __builtin_fmaf(lds[k * 64 + child], value(c, i), s);
            }
            out.set(c, at, s);
        }
    __syncthreads();
}

}  // namespace wm

}  // namespace sapa
