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

// whether a result among those shown to it is infinite or NaN: their largest magnitude.  (What is not finite
// and does not belong to a result meets a weight of zero there, and so for all children (cells) of a
// block at once: one of them is looked at per channel.)
struct NonFinite {
    float m = 0.f;
    __device__ __forceinline__ void see(f32x4 x) {
        m = __builtin_elementwise_maximum(__builtin_elementwise_maximum(m, __builtin_fabsf(x[0])), __builtin_fabsf(x[1]));
        m = __builtin_elementwise_maximum(__builtin_elementwise_maximum(m, __builtin_fabsf(x[2])), __builtin_fabsf(x[3]));
    }
    __device__ __forceinline__ void see(float x) { m = __builtin_elementwise_maximum(m, __builtin_fabsf(x)); }
    __device__ __forceinline__ bool any() const { return !(m < __builtin_inff()); }
};

// every wave's result stores and LDS accesses are done with (the results below overwrite some of the former)
__device__ __forceinline__ void settled() {
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
#endif
}

// What the slow way of a kernel needs to know of it: its only argument, a struct (again from memory), and its
// LDS.  The slow way of the backward kernels is a function of its own that is called with these and not
// inlined: as a part of the kernel it takes registers from the loops before it (both contiguous kernels
// at B=16, C=256, 100x168 in bf16: 718 us, 714 so).
struct Again {
    unsigned long long args;
    u32 lds, blocks, block;
    __device__ __forceinline__ Again(const u32 *l, u32 b) {
#if defined(__HIP_DEVICE_COMPILE__)
        args = (unsigned long long)__builtin_amdgcn_kernarg_segment_ptr();
        lds = lds_address((const __attribute__((address_space(3))) u32 *)l);
        blocks = b, block = blockIdx.x;
#endif
    }
    // in the function called: the same in every lane
    template <typename A> __device__ __forceinline__ A arguments() const {
        A a = {};
#if defined(__HIP_DEVICE_COMPILE__)
        const unsigned long long p = (unsigned long long)__builtin_amdgcn_readfirstlane((u32)(args >> 32)) << 32 |
                                     (u32)__builtin_amdgcn_readfirstlane((u32)args);
        __builtin_memcpy(&a, (const __attribute__((address_space(4))) A *)p, sizeof(A));
#endif
        return a;
    }
    __device__ __forceinline__ float *floats() const {
#if defined(__HIP_DEVICE_COMPILE__)
        return (float *)(__attribute__((address_space(3))) float *)(u32)__builtin_amdgcn_readfirstlane(lds);
#else
        return nullptr;
#endif
    }
    __device__ __forceinline__ u32 of_blocks() const { return __builtin_amdgcn_readfirstlane(blocks); }
    __device__ __forceinline__ u32 workgroup() const { return __builtin_amdgcn_readfirstlane(block); }
};

// one image of a tensor: channel c of pixel i at p[c * cs + i * ps]
template <typename T> struct Plane {
    T *p;
    long cs, ps;
    __device__ __forceinline__ float operator()(int c, long i) const { return (float)p[c * cs + i * ps]; }
    __device__ __forceinline__ void set(int c, long i, float v) const { p[c * cs + i * ps] = (T)v; }
};
template <bool CL, typename T>
__device__ __forceinline__ Plane<T> plane_of(T *t, long n, int channels, long pixels) {
    return Plane<T>{t ? t + n * channels * pixels : t, CL ? 1 : pixels, CL ? channels : 1};
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

// Backward: D (to stat_d) and the gradients of the queries (NULL: not wanted) of the 8 x 8 children from child
// (cy0, cx0) on, K = 5, s = 2.  lds: 128 * 25 floats.
template <typename T, int NT>
__device__ __forceinline__ void exact_grad_q(float *lds, Plane<const T> q, Plane<const T> key, Plane<const T> value,
                                             Plane<const T> grad_out, Plane<T> grad_q, float *stat_d, int d, int C,
                                             int H, int W, int cy0, int cx0) {
    const int tid = threadIdx.x, child = tid % 64;
    const int cy = cy0 + child / 8, cx = cx0 + child % 8, y0 = cy / 2 - 2, x0 = cx / 2 - 2;
    const long at = (long)cy * 2 * W + cx;
    const bool in = cy < 2 * H && cx < 2 * W;
    float *const a = lds, *const g = lds + 25 * 64;
    auto cell = [&](int k) { return (u32)(y0 + k / 5) < (u32)H && (u32)(x0 + k % 5) < (u32)W ? (long)(y0 + k / 5) * W + x0 + k % 5 : -1L; };
    if (in)
        for (int k = tid / 64; k < 25; k += NT / 64) {
            const long i = cell(k);
            a[k * 64 + child] = i < 0 ? 0.f : dot<T>(q, at, key, i, d);
            g[k * 64 + child] = i < 0 ? 0.f : dot<T>(grad_out, at, value, i, C);
        }
    __syncthreads();
    if (in && tid < 64) {
        float m = -__builtin_inff(), sum = 0.f, dsum = 0.f;
        for (int k = 0; k < 25; ++k) m = fmaxf(m, a[k * 64 + child]);
        for (int k = 0; k < 25; ++k) {
            const float e = __builtin_amdgcn_exp2f(__builtin_fmaf(a[k * 64 + child], LOG2E, -m * LOG2E));
            a[k * 64 + child] = e;
            sum += e;
        }
        const float inv = 1.f / sum;
        for (int k = 0; k < 25; ++k) dsum = __builtin_fmaf(a[k * 64 + child] *= inv, g[k * 64 + child], dsum);
        for (int k = 0; k < 25; ++k) a[k * 64 + child] *= g[k * 64 + child] - dsum;
        stat_d[at] = dsum;
    }
    __syncthreads();
    if (in && grad_q.p)
        for (int c = tid / 64; c < d; c += NT / 64) {
            float s = 0.f;
            for (int k = 0; k < 25; ++k) {
                const long i = cell(k);
                if (i >= 0) s = __builtin_fmaf(a[k * 64 + child], key(c, i), s);
            }
            grad_q.set(c, at, s);
        }
    __syncthreads();
}

// Backward: the gradients of the keys and values of the 4 x 4 cells from cell (cy0, cx0) on, which may lie
// outside the image (either tensor NULL: not wanted).  stats: the image's children's maximum (times log2 e),
// 1 / sum and D, `stride` floats apart.  lds: 200 * 16 floats.
template <typename T, int NT>
__device__ __forceinline__ void exact_grad_cells(float *lds, Plane<const T> q, Plane<const T> key, Plane<const T> value,
                                                 Plane<const T> grad_out, const float *stats, long stride, Plane<T> grad_key,
                                                 Plane<T> grad_value, int d, int C, int H, int W, int cy0, int cx0) {
    const int tid = threadIdx.x, cell = tid % 16;
    const int y = cy0 + cell / 4, x = cx0 + cell % 4;
    const long at = (long)y * W + x;
    const bool in = (u32)y < (u32)H && (u32)x < (u32)W;
    float *const a = lds, *const e = lds + 100 * 16;
    // child j = 0 .. 99 of the cell: parent (j / 4 / 5 - 2, j / 4 % 5 - 2) away
    auto child = [&](int j) {
        const int py = y + j / 20 - 2, px = x + j / 4 % 5 - 2;
        return (u32)py < (u32)H && (u32)px < (u32)W ? (long)(2 * py + (j >> 1 & 1)) * 2 * W + 2 * px + (j & 1) : -1L;
    };
    if (in)
        for (int j = tid / 16; j < 100; j += NT / 16) {
            const long i = child(j);
            if (i < 0) continue;
            const float w = __builtin_amdgcn_exp2f(__builtin_fmaf(dot<T>(q, i, key, at, d), LOG2E, -stats[i])) * stats[stride + i];
            a[j * 16 + cell] = w;
            if (grad_key.p) e[j * 16 + cell] = w * (dot<T>(grad_out, i, value, at, C) - stats[2 * stride + i]);
        }
    __syncthreads();
    auto gather = [&](const float *w, const Plane<const T> &hi, const Plane<T> &grad, int channels) {
        if (in && grad.p)
            for (int c = tid / 16; c < channels; c += NT / 16) {
                float s = 0.f;
                for (int j = 0; j < 100; ++j) {
                    const long i = child(j);
                    if (i >= 0) s = __builtin_fmaf(w[j * 16 + cell], hi(c, i), s);
                }
                grad.set(c, at, s);
            }
    };
    gather(a, grad_out, grad_value, C);
    gather(e, q, grad_key, d);
    __syncthreads();
}

}  // namespace wm

}  // namespace sapa
