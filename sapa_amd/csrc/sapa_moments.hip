// Per (image, channel) mean and biased variance of a feature map in one pass
// over it: the statistics that GroupNorm needs (sapa_base.py:17-19,27-31 feed
// norm_y(y) and norm_x(x) to the q / k projections), from which the host folds
// the normalisation into the projection weights.  HBM-bound: every element is
// read once, 16 bytes per lane.
//
// Two kernels, no atomics (results do not depend on scheduling):
//   1. partial sums of (x - shift) and (x - shift)^2 in fp32 over a chunk of an
//      image's pixels, shift = the channel's first element (keeps the squares
//      small when |mean| >> spread);
//        contiguous [B, C, HW]:     one block per (image, channel, chunk), the
//                                   lanes along the pixels;
//        channels-last [B, HW, C]:  one block per (image, chunk), a lane owns 4
//                                   channels and every 256 / (C / 4)-th pixel,
//                                   the pixel lanes are summed through LDS;
//   2. one thread per (image, channel) adds the chunks in order and writes
//      mean = shift + S1 / HW, var = S2 / HW - (S1 / HW)^2.
#include "kernels.hpp"

#include <mutex>

namespace sapa {

namespace moments {

typedef unsigned u32;
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef u32 u32x2 __attribute__((ext_vector_type(2)));
typedef u32 u32x4 __attribute__((ext_vector_type(4)));

// N consecutive elements -> floats
template <typename T, int N> struct Pack;
template <> struct Pack<float, 4> {
    static __device__ __forceinline__ void load(const float *p, float (&v)[4]) {
        const f32x4 r = __builtin_nontemporal_load((const f32x4 *)p);
        v[0] = r[0], v[1] = r[1], v[2] = r[2], v[3] = r[3];
    }
};
template <typename H> struct Pack<H, 8> {
    static __device__ __forceinline__ void load(const H *p, float (&v)[8]) {
        union { u32x4 u; H h[8]; } x;
        x.u = __builtin_nontemporal_load((const u32x4 *)p);
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = (float)x.h[i];
    }
};
template <typename H> struct Pack<H, 4> {
    static __device__ __forceinline__ void load(const H *p, float (&v)[4]) {
        union { u32x2 u; H h[4]; } x;
        x.u = __builtin_nontemporal_load((const u32x2 *)p);
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = (float)x.h[i];
    }
};

// sum over the 256 threads of a block; the result is valid in thread 0
__device__ __forceinline__ void block_sum2(float &a, float &b, float (*red)[2]) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        a += __shfl_xor(a, o);
        b += __shfl_xor(b, o);
    }
    const int wave = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) red[wave][0] = a, red[wave][1] = b;
    __syncthreads();
    if (threadIdx.x == 0) {
        a = red[0][0] + red[1][0] + red[2][0] + red[3][0];
        b = red[0][1] + red[1][1] + red[2][1] + red[3][1];
    }
}

// One feature of a launch; a launch takes one or two (of the same B and C: a module's query and key
// features; chunks = 0: none), the second's `rows` x chunks workgroups behind all of the first's.  (With the
// chunks of both beside each other in every row the chip reads two tensors in turn: fp32, B=16, C=256,
// 100x167 -> 200x334, 253 us against 208 for two launches.)
template <typename T> struct Feature {
    const T *x;
    float *part;
    long HW, seg;
    int chunks;
};
template <typename F>
__device__ __forceinline__ F feature_of(const F &f0, const F &f1, int rows, int &row, int &chunk) {
    const unsigned first = (unsigned)rows * (unsigned)f0.chunks;
    const bool second = blockIdx.x >= first;
    const F f = second ? f1 : f0;
    const unsigned id = blockIdx.x - (second ? first : 0u);
    row = (int)(id / (unsigned)f.chunks);
    chunk = (int)(id % (unsigned)f.chunks);
    return f;
}

// contiguous layout: row = image * C + channel; VEC elements per load
// (1: any alignment)
template <typename T, int VEC>
__global__ void __launch_bounds__(256)
partial_nchw_kernel(Feature<T> f0, Feature<T> f1, int rows) {
    __shared__ float red[4][2];
    int row, chunk;
    const Feature<T> f = feature_of(f0, f1, rows, row, chunk);
    const long bc = row;
    const long HW = f.HW, seg = f.seg;
    const int chunks = f.chunks;
    float *const part = f.part;
    const T *xc = f.x + bc * HW;
    const float shift = (float)xc[0];
    const long lo = chunk * seg, hi = lo + seg < HW ? lo + seg : HW;
    float s1 = 0.f, s2 = 0.f;
    if constexpr (VEC == 1) {
        for (long i = lo + threadIdx.x; i < hi; i += 256) {
            const float v = (float)xc[i] - shift;
            s1 += v;
            s2 = fma_(v, v, s2);
        }
    } else {
        for (long i = lo + (long)threadIdx.x * VEC; i < hi; i += 256 * VEC) {
            float v[VEC];
            Pack<T, VEC>::load(xc + i, v);
#pragma unroll
            for (int e = 0; e < VEC; ++e) {
                const float t = v[e] - shift;
                s1 += t;
                s2 = fma_(t, t, s2);
            }
        }
    }
    block_sum2(s1, s2, red);
    if (threadIdx.x == 0) {
        part[(bc * chunks + chunk) * 2] = s1;
        part[(bc * chunks + chunk) * 2 + 1] = s2;
    }
}

#ifndef SAPA_MOMENTS_UNROLL
#define SAPA_MOMENTS_UNROLL 8
#endif
// channels-last layout: row = image; thread = (pixel lane, group of
// CPT channels); SAPA_MOMENTS_UNROLL pixels per thread are in flight at a time
template <typename T, int CPT>
__global__ void __launch_bounds__(256)
partial_nhwc_kernel(Feature<T> f0, Feature<T> f1, int rows, int C) {
    __shared__ float red[256][2 * CPT];
    int b, chunk;
    const Feature<T> f = feature_of(f0, f1, rows, b, chunk);
    const long HW = f.HW, seg = f.seg;
    const int chunks = f.chunks;
    const T *const x = f.x;
    float *const part = f.part;
    const int nq = C / CPT, npl = 256 / nq;            // channel groups, pixel lanes
    const int quad = threadIdx.x % nq, pl = threadIdx.x / nq;
    const T *xb = x + (long)b * HW * C + CPT * quad;
    float shift[CPT], s1[CPT], s2[CPT];
    Pack<T, CPT>::load(xb, shift);
#pragma unroll
    for (int e = 0; e < CPT; ++e) s1[e] = 0.f, s2[e] = 0.f;
    const long lo = chunk * seg, hi = lo + seg < HW ? lo + seg : HW;
    if (pl < npl) {
        long p = lo + pl;
        constexpr int U = SAPA_MOMENTS_UNROLL;
        for (; p + (U - 1) * npl < hi; p += U * npl) {
            float v[U][CPT];
#pragma unroll
            for (int u = 0; u < U; ++u) Pack<T, CPT>::load(xb + (p + u * npl) * C, v[u]);
#pragma unroll
            for (int u = 0; u < U; ++u)
#pragma unroll
                for (int e = 0; e < CPT; ++e) {
                    const float t = v[u][e] - shift[e];
                    s1[e] += t;
                    s2[e] = fma_(t, t, s2[e]);
                }
        }
        for (; p < hi; p += npl) {
            float v[CPT];
            Pack<T, CPT>::load(xb + p * C, v);
#pragma unroll
            for (int e = 0; e < CPT; ++e) {
                const float t = v[e] - shift[e];
                s1[e] += t;
                s2[e] = fma_(t, t, s2[e]);
            }
        }
    }
#pragma unroll
    for (int e = 0; e < CPT; ++e) red[threadIdx.x][e] = s1[e], red[threadIdx.x][CPT + e] = s2[e];
    __syncthreads();
    if (pl == 0) {
        float *out = part + (((long)b * chunks + chunk) * C + CPT * quad) * 2;
#pragma unroll
        for (int e = 0; e < CPT; ++e) {
            float a = 0.f, q = 0.f;
            for (int l = 0; l < npl; ++l) a += red[l * nq + quad][e], q += red[l * nq + quad][CPT + e];
            out[2 * e] = a;
            out[2 * e + 1] = q;
        }
    }
}

// thread = (image, channel): the chunks in order
template <typename T, bool CL>
__global__ void __launch_bounds__(256)
finish_kernel(const T *__restrict__ x, const float *__restrict__ part, float *__restrict__ mean_var,
              int B, int C, long HW, int chunks) {
    const long i = (long)blockIdx.x * 256 + threadIdx.x;
    if (i >= (long)B * C) return;
    const int b = (int)(i / C), c = (int)(i % C);
    float s1 = 0.f, s2 = 0.f;
    auto at = [&](int k) { return CL ? part + (((long)b * chunks + k) * C + c) * 2 : part + (i * chunks + k) * 2; };
    // (eight chunks' loads in flight at a time; the additions in the chunks' order)
    int k = 0;
    for (; k + 8 <= chunks; k += 8) {
        float a[8], q[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) a[u] = at(k + u)[0], q[u] = at(k + u)[1];
#pragma unroll
        for (int u = 0; u < 8; ++u) s1 += a[u], s2 += q[u];
    }
    for (; k < chunks; ++k) {
        s1 += at(k)[0];
        s2 += at(k)[1];
    }
    const float shift = (float)(CL ? x[(long)b * HW * C + c] : x[i * HW]);
    const float m = s1 / (float)HW;
    mean_var[2 * i] = shift + m;
    mean_var[2 * i + 1] = __builtin_fmaxf(s2 / (float)HW - m * m, 0.f);
}

// pixels per chunk and number of chunks: about `target` blocks in all, at least
// `min_px` pixels per chunk
static void chunking(long HW, long blocks_per_chunk_set, long target, long min_px, long &seg,
                     int &chunks) {
    long want = (target + blocks_per_chunk_set - 1) / blocks_per_chunk_set;
    long most = (HW + min_px - 1) / min_px;
    long n = want < most ? want : most;
    if (n < 1) n = 1;
    if (n > 4096) n = 4096;
    seg = (HW + n - 1) / n;
    seg = (seg + 7) / 8 * 8;                       // whole 16-byte loads in every chunk
    chunks = (int)((HW + seg - 1) / seg);
}
#ifndef SAPA_MOMENTS_CL_TUNE
#define SAPA_MOMENTS_CL_TUNE 2048, 1024
#endif
static void chunking_for(long HW, int B, int C, bool cl, long &seg, int &chunks) {
    if (cl) chunking(HW, B, SAPA_MOMENTS_CL_TUNE, seg, chunks);
    else chunking(HW, (long)B * C, 4096, 512, seg, chunks);
}

// the partial sums of one or two features (x1 null: one).  Two planar features of which one cannot be read in
// vectors take a launch each: the other one must not pay for it (fp32, a high-res feature beside a low-res
// one of 13 x 13 cells)
template <typename T>
static void launch_partial(const T *x0, float *ws0, long HW0, const T *x1, float *ws1, long HW1, int B, int C, bool cl,
                           hipStream_t st) {
    Feature<T> f0{x0, ws0, HW0, 0, 0}, f1{x1, ws1, HW1, 0, 0};
    chunking_for(HW0, B, C, cl, f0.seg, f0.chunks);
    if (x1) chunking_for(HW1, B, C, cl, f1.seg, f1.chunks);
    constexpr int VEC = 16 / (int)sizeof(T);
    if (x1 && !cl && (HW0 % VEC == 0) != (HW1 % VEC == 0)) {
        launch_partial<T>(x0, ws0, HW0, nullptr, nullptr, 0, B, C, cl, st);
        return launch_partial<T>(x1, ws1, HW1, nullptr, nullptr, 0, B, C, cl, st);
    }
    const int rows = cl ? B : B * C;
    const dim3 grid((unsigned)rows * (unsigned)(f0.chunks + f1.chunks));
    const bool aligned = ((uintptr_t)x0 | (uintptr_t)x1) % 16 == 0;
    if (cl) {
        // 16 bytes per lane where the channel count and the alignment allow it
        constexpr int WIDE = 16 / (int)sizeof(T);
        if (WIDE == 8 && C % 8 == 0 && aligned)
            hipLaunchKernelGGL((partial_nhwc_kernel<T, WIDE>), grid, dim3(256), 0, st, f0, f1, rows, C);
        else
            hipLaunchKernelGGL((partial_nhwc_kernel<T, 4>), grid, dim3(256), 0, st, f0, f1, rows, C);
    } else {
        if (HW0 % VEC == 0 && aligned)
            hipLaunchKernelGGL((partial_nchw_kernel<T, VEC>), grid, dim3(256), 0, st, f0, f1, rows);
        else
            hipLaunchKernelGGL((partial_nchw_kernel<T, 1>), grid, dim3(256), 0, st, f0, f1, rows);
    }
}

template <typename T>
static hipError_t launch_t(const T *x, float *ws, float *mean_var, int B, int C, long HW, bool cl,
                           hipStream_t st) {
    launch_partial<T>(x, ws, HW, nullptr, nullptr, 0, B, C, cl, st);
    long seg;
    int chunks;
    chunking_for(HW, B, C, cl, seg, chunks);
    auto kern = cl ? finish_kernel<T, true> : finish_kernel<T, false>;
    hipLaunchKernelGGL(kern, dim3(((long)B * C + 255) / 256), dim3(256), 0, st, x, ws, mean_var, B, C, HW, chunks);
    return hipGetLastError();
}

// GroupNorm folded into a 1x1 projection, per image: from the (image, channel)
// moments, gamma / beta and the projection's weight W [O, C] and bias,
//   rstd_g   = 1 / sqrt(var_g + eps),  group moments from the channel moments
//   W'[b,o,c] = W[o,c] * gamma[c] * rstd_g(c)
//   b'[b,o]   = bias[o] + sum_c W[o,c] * (beta[c] - mean_g(c) * gamma[c] * rstd_g(c))
// so that  conv(groupnorm(x))[b] = W'[b] x[b] + b'[b].  Block = (image, 4 output
// rows): scale and shift of every channel go through LDS (recomputed per block:
// a few hundred operations), then one wave per output row.
template <typename T>
__global__ void __launch_bounds__(256)
fold_kernel(const float *__restrict__ mean_var, const T *__restrict__ gamma,
            const T *__restrict__ beta, const T *__restrict__ w, const T *__restrict__ bias,
            T *__restrict__ w_out, T *__restrict__ b_out, int C, int O, int G, float eps) {
    extern __shared__ float sh[];                  // scale[C], shift[C]
    float *scale = sh, *shift = sh + C;
    const int b = blockIdx.x, per = C / G;
    const float *mv = mean_var + (long)b * C * 2;
    for (int g = threadIdx.x; g < G; g += 256) {
        float m = 0.f;
        for (int c = g * per; c < (g + 1) * per; ++c) m += mv[2 * c];
        m /= (float)per;
        float v = 0.f;
        for (int c = g * per; c < (g + 1) * per; ++c) {
            const float dm = mv[2 * c] - m;
            v += mv[2 * c + 1] + dm * dm;
        }
        const float rstd = 1.f / __builtin_sqrtf(v / (float)per + eps);
        for (int c = g * per; c < (g + 1) * per; ++c) {
            const float ga = gamma ? (float)gamma[c] : 1.f, be = beta ? (float)beta[c] : 0.f;
            scale[c] = ga * rstd;
            shift[c] = be - m * ga * rstd;
        }
    }
    __syncthreads();
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for (int o = blockIdx.y * 4 + wave; o < O; o += 4 * gridDim.y) {
        const T *wr = w + (long)o * C;
        T *wo = w_out + ((long)b * O + o) * C;
        float acc = 0.f;
        for (int c = lane; c < C; c += 64) {
            const float x = (float)wr[c];
            wo[c] = (T)(x * scale[c]);
            acc = fma_(x, shift[c], acc);
        }
#pragma unroll
        for (int d = 32; d > 0; d >>= 1) acc += __shfl_xor(acc, d);
        if (lane == 0) b_out[(long)b * O + o] = (T)(acc + (bias ? (float)bias[o] : 0.f));
    }
}

// finish_kernel and fold_kernel in one launch, for a caller that wants the weights only: every block
// adds up the partial sums of its image's channels again (from the cache: C * chunks * 8 bytes per
// `rows` output rows).  Bound by the latency of its loads: what depends on no other load is requested
// at once, and where an image has many chunks (`parts` > 1) several threads share a channel's, so
// that a thread waits for a few batches of 16 instead of for all of them in turn.  Per feature, 2.4 + 6.2
// us for the two kernels and 5 for this one at B=8, C=256, 16x16 in bf16, 6 + 8 and 10 at
// B=16, C=256, 200x336 in channels-last bf16 (128 chunks).
constexpr int kFoldChannels = 2048;                // 4 floats of LDS each
// One or two features and their projections per launch: the second's blocks of rows behind the
// first's `blocks0` along blockIdx.y.  (Two at once: the smaller feature's latencies lie beside the
// other's; module forward B=8, C=256, 16x16 in bf16 57 -> 47 us, B=16, 100x168 channels-last 492 -> 474.)
template <typename T> struct Fold {
    const T *x;
    const float *part;
    const T *gamma, *beta, *w, *bias;
    T *w_out, *b_out;
    long HW;
    int chunks, parts;
};
template <typename T, bool CL>
__global__ void __launch_bounds__(1024)
finish_fold_kernel(Fold<T> f0, Fold<T> f1, int blocks0, int C, int O, int G, float eps, int rows) {
    const bool second = (int)blockIdx.y >= blocks0;
    const Fold<T> f = second ? f1 : f0;
    const int block = (int)blockIdx.y - (second ? blocks0 : 0), chunks = f.chunks, parts = f.parts;
    const long HW = f.HW;
    const T *__restrict__ x = f.x, *__restrict__ gamma = f.gamma, *__restrict__ beta = f.beta, *__restrict__ w = f.w,
            *__restrict__ bias = f.bias;
    const float *__restrict__ part = f.part;
    T *__restrict__ w_out = f.w_out, *__restrict__ b_out = f.b_out;
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    extern __shared__ float sh[];                  // mean[C], var[C], scale[C], shift[C]; before: sums[parts][C][2]
    float *mean = sh, *var = sh + C, *scale = sh + 2 * C, *shift = sh + 3 * C;
    f32x2 *sums = (f32x2 *)(sh + 4 * C);
    const int nt = blockDim.x, nw = nt / 64, b = blockIdx.x, per = C / G;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int o0 = block * rows + wave, o1 = (block + 1) * rows < O ? (block + 1) * rows : O;
    float first[4];                                // the first 256 channels of the wave's first row
#pragma unroll
    for (int u = 0; u < 4; ++u) first[u] = o0 < o1 && lane + 64 * u < C ? (float)w[(long)o0 * C + lane + 64 * u] : 0.f;
    // sums of a channel's chunks k0 .. k1 - 1, in their order
    auto add_up = [&](int c, int k0, int k1) {
        const long i = (long)b * C + c;
        auto at = [&](int k) {
            return *(const f32x2 *)(CL ? part + (((long)b * chunks + k) * C + c) * 2 : part + (i * chunks + k) * 2);
        };
        f32x2 s = {0.f, 0.f};
        int k = k0;
        for (; k + 16 <= k1; k += 16) {
            f32x2 v[16];
#pragma unroll
            for (int u = 0; u < 16; ++u) v[u] = at(k + u);
#pragma unroll
            for (int u = 0; u < 16; ++u) s[0] += v[u][0], s[1] += v[u][1];
        }
        for (; k < k1; k += 4) {
            f32x2 v[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) v[u] = at(k + u < k1 ? k + u : k1 - 1);
#pragma unroll
            for (int u = 0; u < 4; ++u)
                if (k + u < k1) s[0] += v[u][0], s[1] += v[u][1];
        }
        return s;
    };
    if (parts > 1) {
        const int len = (chunks + parts - 1) / parts;
        for (int i = threadIdx.x; i < parts * C; i += nt) {
            const int k0 = i / C * len, k1 = k0 + len < chunks ? k0 + len : chunks;
            sums[i] = add_up(i % C, k0, k1);
        }
        __syncthreads();
    }
    for (int c = threadIdx.x; c < C; c += nt) {
        const float origin = (float)(CL ? x[(long)b * HW * C + c] : x[((long)b * C + c) * HW]);
        f32x2 s;
        if (parts > 1) {
            s = sums[c];
            for (int p = 1; p < parts; ++p) s[0] += sums[p * C + c][0], s[1] += sums[p * C + c][1];
        } else {
            s = add_up(c, 0, chunks);
        }
        const float m = s[0] / (float)HW;
        mean[c] = origin + m;
        var[c] = __builtin_fmaxf(s[1] / (float)HW - m * m, 0.f);
    }
    __syncthreads();
    // every channel's thread forms its group's moments
    for (int c = threadIdx.x; c < C; c += nt) {
        const float ga = gamma ? (float)gamma[c] : 1.f, be = beta ? (float)beta[c] : 0.f;
        const int g0 = c / per * per;
        float m = 0.f;
#pragma unroll 8
        for (int k = 0; k < per; ++k) m += mean[g0 + k];
        m /= (float)per;
        float v = 0.f;
#pragma unroll 8
        for (int k = 0; k < per; ++k) {
            const float dm = mean[g0 + k] - m;
            v += var[g0 + k] + dm * dm;
        }
        const float rstd = 1.f / __builtin_sqrtf(v / (float)per + eps);
        scale[c] = ga * rstd;
        shift[c] = be - m * ga * rstd;
    }
    __syncthreads();
    for (int o = o0; o < o1; o += nw) {
        const T *wr = w + (long)o * C;
        T *wo = w_out + ((long)b * O + o) * C;
        float acc = 0.f;
        for (int c = lane, u = 0; c < C; c += 64, ++u) {
            const float v = o == o0 && u < 4 ? (u == 0 ? first[0] : u == 1 ? first[1] : u == 2 ? first[2] : first[3]) : (float)wr[c];
            wo[c] = (T)(v * scale[c]);
            acc = fma_(v, shift[c], acc);
        }
#pragma unroll
        for (int d = 32; d > 0; d >>= 1) acc += __shfl_xor(acc, d);
        if (lane == 0) b_out[(long)b * O + o] = (T)(acc + (bias ? (float)bias[o] : 0.f));
    }
}

template <typename T>
static hipError_t norm_fold_t(const NormFold *f, int n, int B, int C, int O, int G, float eps, bool cl, hipStream_t st) {
    const bool two = n == 2;
    launch_partial<T>((const T *)f[0].x, (float *)f[0].workspace, f[0].HW, two ? (const T *)f[1].x : nullptr,
                      two ? (float *)f[1].workspace : nullptr, two ? f[1].HW : 0, B, C, cl, st);
    Fold<T> a[2] = {};
    bool many = false;
    for (int i = 0; i < n; ++i) {
        long seg;
        a[i] = Fold<T>{(const T *)f[i].x, (const float *)f[i].workspace, (const T *)f[i].gamma, (const T *)f[i].beta,
                       (const T *)f[i].w, (const T *)f[i].bias, (T *)f[i].w_out, (T *)f[i].b_out, f[i].HW, 0, 1};
        chunking_for(f[i].HW, B, C, cl, seg, a[i].chunks);
        many |= a[i].chunks > 16;
    }
    // few chunks: a thread per channel, a row per wave of 4; else up to 1024 threads that share a
    // channel's chunks in runs of 16 or more, and 16 rows for what they fetch
    const int nt = many ? 1024 : 256, rows = many ? 16 : 4, blocks = (O + rows - 1) / rows;
    int parts = 1;
    for (int i = 0; i < n; ++i) {
        if (many && C < nt) a[i].parts = nt / C;
        if (a[i].parts > a[i].chunks / 16) a[i].parts = a[i].chunks / 16 < 1 ? 1 : a[i].chunks / 16;
        if (a[i].parts > parts) parts = a[i].parts;
    }
    const size_t lds = (size_t)(4 * C + (parts > 1 ? 2 * parts * C : 0)) * sizeof(float);
    auto kern = cl ? finish_fold_kernel<T, true> : finish_fold_kernel<T, false>;
    hipLaunchKernelGGL(kern, dim3(B, n * blocks), dim3(nt), lds, st, a[0], a[1], blocks, C, O, G, eps, rows);
    return hipGetLastError();
}

template <typename T>
static hipError_t fold_t(const float *mean_var, const void *gamma, const void *beta, const void *w,
                         const void *bias, void *w_out, void *b_out, int B, int C, int O, int G,
                         float eps, hipStream_t st) {
    hipLaunchKernelGGL((fold_kernel<T>), dim3(B, (O + 3) / 4), dim3(256), 2 * C * sizeof(float), st, mean_var,
                       (const T *)gamma, (const T *)beta, (const T *)w, (const T *)bias, (T *)w_out,
                       (T *)b_out, C, O, G, eps);
    return hipGetLastError();
}

}  // namespace moments

// bytes of workspace channel_moments_launch needs for these extents
long channel_moments_workspace(int B, int C, long HW, bool channels_last) {
    long seg;
    int chunks;
    moments::chunking_for(HW, B, C, channels_last, seg, chunks);
    return (long)B * C * chunks * 2 * (long)sizeof(float);
}

static bool channel_moments_served(const void *x, int B, int C, bool channels_last, int dtype) {
    if (!channels_last) return (long)B * C <= 65535;
    const int esize = dtype == 0 ? 4 : 2;
    return C % 4 == 0 && C <= 1024 && (uintptr_t)x % (4 * esize) == 0 && B <= 65535;
}

// x: [B, C, HW] contiguous or [B, HW, C] (channels_last), f32 / f16 / bf16;
// mean_var: [B, C, 2] fp32.  Channels-last needs C % 4 == 0, C <= 1024 and x
// aligned to 4 elements; the contiguous layout B * C <= 65535.
// hipErrorNotSupported otherwise.
hipError_t channel_moments_launch(const void *x, void *workspace, float *mean_var, int B, int C,
                                  long HW, bool channels_last, int dtype, hipStream_t st) {
    if (!channel_moments_served(x, B, C, channels_last, dtype)) return hipErrorNotSupported;
    float *ws = (float *)workspace;
    switch (dtype) {
        case 0: return moments::launch_t((const float *)x, ws, mean_var, B, C, HW, channels_last, st);
        case 2: return moments::launch_t((const f16_t *)x, ws, mean_var, B, C, HW, channels_last, st);
        case 3: return moments::launch_t((const bf16_t *)x, ws, mean_var, B, C, HW, channels_last, st);
        default: return hipErrorNotSupported;
    }
}

// ---- the same statistics for callers that cannot bring a workspace ----
//
// The partial sums go to a fixed array in device memory that is part of the
// library's code object: no allocation on any path, so the call can be made
// under stream capture or from a loop that must not touch the allocator.
// Every device holds its own copy of the array at its own address; host code
// only ever uses the address hipGetSymbolAddress reports for the current
// device (the array's name is not a device address on the host side).
}  // namespace sapa

constexpr long kStaticScratchBytes = 8L << 20;
static __device__ __align__(256) unsigned char scratch[kStaticScratchBytes];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mutex;
void *g_scratch_ptr[kMaxDevices] = {};

// address of `scratch` on the current device; looked up once per device
hipError_t scratch_address(void **out) {
    int dev = -1;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    if (dev < 0 || dev >= kMaxDevices) return hipErrorInvalidDevice;
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (!g_scratch_ptr[dev]) {
        void *p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return e;
        if (!p) return hipErrorInvalidSymbol;
        g_scratch_ptr[dev] = p;
    }
    *out = g_scratch_ptr[dev];
    return hipSuccess;
}
}  // namespace

namespace sapa {

long channel_moments_static_capacity() { return kStaticScratchBytes; }

// channel_moments_launch with the partial sums in the library's own fixed
// array.  The caller has checked that channel_moments_workspace(...) fits
// channel_moments_static_capacity().  Every partial sum that the second kernel
// reads is written by the first one of the same call, so nothing has to be
// cleared between calls; two calls in flight on one device share the array and
// must not overlap.
hipError_t channel_moments_static_launch(const void *x, float *mean_var, int B, int C, long HW,
                                         bool channels_last, int dtype, hipStream_t st) {
    if (channel_moments_workspace(B, C, HW, channels_last) > kStaticScratchBytes)
        return hipErrorInvalidValue;
    void *ws = nullptr;
    const hipError_t e = scratch_address(&ws);
    if (e != hipSuccess) return e;
    return channel_moments_launch(x, ws, mean_var, B, C, HW, channels_last, dtype, st);
}

// mean_var [B, C, 2] fp32 (channel_moments_launch); gamma, beta [C] or null, w
// [O, C], bias [O] or null, all of type `dtype` (f32 / f16 / bf16); w_out
// [B, O, C] and b_out [B, O] of the same type.  C % G == 0, C <= 8192.
hipError_t groupnorm_fold_launch(const float *mean_var, const void *gamma, const void *beta,
                                 const void *w, const void *bias, void *w_out, void *b_out, int B,
                                 int C, int O, int G, float eps, int dtype, hipStream_t st) {
    if (G < 1 || C % G != 0 || C > 8192) return hipErrorNotSupported;
    switch (dtype) {
        case 0: return moments::fold_t<float>(mean_var, gamma, beta, w, bias, w_out, b_out, B, C, O, G, eps, st);
        case 2: return moments::fold_t<f16_t>(mean_var, gamma, beta, w, bias, w_out, b_out, B, C, O, G, eps, st);
        case 3: return moments::fold_t<bf16_t>(mean_var, gamma, beta, w, bias, w_out, b_out, B, C, O, G, eps, st);
        default: return hipErrorNotSupported;
    }
}

// Moments and folded projection weights of one feature, or of two with the same B, C, O, G and eps,
// in two launches; f[i].workspace: channel_moments_workspace bytes each.  What
// channel_moments_launch and groupnorm_fold_launch require holds for each; C <= 2048.
// hipErrorNotSupported otherwise, nothing launched.
bool norm_fold_supported(int B, int C, int G, bool channels_last, int dtype) {
    return (dtype == 0 || dtype == 2 || dtype == 3) && G >= 1 && C % G == 0 && C <= moments::kFoldChannels &&
           channel_moments_served(nullptr, B, C, channels_last, dtype);
}

hipError_t norm_fold_launch(const NormFold *f, int n, int B, int C, int O, int G, float eps, bool channels_last,
                            int dtype, hipStream_t st) {
    if (n < 1 || n > 2 || !norm_fold_supported(B, C, G, channels_last, dtype)) return hipErrorNotSupported;
    for (int i = 0; i < n; ++i)
        if (!channel_moments_served(f[i].x, B, C, channels_last, dtype)) return hipErrorNotSupported;
    switch (dtype) {
        case 0: return moments::norm_fold_t<float>(f, n, B, C, O, G, eps, channels_last, st);
        case 2: return moments::norm_fold_t<f16_t>(f, n, B, C, O, G, eps, channels_last, st);
        case 3: return moments::norm_fold_t<bf16_t>(f, n, B, C, O, G, eps, channels_last, st);
        default: return hipErrorNotSupported;
    }
}

}  // namespace sapa
