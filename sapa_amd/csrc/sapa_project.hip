// 1x1 projection of a channels-last 16-bit feature map with per-image weights:
//   out[b, p, o] = sum_c x[b, p, c] * w[b, o, c] (+ bias[b, o]),   x [B, HW, C],
//   w [B, O, C], out [B, HW, O], fp16 / bf16, fp32 accumulation
// -- the q / k projections of the SAPA modules (sapa_base.py:32-35) after
// GroupNorm has been folded into per-image weights.  O is small (32 .. 128), so
// the operation is a stream over x: 2 C bytes read and 2 O written per pixel.
//
//   * a workgroup of 4 waves serves one image; its weights (O x C, up to 64 KB)
//     sit in LDS, rows padded by 16 bytes so that the matrix instruction's B
//     operand reads (16 rows x 4 column groups) fall on disjoint banks;
//   * a wave takes tiles of 16 consecutive pixels: 16 C-byte records, one
//     contiguous run of memory, fetched as 16 bytes per lane with the next
//     tile's loads in flight during the current tile's arithmetic, and passed
//     through a wave-private LDS tile (rows padded the same way) into the A
//     operand layout of v_mfma_f32_16x16x32 (row = pixel);
//   * the 16 x 16 results per output tile go back through LDS, so that a lane
//     stores 16 contiguous bytes and the wave one contiguous run of 32 O bytes.
//
// fp32 features (project32_kernel) take the same stream through the bf16 matrix
// instruction: every fp32 number is the exact sum of three bf16 numbers (8 + 8 + 8
// significant bits), a product of two bf16 numbers is exact in fp32, and of the nine
// piece products of x * w the six largest are kept (the other three are below 2^-23 of
// the product): six v_mfma_f32_16x16x32_bf16 per fp32 matrix step, fp32 sums -- an
// fp32 dot product to fp32 rounding at 32 / 6 times the rate of the fp32 matrix
// instruction, which leaves the kernel waiting for memory, not arithmetic.  The image's
// weights are taken apart once per workgroup into three bf16 planes in LDS; x goes
// from global memory straight into the A-operand registers (a lane reads two 16-byte
// pieces of its pixel's record per step of 32 channels) and is taken apart there.
//
// WIDE kernels: weights [OT][C] and bias [OT] shared by all images, any number OT of outputs (a
// multiple of 8) in blocks of O, one per blockIdx.z -- the plain 1x1 convolutions of SAPADeform
// (128 query and key channels, 72 .. 800 offset channels).  The feature is read once per block; the
// blocks of one pixel range run at the same time, so all but one of those reads come from a cache.
// (SAPA-D module, 256 channels: B=8, 64x64, 9 points, fp32 382 us with library convolutions and their
// bias passes, 298 with these; 25 points 638, 492; bf16 channels-last 361, 239.  What is left there in
// fp32 is the matrix work of the six piece products: 30 us per 8.6 GFLOP at the rate of a large product.)
#include "kernels.hpp"
#include "project_plan.hpp"

namespace sapa {

namespace project {

// where a workgroup's block of outputs lies: OT outputs in all (the stride of a channels-last
// record), o0 the first of this block, `left` its number
struct Span {
    int OT, o0, left;
};
template <int O, bool WIDE>
__device__ __forceinline__ Span span_of(int outputs) {
    if (!WIDE) return Span{O, 0, O};
    const int o0 = blockIdx.z * O;
    return Span{outputs, o0, outputs - o0 < O ? outputs - o0 : O};
}

// A launch serves one feature, or two of the same B, C and O (a module's query and key features; blocks = 0: none), the
// second's workgroups of an image behind the first's.  (Two that together do not fill the chip, see project_launch.)
template <typename T> struct Feature {
    const T *x, *w, *bias;
    T *out;
    long HW;
    int tiles, blocks;                            // tiles per wave, workgroups per image
};

typedef unsigned u32;
typedef u32 u32x2 __attribute__((ext_vector_type(2)));
typedef u32 u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// The result stores of the buffer kernels below carry their whole offset in the vector operand:
// with a scalar offset register the compiler leaves no wait state between a 16-byte buffer store
// and an instruction that overwrites its data registers, and the first dword of a piece was then
// now and then stored with the overwriting value (once a second workgroup on the CU kept the store
// waiting: 16-bit planes, 16 images of 200 x 336 pixels, 5000 of 69 M results).

template <typename T> struct Mma32;
template <> struct Mma32<f16_t> {
    static __device__ __forceinline__ f32x4 run(u32x4 a, u32x4 b, f32x4 c) {
        typedef _Float16 v8 __attribute__((ext_vector_type(8)));
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(v8, a), __builtin_bit_cast(v8, b), c, 0, 0, 0);
    }
};
template <> struct Mma32<bf16_t> {
    static __device__ __forceinline__ f32x4 run(u32x4 a, u32x4 b, f32x4 c) {
        typedef __bf16 v8 __attribute__((ext_vector_type(8)));
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8, a), __builtin_bit_cast(v8, b), c, 0, 0, 0);
    }
};

template <typename T>
__device__ __forceinline__ u32 pack2(float a, float b) {
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    typedef T tx2 __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(u32, __builtin_convertvector(f32x2{a, b}, tx2));
}

// C input channels, O outputs (both multiples of 16); tiles of 16 pixels
template <typename T, int C, int O, bool WIDE>
__global__ void __launch_bounds__(256)
project_kernel(Feature<T> f0, Feature<T> f1, int outputs) {
    const bool second = (int)blockIdx.x >= f0.blocks;
    const Feature<T> f = second ? f1 : f0;
    const long block = (int)blockIdx.x - (second ? f0.blocks : 0);
    const int b = blockIdx.y;
    const T *__restrict__ const x = f.x, *__restrict__ const w = f.w, *__restrict__ const bias = f.bias;
    T *__restrict__ const out = f.out;
    const long HW = f.HW;
    const int tiles_per_wave = f.tiles;
    constexpr int RW = C / 2 + 4;                 // dwords per padded row of C 16-bit values
    constexpr int NL = C / 32;                    // 16-byte loads per lane and tile (16 rows of 2 C bytes)
    constexpr int NT = O / 16;                    // output tiles of 16 columns
    constexpr int OW = O / 2 + 4;                 // dwords per padded row of the result tile
    constexpr int XT = 16 * RW > 16 * OW ? 16 * RW : 16 * OW;   // dwords of a wave's tile (x, then results)
    extern __shared__ __attribute__((aligned(16))) u32 sh[];
    u32 *wl = sh;                                 // weights: O rows of RW dwords
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    u32 *xt = sh + O * RW + wave * XT;            // this wave's tile
    const T *xb = x + (long)b * HW * C;
    const Span sp = span_of<O, WIDE>(outputs);
    T *ob = out + (long)b * HW * sp.OT;

    // the image's weights -> LDS (16 bytes per thread and step)
    {
        const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc(
            (void *)(w + (WIDE ? (long)sp.o0 : (long)b * O) * C), 0, sp.left * C * 2, 0x00020000);
        static_assert(O * C / 8 % 256 == 0, "whole steps");
#pragma unroll
        for (int k = 0; k < O * C / 8 / 256; ++k) {
            const int i = k * 256 + threadIdx.x, row = i / (C / 8), col = i % (C / 8);
            *(u32x4 *)(wl + row * RW + 4 * col) = __builtin_amdgcn_raw_buffer_load_b128(rw, (u32)i * 16u, 0, 0);
        }
    }
    __syncthreads();

    const long ntiles = (HW + 15) / 16;
    const long t0 = (block * 4 + wave) * tiles_per_wave;
    const long t1 = t0 + tiles_per_wave < ntiles ? t0 + tiles_per_wave : ntiles;
    const int r16 = lane & 15, kg = lane >> 4;    // row / column of a 16 x 16 tile, k group
    float bv[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
        bv[nt] = bias && 16 * nt + r16 < sp.left ? (float)bias[(WIDE ? (long)sp.o0 : (long)b * O) + 16 * nt + r16] : 0.f;

    // a tile's 16 records are one run of 32 C bytes: lane l takes 16-byte piece
    // j * 64 + l (pieces past the image: zeros)
    u32x4 st[NL];
    auto load_tile = [&](long t) __attribute__((always_inline)) {
        const long base = t * 16 * (C / 8), limit = HW * (C / 8);   // in 16-byte pieces
        const u32x4 *src = (const u32x4 *)xb;
#pragma unroll
        for (int j = 0; j < NL; ++j) {
            const long i = base + j * 64 + lane;
            st[j] = u32x4{0u, 0u, 0u, 0u};
            if (i < limit) st[j] = __builtin_nontemporal_load(src + i);
        }
    };
    if (t0 < t1) load_tile(t0);
    for (long t = t0; t < t1; ++t) {
        // registers -> the wave's LDS tile (row = pixel)
#pragma unroll
        for (int j = 0; j < NL; ++j) {
            const int i = j * 64 + lane, row = i / (C / 8), col = i % (C / 8);
            *(u32x4 *)(xt + row * RW + 4 * col) = st[j];
        }
        if (t + 1 < t1) load_tile(t + 1);
        f32x4 acc[NT];
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) acc[nt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < C / 32; ++ks) {
            // A: pixel r16, channels 32 ks + 8 kg .. +7; B: output 16 nt + r16, same channels.  (16-byte
            // reads: the 16 rows of a lane group lie on different bank quads, which they do not with 8
            // bytes and v_mfma_f32_16x16x16: 16 images of 200 x 336 and 100 x 168 pixels, 256 -> 64, 187 -> 176 us)
            const u32x4 a = *(const u32x4 *)(xt + r16 * RW + 16 * ks + 4 * kg);
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) {
                if (WIDE && 16 * nt >= sp.left) break;
                const u32x4 bm = *(const u32x4 *)(wl + (16 * nt + r16) * RW + 16 * ks + 4 * kg);
                acc[nt] = Mma32<T>::run(a, bm, acc[nt]);
            }
        }
        // acc[nt][i]: pixel 4 kg + i, output 16 nt + r16 -> the tile again, as 16-bit
        // rows of O values (the x tile has been consumed by this wave's own reads)
        unsigned short *rt = (unsigned short *)xt;
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const u32 h = pack2<T>(acc[nt][i] + bv[nt], 0.f);
                rt[(4 * kg + i) * (2 * OW) + 16 * nt + r16] = (unsigned short)h;
            }
        if (WIDE) {
            // 16 pieces of 2 O bytes, one per pixel's record
#pragma unroll
            for (int j = 0; j < (16 * O / 8 + 63) / 64; ++j) {
                const int i = j * 64 + lane, row = i / (O / 8), col = i % (O / 8);
                if (i < 16 * O / 8 && 8 * col < sp.left && t * 16 + row < HW)
                    __builtin_nontemporal_store(*(const u32x4 *)(xt + row * OW + 4 * col),
                                                (u32x4 *)(ob + (t * 16 + row) * sp.OT + sp.o0 + 8 * col));
            }
            continue;
        }
        // 16 rows of 2 O bytes -> one contiguous run of 32 O bytes
        const long obase = t * 16 * (O / 8), olimit = HW * (O / 8);
#pragma unroll
        for (int j = 0; j < (16 * O / 8 + 63) / 64; ++j) {
            const int i = j * 64 + lane, row = i / (O / 8), col = i % (O / 8);
            if (i < 16 * O / 8 && obase + i < olimit)
                __builtin_nontemporal_store(*(const u32x4 *)(xt + row * OW + 4 * col),
                                            (u32x4 *)ob + obase + i);
        }
    }
}

// n features in tiles of `pixels`: false where there are too many workgroups
template <typename T>
static bool spread16(const ProjectFeature *p, int n, Feature<T> (&f)[2], int B, int pixels, int blocks_o, int resident) {
    long tiles[2] = {0, 0};
    for (int i = 0; i < n; ++i) tiles[i] = (p[i].HW + pixels - 1) / pixels;
    const Spread s = plan16(tiles, (long)B * blocks_o, resident);
    for (int i = 0; i < n; ++i)
        f[i] = Feature<T>{(const T *)p[i].x, (const T *)p[i].w, (const T *)p[i].bias, (T *)p[i].out, p[i].HW, (int)s.per, (int)s.blocks[i]};
    return s.blocks[0] <= 65535 * 32L && s.blocks[1] <= 65535 * 32L && B <= 65535 && blocks_o <= 65535;
}

template <typename T, int C, int O, bool WIDE = false>
static hipError_t launch_co(const ProjectFeature *p, int n, int B, hipStream_t st, int outputs = O) {
    constexpr int RW = C / 2 + 4, OW = O / 2 + 4;
    constexpr int XT = 16 * RW > 16 * OW ? 16 * RW : 16 * OW;
    constexpr size_t lds = (size_t)(O * RW + 4 * XT) * 4;
    static_assert(lds <= 160 * 1024, "weights and tiles must fit LDS");
    const int blocks_o = (outputs + O - 1) / O;
    // two workgroups are resident per CU (LDS) and the part has 256 CUs: one round of at most 512
    // workgroups (16 images of 100 x 168 pixels, 256 -> 64: 37 us against
    // 46 with a fixed 8 tiles per wave; 200 x 336 pixels: 141 against 146)
    Feature<T> f[2] = {};
    if (!spread16(p, n, f, B, 16, blocks_o, lds > 80 * 1024 ? 1 : 2)) return hipErrorNotSupported;
    auto kern = project_kernel<T, C, O, WIDE>;
    if (lds > 64 * 1024) {
        // more than the default 64 KB per workgroup: ask for it; a device that
        // cannot give it is not served by this kernel
        int dev = 0, most = 0;
        if (hipGetDevice(&dev) != hipSuccess ||
            hipDeviceGetAttribute(&most, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) != hipSuccess ||
            (size_t)most < lds ||
            hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize,
                                (int)lds) != hipSuccess) {
            (void)hipGetLastError();
            return hipErrorNotSupported;
        }
    }
    hipLaunchKernelGGL(kern, dim3((unsigned)(f[0].blocks + f[1].blocks), B, blocks_o), dim3(256), lds, st, f[0], f[1],
                       outputs);
    return hipGetLastError();
}

// ---- 16-bit, contiguous feature (planes) ----
// x [B, C, HW]: a lane fetches 8 neighbouring pixels of one channel (a wave: 8 channels x 128
// bytes per load); a reduction step's 32 channels x 64 pixels pass through a wave-private LDS
// tile [channel][pixel] from which ds_read_tr16_b64 hands every lane its pixel's 4 channels (rows
// of 160 bytes: the four rows of a transposing read lie on disjoint banks).  Same order of the
// channels inside a step as in the fp32 kernel below; weights [O][C] in that order in LDS.
// Tiles of 64 pixels (four blocks of 16 matrix rows).  OUT_CL: out [B, HW, O], else [B, O, HW].
// HW a multiple of 8 (16-byte pieces never run from one plane into the next).
template <typename T, int C, int O, bool OUT_CL, bool WIDE>
__global__ void __launch_bounds__(256)
project16p_kernel(Feature<T> f0, Feature<T> f1, int outputs) {
    const bool second = (int)blockIdx.x >= f0.blocks;
    const Feature<T> f = second ? f1 : f0;
    const long block = (int)blockIdx.x - (second ? f0.blocks : 0);
    const int b = blockIdx.y;
    const T *__restrict__ const x = f.x, *__restrict__ const w = f.w, *__restrict__ const bias = f.bias;
    T *__restrict__ const out = f.out;
    const long HW = f.HW;
    const int tiles_per_wave = f.tiles;
    typedef short s16x4 __attribute__((ext_vector_type(4)));
    constexpr int NW = 4;
    constexpr int RW = C / 2 + 4;                 // dwords per padded row of C 16-bit values
    constexpr int NT = O / 16;                    // output tiles of 16 columns
    constexpr int OW = O / 2 + 4;                 // dwords per padded row of the result tile (channels-last)
    constexpr int PW = 64 / 2 + 4;                // ... of a block of 16 outputs x 64 pixels (planes)
    constexpr int XS = 64 / 2 + 8;                // dwords per row of the x tile: 160 bytes
    constexpr int KS = C / 32;                    // reduction steps
    constexpr int RING = KS < 4 ? KS : 4;         // steps of x in flight
    constexpr int RT = OUT_CL ? 16 * OW : 16 * PW;
    constexpr int WF = RT > 32 * XS ? RT : 32 * XS;
    static_assert(KS % RING == 0, "the ring of x registers is indexed by the step");
    extern __shared__ __attribute__((aligned(16))) u32 sh[];
    u32 *wl = sh;                                 // weights: O rows of RW dwords
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    u32 *xt = sh + O * RW + wave * WF;            // this wave's x tile / result tile
    const Span sp = span_of<O, WIDE>(outputs);
    // the image's weights -> LDS, 8 channels per thread and step: two groups of 4, which lie 8
    // places apart in the step's order
    {
        const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc(
            (void *)(w + (WIDE ? (long)sp.o0 : (long)b * O) * C), 0, sp.left * C * 2, 0x00020000);
        static_assert(O * C / 8 % (64 * NW) == 0, "whole steps");
#pragma unroll
        for (int k = 0; k < O * C / 8 / (64 * NW); ++k) {
            const int i = k * 64 * NW + threadIdx.x, o = i / (C / 8), c = 8 * (i % (C / 8)), cs = c % 32;
            const int pos = 32 * (c / 32) + 8 * ((cs % 16) / 4) + 4 * (cs / 16);
            const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(rw, (u32)i * 16u, 0, 0);
            u32 *dst = wl + o * RW + pos / 2;
            *(u32x2 *)dst = u32x2{v[0], v[1]};
            *(u32x2 *)(dst + 4) = u32x2{v[2], v[3]};
        }
    }
    __syncthreads();

    const long ntiles = (HW + 63) / 64;
    const long t0 = (block * NW + wave) * tiles_per_wave;
    const long t1 = t0 + tiles_per_wave < ntiles ? t0 + tiles_per_wave : ntiles;
    if (t0 >= t1) return;
    const int r16 = lane & 15, kg = lane >> 4;
    float bv[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
        bv[nt] = bias && 16 * nt + r16 < sp.left ? (float)bias[(WIDE ? (long)sp.o0 : (long)b * O) + 16 * nt + r16] : 0.f;

    const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(
        (void *)(x + (long)b * HW * C), 0, (int)(HW * C * 2), 0x00020000);
    // (planes: from the block's first plane to the end of its last, so that the rest is dropped)
    const __amdgpu_buffer_rsrc_t ro = __builtin_amdgcn_make_buffer_rsrc(
        (void *)(out + ((long)b * sp.OT + (OUT_CL ? 0 : sp.o0)) * HW), 0,
        (int)(HW * (OUT_CL ? sp.OT : sp.left) * 2), 0x00020000);
    // step (t, ks) of x: piece j = pixels 8 (lane % 8) .. + 7 of channel 8 j + lane / 8 of the step
    const u32 xoff = (u32)((lane >> 3) * HW + 8 * (lane & 7)) * 2u, xstride = (u32)(8 * HW * 2);
    u32x4 raw[RING][4];
    auto load_step = [&](int slot, long t, int ks) __attribute__((always_inline)) {
        const u32 so = (u32)((32L * ks * HW + t * 64) * 2);
#pragma unroll
        for (int j = 0; j < 4; ++j)
            raw[slot][j] = __builtin_amdgcn_raw_buffer_load_b128(rx, xoff + (u32)j * xstride, so, 0);
    };
    u32 *const xw = xt + (lane >> 3) * XS + 4 * (lane & 7);
    // transposing reads: lane L of a 16-lane block addresses row L / 4, pixels 4 (L % 4) .. + 3 of
    // the block's 16 and receives pixel L's value of the 4 rows; block kg takes channels 4 kg ..
    // (and 16 + 4 kg ..) of the step
    const u32 *const xr = xt + (4 * kg + (r16 >> 2)) * XS + 2 * (r16 & 3);
#pragma unroll
    for (int k = 0; k < RING; ++k) load_step(k, t0, k);
    for (long t = t0; t < t1; ++t) {
        f32x4 acc[4][NT];
#pragma unroll
        for (int mb = 0; mb < 4; ++mb)
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) acc[mb][nt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
#pragma unroll
            for (int j = 0; j < 4; ++j) *(u32x4 *)(xw + 8 * j * XS) = raw[ks % RING][j];
            if (ks + RING < KS) load_step(ks % RING, t, ks + RING);
            else if (t + 1 < t1) load_step(ks % RING, t + 1, ks + RING - KS);
            u32x4 a[4];
#pragma unroll
            for (int mb = 0; mb < 4; ++mb) {
                const u32x2 lo = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                                     (s16x4 __attribute__((address_space(3))) *)(xr + 8 * mb)));
                const u32x2 hi = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                                     (s16x4 __attribute__((address_space(3))) *)(xr + 16 * XS + 8 * mb)));
                a[mb] = u32x4{lo[0], lo[1], hi[0], hi[1]};
            }
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) {
                if (WIDE && 16 * nt >= sp.left) break;
                const u32x4 bm = *(const u32x4 *)(wl + (16 * nt + r16) * RW + 16 * ks + 4 * kg);
#pragma unroll
                for (int mb = 0; mb < 4; ++mb) acc[mb][nt] = Mma32<T>::run(a[mb], bm, acc[mb][nt]);
            }
        }
        // acc[mb][nt][i]: pixel 16 mb + 4 kg + i, output 16 nt + r16
        if (OUT_CL) {
            // 16 rows of 2 O bytes per block -> one contiguous run of 32 O bytes
            unsigned short *rt = (unsigned short *)xt;
#pragma unroll
            for (int mb = 0; mb < 4; ++mb) {
#pragma unroll
                for (int nt = 0; nt < NT; ++nt)
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        rt[(4 * kg + i) * (2 * OW) + 16 * nt + r16] = (unsigned short)pack2<T>(acc[mb][nt][i] + bv[nt], 0.f);
                const u32 obase = (u32)(((t * 64 + 16 * mb) * sp.OT + sp.o0) * 2);
#pragma unroll
                for (int j = 0; j < (16 * O / 8 + 63) / 64; ++j) {
                    const int i = j * 64 + lane, row = i / (O / 8), col = i % (O / 8);
                    const u32 off = WIDE ? (u32)((row * sp.OT + 8 * col) * 2) : (u32)(i * 16);
                    if ((16 * O / 8 % 64 == 0 || i < 16 * O / 8) && (!WIDE || 8 * col < sp.left))
                        __builtin_amdgcn_raw_buffer_store_b128(*(const u32x4 *)(xt + row * OW + 4 * col), ro, off + obase, 0, 2);
                }
            }
        } else {
            // a block of 16 outputs x 64 pixels (a lane holds 4 neighbouring pixels), then 16 rows of
            // 128 bytes; pieces past the plane's end are dropped
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) {
                if (WIDE && 16 * nt >= sp.left) break;
#pragma unroll
                for (int mb = 0; mb < 4; ++mb)
                    *(u32x2 *)(xt + r16 * PW + 8 * mb + 2 * kg) =
                        u32x2{pack2<T>(acc[mb][nt][0] + bv[nt], acc[mb][nt][1] + bv[nt]),
                              pack2<T>(acc[mb][nt][2] + bv[nt], acc[mb][nt][3] + bv[nt])};
                const u32 obase = (u32)((16L * nt * HW + t * 64) * 2);
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    const int row = 8 * j + (lane >> 3), col = lane & 7;
                    const u32 off = t * 64 + 8 * col < HW ? (u32)(row * HW + 8 * col) * 2u : 0x80000000u;
                    __builtin_amdgcn_raw_buffer_store_b128(*(const u32x4 *)(xt + row * PW + 4 * col), ro, off + obase, 0, 2);
                }
            }
        }
    }
}

template <typename T, int C, int O, bool OUT_CL, bool WIDE = false>
static hipError_t launch16p_co(const ProjectFeature *p, int n, int B, hipStream_t st, int outputs = O) {
    constexpr int RT = OUT_CL ? 16 * (O / 2 + 4) : 16 * 36, XT = 32 * 40;
    constexpr size_t lds = (size_t)(O * (C / 2 + 4) + 4 * (RT > XT ? RT : XT)) * 4;
    static_assert(lds <= 64 * 1024, "weights and tiles within the default LDS of a workgroup");
    for (int i = 0; i < n; ++i)
        if (p[i].HW % 8 != 0 || p[i].HW * (long)(C > outputs ? C : outputs) * 2 >= (1L << 31)) return hipErrorNotSupported;
    const int blocks_o = (outputs + O - 1) / O;
    // two workgroups are resident per CU (their registers) and the part has 256 CUs: one round of
    // at most 512 workgroups (q projection at 16 x 200 x 336 pixels:
    // 140 us against 152 with 704 workgroups)
    Feature<T> f[2] = {};
    if (!spread16(p, n, f, B, 64, blocks_o, 2)) return hipErrorNotSupported;
    hipLaunchKernelGGL((project16p_kernel<T, C, O, OUT_CL, WIDE>), dim3((unsigned)(f[0].blocks + f[1].blocks), B, blocks_o),
                       dim3(256), lds, st, f[0], f[1], outputs);
    return hipGetLastError();
}

template <typename T, bool OUT_CL>
static hipError_t launch16p(const ProjectFeature *p, int n, int B, int C, int O, hipStream_t st) {
#define SAPA_PROJECT_CASE(CV, OV) \
    if (C == CV && O == OV) return launch16p_co<T, CV, OV, OUT_CL>(p, n, B, st);
    SAPA_PROJECT_CASE(64, 32) SAPA_PROJECT_CASE(64, 64)
    SAPA_PROJECT_CASE(128, 32) SAPA_PROJECT_CASE(128, 64)
    SAPA_PROJECT_CASE(256, 32) SAPA_PROJECT_CASE(256, 64)
    SAPA_PROJECT_CASE(512, 32)
#undef SAPA_PROJECT_CASE
    return hipErrorNotSupported;
}

// ---- fp32 ----
// the three bf16 pieces of two fp32 numbers, each pair packed in a dword (x0 in the low half)
struct Pieces {
    u32 hi, mid, lo;
};
__device__ __forceinline__ Pieces split2(float x0, float x1) {
    const u32 TOP = 0xffff0000u, SEL = 0x07060302u;        // SEL: the upper halves of two dwords
    const u32 u0 = __builtin_bit_cast(u32, x0), u1 = __builtin_bit_cast(u32, x1);
    const float r0 = x0 - __builtin_bit_cast(float, u0 & TOP), r1 = x1 - __builtin_bit_cast(float, u1 & TOP);
    const u32 v0 = __builtin_bit_cast(u32, r0), v1 = __builtin_bit_cast(u32, r1);
    const float l0 = r0 - __builtin_bit_cast(float, v0 & TOP), l1 = r1 - __builtin_bit_cast(float, v1 & TOP);
    Pieces p;
    p.hi = __builtin_amdgcn_perm(u1, u0, SEL);
    p.mid = __builtin_amdgcn_perm(v1, v0, SEL);
    p.lo = __builtin_amdgcn_perm(__builtin_bit_cast(u32, l1), __builtin_bit_cast(u32, l0), SEL);
    return p;
}
__device__ __forceinline__ f32x4 mma32(u32x4 a, u32x4 b, f32x4 c) {
    typedef __bf16 v8 __attribute__((ext_vector_type(8)));
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8, a), __builtin_bit_cast(v8, b), c, 0, 0, 0);
}

// C input channels (a multiple of 32), O outputs (a multiple of 16); NW = 8 or 12 waves, tiles of 32
// pixels (two blocks of 16 matrix rows share every weight operand read from LDS).
// Reduction step ks takes channels 32 ks ..; inside it lane group kg holds channels
// 4 kg .. + 3 and 16 + 4 kg .. + 3 (two 16-byte pieces of memory; the 16 lanes of a piece
// read 64 contiguous bytes per pixel) -- the weight planes are stored in that order.
//
// IN_CL = false: x is [B, C, HW] (contiguous planes).  A lane fetches 4 neighbouring pixels of
// one channel (a wave: 8 channels x 128 bytes per load), four such loads per step, and the step's
// 32 channels x 32 pixels pass through a wave-private LDS tile from which the A operands are read
// as single dwords (the 16-pixel halves of a row swapped for every other group of 4 channels, so
// that the two channel groups of a half-wave read disjoint banks).  OUT_CL = false: out is
// [B, O, HW]; a block of 16 outputs x 32 pixels goes back through LDS and leaves as 128-byte rows
// (HW a multiple of 4: a 16-byte piece never runs from one plane into the next).
// Twelve waves (launch32_co says where): what bounds the kernel is the chain of a step (tile through LDS, pieces,
// matrix products), which three waves per SIMD hide better than two, and a round's tiles divide more finely
// (16 images, 256 -> 64: 100x168 pixels 81 -> 77 us, 50x84 35 -> 24, channels-last 86 -> 76 and 28 -> 22; 200x336
// 311 -> 300).  Their 168 registers hold two steps of x in flight instead of four; 256 -> 64 still spills 3 (planes
// to channels-last 8), 512 -> 32 2 to 5, 64 -> 64 2 to 11, 128 -> 64 from planes 11 and from channels-last
// features 19 registers.
// The tiles of a workgroup: wave after wave, so that the waves read neighbouring pieces of a plane (a plane of no whole
// cache lines is otherwise read twice at every piece's end: 128 -> 128, 3 images 150x134 28.3 -> 22.1 us, 14 images 66x82
// 41.7 -> 33.1); eight waves on planes of whole lines or on channels-last features a run of them each (neighbouring
// tiles: 256 -> 64, 8 images 128x128 38.3 -> 43.0 us, 256 -> 128, 4 images 31.3 -> 34.3; channels-last 64 -> 32, one
// image 32x32 4.05 -> 4.6).
template <int C, int O, bool IN_CL, bool OUT_CL, bool WIDE, int NW>
__global__ void __launch_bounds__(64 * NW)
project32_kernel(Feature<float> f0, Feature<float> f1, int waves, int outputs) {
    const bool second = (int)blockIdx.x >= f0.blocks;
    const Feature<float> f = second ? f1 : f0;
    const long block = (int)blockIdx.x - (second ? f0.blocks : 0);
    const int b = blockIdx.y;
    const float *__restrict__ const x = f.x, *__restrict__ const w = f.w, *__restrict__ const bias = f.bias;
    float *__restrict__ const out = f.out;
    const long HW = f.HW;
    const int tiles_per_wave = f.tiles;
    static_assert(IN_CL ? OUT_CL : true, "channels-last features give channels-last projections");
    constexpr int RW = C / 2 + 4;                 // dwords per padded row of C bf16 values
    constexpr int PLANE = O * RW;                 // dwords per piece plane
    constexpr int NT = O / 16;                    // output tiles of 16 columns
    constexpr int OS = O + 4;                     // floats per padded row of the result tile (channels-last)
    constexpr int PS = 32 + 4;                    // ... of a block of 16 outputs x 32 pixels (planes)
    constexpr int XB = IN_CL ? 0 : 32 * 32;       // floats of the wave's x tile
    constexpr int RT = OUT_CL ? 16 * OS : 16 * PS;
    constexpr int WF = RT > XB ? RT : XB;         // floats of a wave's LDS (x tile, then results)
    constexpr int KS = C / 32;                    // reduction steps
    constexpr int RING = KS < 4 || (O == 64 && NW > 8) ? 2 : 4;        // steps of x in flight
    static_assert(KS % RING == 0, "the ring of x registers is indexed by the step");
    extern __shared__ __attribute__((aligned(16))) u32 sh[];
    u32 *wl = sh;                                 // weights: 3 planes of O rows of RW dwords
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    float *rt = (float *)(sh + 3 * PLANE) + wave * WF;          // this wave's x tile / result tile
    const Span sp = span_of<O, WIDE>(outputs);

    const long ntiles = (HW + 31) / 32;
    // tiles t0, t0 + stride .. below t1 (waves past `waves` help with the weights only)
    const bool neighbours = NW > 8 || (!IN_CL && HW % 32 != 0);
    const long first = block * waves * tiles_per_wave, last = first + (long)waves * tiles_per_wave;
    const long t0 = neighbours ? first + wave : (block * waves + wave) * tiles_per_wave;
    const long t1 = wave >= waves ? t0 : neighbours ? (last < ntiles ? last : ntiles)
                                                    : (t0 + tiles_per_wave < ntiles ? t0 + tiles_per_wave : ntiles);
    const long stride = neighbours ? waves : 1;
    const int r16 = lane & 15, kg = lane >> 4;    // row / column of a 16 x 16 tile, k group
    float bv[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
        bv[nt] = bias && 16 * nt + r16 < sp.left ? bias[(WIDE ? (long)sp.o0 : (long)b * O) + 16 * nt + r16] : 0.f;

    // byte offsets inside the image: out of range = past the last pixel = zeros / dropped
    const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(
        (void *)(x + (long)b * HW * C), 0, (int)(HW * C * 4), 0x00020000);
    const __amdgpu_buffer_rsrc_t ro = __builtin_amdgcn_make_buffer_rsrc(
        (void *)(out + ((long)b * sp.OT + (OUT_CL ? 0 : sp.o0)) * HW), 0,
        (int)(HW * (OUT_CL ? sp.OT : sp.left) * 4), 0x00020000);
    // step (t, ks) of x, 4 pieces of 16 bytes per lane.  Channels-last: blocks mb = 0, 1 x pieces
    // h = 0, 1 of pixel r16's record.  Planes: piece j = pixels 4 (lane % 8) .. + 3 of channel
    // 8 j + lane / 8 of the step
    const u32 xoff = IN_CL ? (u32)(r16 * C + 4 * kg) * 4u : (u32)((lane >> 3) * HW + 4 * (lane & 7)) * 4u;
    const u32 xstride = IN_CL ? 0u : (u32)(8 * HW * 4);
    u32x4 raw[RING][2][2];
    auto load_step = [&](int slot, long t, int ks) __attribute__((always_inline)) {
        const u32 so = IN_CL ? (u32)((t * 32 * C + 32 * ks) * 4) : (u32)((32L * ks * HW + t * 32) * 4);
#pragma unroll
        for (int mb = 0; mb < 2; ++mb)
#pragma unroll
            for (int h = 0; h < 2; ++h)
                raw[slot][mb][h] = __builtin_amdgcn_raw_buffer_load_b128(
                    rx, IN_CL ? xoff + (u32)((mb * 16 * C + 16 * h) * 4) : xoff + (u32)(2 * mb + h) * xstride, so, 0);
    };
    // (planes) the x tile [32 channels][32 pixels]: where this lane writes its pieces, and where it
    // reads channel 4 kg (+ 16) of pixel r16 (+ 16)
    float *const xw = rt + (lane >> 3) * 32 + (((lane & 7) ^ ((lane >> 5) << 2)) << 2);
    const float *const xr = rt + 4 * kg * 32 + ((((r16 >> 2)) ^ ((kg & 1) << 2)) << 2) + (r16 & 3);
    // (x first: the weights come in behind its latency; a wave without a tile loads zeros or a
    // neighbouring wave's pixels)
#pragma unroll
    for (int k = 0; k < RING; ++k) load_step(k, t0, k);
    // the image's weights, taken apart, -> LDS, four neighbouring channels per thread and step, all
    // loads in flight together (outputs past the last: past the descriptor, zeros)
    {
        const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc(
            (void *)(w + (WIDE ? (long)sp.o0 : (long)b * O) * C), 0, sp.left * C * 4, 0x00020000);
        constexpr int PIECES = O * C / 4, N = (PIECES + 64 * NW - 1) / (64 * NW);
        u32x4 v[N];
#pragma unroll
        for (int k = 0; k < N; ++k)
            v[k] = __builtin_amdgcn_raw_buffer_load_b128(rw, (u32)(k * 64 * NW + threadIdx.x) * 16u, 0, 0);
#pragma unroll
        for (int k = 0; k < N; ++k) {
            const int i = k * 64 * NW + threadIdx.x, o = i / (C / 4), c = 4 * (i % (C / 4)), cs = c % 32;
            if (PIECES % (64 * NW) != 0 && i >= PIECES) break;
            const int pos = 32 * (c / 32) + 8 * ((cs % 16) / 4) + 4 * (cs / 16);
            const f32x4 f = __builtin_bit_cast(f32x4, v[k]);
            const Pieces p0 = split2(f[0], f[1]), p1 = split2(f[2], f[3]);
            u32 *dst = wl + o * RW + pos / 2;
            *(u32x2 *)dst = u32x2{p0.hi, p1.hi};
            *(u32x2 *)(dst + PLANE) = u32x2{p0.mid, p1.mid};
            *(u32x2 *)(dst + 2 * PLANE) = u32x2{p0.lo, p1.lo};
        }
    }
    __syncthreads();
    if (t0 >= t1) return;
    // An infinite feature or weight has no three pieces (inf - inf), and inf times a piece that is zero is no
    // number: a tile with a result that is not finite is formed again in plain fp32 products (a lane:
    // a pixel, every other output), which are infinite or NaN where a convolution's are.
    auto again = [&](long t, float largest) __attribute__((always_inline)) {
        if (__builtin_expect(__builtin_amdgcn_ballot_w64(!(largest < __builtin_inff())) == 0, 1)) return;
#if defined(__HIP_DEVICE_COMPILE__)
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");          // (the results below overwrite the tile's)
#endif
        const long p = t * 32 + (lane & 31);
        if (p >= HW) return;
        const float *xp = x + (long)b * HW * C + (IN_CL ? p * C : p);
        for (int o = lane >> 5; o < sp.left; o += 2) {
            const float *wp = w + ((WIDE ? (long)sp.o0 : (long)b * O) + o) * C;
            float r = 0.f;
            for (int c = 0; c < C; ++c) r = fmaf(xp[IN_CL ? (long)c : c * HW], wp[c], r);
            if (bias) r += bias[(WIDE ? (long)sp.o0 : (long)b * O) + o];
            out[OUT_CL ? ((long)b * HW + p) * sp.OT + sp.o0 + o : ((long)b * sp.OT + sp.o0 + o) * HW + p] = r;
        }
    };
    for (long t = t0; t < t1; t += stride) {
        f32x4 acc[2][NT], low[2][NT];
#pragma unroll
        for (int mb = 0; mb < 2; ++mb)
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) acc[mb][nt] = low[mb][nt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            u32x4 ahi[2], amid[2], alo[2];
            if (!IN_CL) {
#pragma unroll
                for (int j = 0; j < 4; ++j) *(u32x4 *)(xw + 8 * j * 32) = raw[ks % RING][j >> 1][j & 1];
            }
#pragma unroll
            for (int mb = 0; mb < 2; ++mb) {
                f32x4 p0, p1;
                if (IN_CL) {
                    p0 = __builtin_bit_cast(f32x4, raw[ks % RING][mb][0]);
                    p1 = __builtin_bit_cast(f32x4, raw[ks % RING][mb][1]);
                } else {
                    // (block mb: the other 16-pixel half of the row, i.e. piece index bit 2 flipped)
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        p0[e] = xr[e * 32 + (mb ? 16 - 32 * (kg & 1) : 0)];
                        p1[e] = xr[(16 + e) * 32 + (mb ? 16 - 32 * (kg & 1) : 0)];
                    }
                }
                const Pieces s0 = split2(p0[0], p0[1]), s1 = split2(p0[2], p0[3]);
                const Pieces s2 = split2(p1[0], p1[1]), s3 = split2(p1[2], p1[3]);
                ahi[mb] = u32x4{s0.hi, s1.hi, s2.hi, s3.hi};
                amid[mb] = u32x4{s0.mid, s1.mid, s2.mid, s3.mid};
                alo[mb] = u32x4{s0.lo, s1.lo, s2.lo, s3.lo};
            }
            // the ring slot is free: the step RING further on (of this tile or of the next)
            if (ks + RING < KS) load_step(ks % RING, t, ks + RING);
            else if (t + stride < t1) load_step(ks % RING, t + stride, ks + RING - KS);
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) {
                if (WIDE && 16 * nt >= sp.left) break;
                const u32 *wp = wl + (16 * nt + r16) * RW + 16 * ks + 4 * kg;
                const u32x4 bhi = *(const u32x4 *)wp, bmid = *(const u32x4 *)(wp + PLANE), blo = *(const u32x4 *)(wp + 2 * PLANE);
#pragma unroll
                for (int mb = 0; mb < 2; ++mb) {
                    // smallest terms first, in a sum of their own: added to the large one term by term each
                    // would round it again (C = 64 .. 512, 128 .. 800 outputs: relative error 1.0 .. 3.4e-7 so,
                    // library convolutions 0.9 .. 2.8e-7, now 0.7 .. 1.4e-7; the same time)
                    f32x4 a = mma32(ahi[mb], blo, low[mb][nt]);
                    a = mma32(alo[mb], bhi, a);
                    a = mma32(amid[mb], bmid, a);
                    a = mma32(ahi[mb], bmid, a);
                    low[mb][nt] = mma32(amid[mb], bhi, a);
                    acc[mb][nt] = mma32(ahi[mb], bhi, acc[mb][nt]);
                }
            }
            // (nothing of a later step moves up: it would not fit the registers of 12 waves)
            if (NW > 8) __builtin_amdgcn_sched_barrier(0);
        }
        float largest = 0.f;
#pragma unroll
        for (int mb = 0; mb < 2; ++mb)
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) {
                acc[mb][nt] += low[mb][nt];
#pragma unroll
                for (int i = 0; i < 4; ++i) largest = __builtin_elementwise_maximum(largest, __builtin_fabsf(acc[mb][nt][i]));
            }
        // acc[mb][nt][i]: pixel 16 mb + 4 kg + i, output 16 nt + r16
        if (!OUT_CL) {
            // planes: a block of 16 outputs x 32 pixels -> the wave's tile (a lane holds 4
            // neighbouring pixels), then 16 rows of 128 bytes; pieces past the plane's end are dropped
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) {
                if (WIDE && 16 * nt >= sp.left) break;
#pragma unroll
                for (int mb = 0; mb < 2; ++mb) {
                    const f32x4 v = {acc[mb][nt][0] + bv[nt], acc[mb][nt][1] + bv[nt], acc[mb][nt][2] + bv[nt],
                                     acc[mb][nt][3] + bv[nt]};
                    *(f32x4 *)(rt + r16 * PS + 16 * mb + 4 * kg) = v;
                }
                const u32 obase = (u32)((16L * nt * HW + t * 32) * 4);
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    const int row = 8 * j + (lane >> 3), col = lane & 7;
                    const u32 off = t * 32 + 4 * col < HW ? (u32)(row * HW + 4 * col) * 4u : 0x80000000u;
                    __builtin_amdgcn_raw_buffer_store_b128(*(const u32x4 *)(rt + row * PS + 4 * col), ro, off + obase, 0, 2);
                }
            }
            again(t, largest);
            continue;
        }
        // channels-last: the wave's tile, then 16 rows of 4 O bytes -> one contiguous run of 64 O
        // bytes per block
#pragma unroll
        for (int mb = 0; mb < 2; ++mb) {
#pragma unroll
            for (int nt = 0; nt < NT; ++nt)
#pragma unroll
                for (int i = 0; i < 4; ++i) rt[(4 * kg + i) * OS + 16 * nt + r16] = acc[mb][nt][i] + bv[nt];
            const u32 obase = (u32)(((t * 32 + 16 * mb) * sp.OT + sp.o0) * 4);
#pragma unroll
            for (int j = 0; j < (16 * O / 4 + 63) / 64; ++j) {
                const int i = j * 64 + lane, row = i / (O / 4), col = i % (O / 4);
                const u32 off = WIDE ? (u32)((row * sp.OT + 4 * col) * 4) : (u32)(i * 16);
                if ((16 * O / 4 % 64 == 0 || i < 16 * O / 4) && (!WIDE || 4 * col < sp.left))
                    __builtin_amdgcn_raw_buffer_store_b128(*(const u32x4 *)(rt + row * OS + 4 * col), ro, off + obase, 0, 2);
            }
        }
        again(t, largest);
    }
}

template <int C, int O, bool IN_CL, bool OUT_CL, bool WIDE, int NW>
static hipError_t launch32_waves(const ProjectFeature *p, int n, int B, hipStream_t st, int outputs, const Spread &s) {
    constexpr int RT = OUT_CL ? 16 * (O + 4) : 16 * 36, XB = IN_CL ? 0 : 32 * 32;
    constexpr size_t lds = (size_t)(3 * O * (C / 2 + 4) + NW * (RT > XB ? RT : XB)) * 4;
    static_assert(lds <= 160 * 1024, "weights and tiles must fit LDS");
    const int blocks_o = (outputs + O - 1) / O;
    Feature<float> f[2] = {};
    for (int i = 0; i < n; ++i)
        f[i] = Feature<float>{(const float *)p[i].x, (const float *)p[i].w, (const float *)p[i].bias, (float *)p[i].out, p[i].HW,
                              (int)s.per, (int)s.blocks[i]};
    if (s.blocks[0] > 65535 * 32L || s.blocks[1] > 65535 * 32L || B > 65535 || blocks_o > 65535) return hipErrorNotSupported;
    auto kern = project32_kernel<C, O, IN_CL, OUT_CL, WIDE, NW>;
    if (lds > 64 * 1024) {
        int dev = 0, most = 0;
        if (hipGetDevice(&dev) != hipSuccess ||
            hipDeviceGetAttribute(&most, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) != hipSuccess ||
            (size_t)most < lds ||
            hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize,
                                (int)lds) != hipSuccess) {
            (void)hipGetLastError();
            return hipErrorNotSupported;
        }
    }
    hipLaunchKernelGGL(kern, dim3((unsigned)(f[0].blocks + f[1].blocks), B, blocks_o), dim3(64 * NW), lds, st, f[0], f[1],
                       s.waves, outputs);
    return hipGetLastError();
}

template <int C, int O, bool IN_CL, bool OUT_CL, bool WIDE = false>
static hipError_t launch32_co(const ProjectFeature *p, int n, int B, hipStream_t st, int outputs = O) {
    long ntiles[2] = {0, 0};
    for (int i = 0; i < n; ++i) {
        if (!OUT_CL && p[i].HW % 4 != 0) return hipErrorNotSupported;
        // 32-bit byte offsets inside an image
        if (p[i].HW * (long)(C > outputs ? C : outputs) * 4 >= (1L << 31)) return hipErrorNotSupported;
        ntiles[i] = (p[i].HW + 31) / 32;
    }
    const long sets = (long)B * ((outputs + O - 1) / O);     // sets: workgroups that share a pixel range's place
    const Spread s8 = plan32(ntiles, sets, 8), s12 = plan32(ntiles, sets, 12);
    // Twelve waves where they shorten a wave's chain of tiles to what is asked for below (eight have twice the steps of
    // x in flight and no bar to moving work between steps).  us with 8 / 12 waves, from planes: 5 tiles to 3 each
    // (256 -> 64, 16 images 100x168) 66 / 60, 3 to 2 (256 -> 288, 8 images 64x64) 41.8 / 38.6, but 4 to 3
    // (256 -> 400, 8 images 64x64) 45.3 / 46.5 and 11 to 8 (14 images 66x82, 800 outputs) 160 / 187 of 128 channels, 242 / 265
    // of 256; from channels-last features 5 to 3 (256 -> 64) 64.9 / 61.9, but 7 to 5 (256 -> 288, 14 images 72x68) 70 / 74
    // and, spilling, 5 to 3 at 128 -> 64 37 / 38.5 .. 42; of 64 channels 5 to 3 (64 -> 64, 16 images 100x168) 24.7 / 23.6, 9
    // to 6 (64 -> 800, 16 images 50x84) 70.7 / 73.3; 128 -> 32 with 2 tiles to 1 (16 images 50x84) 11.7 / 14.1.  Tenths
    // of eight waves' tiles per tile of twelve waves:
    constexpr int ASKED = C == 128 && O == 32 ? 1 << 20 : !IN_CL ? 15 : C == 128 ? 20 : C == 64 ? 16 : 15;
    // (of 64 channels not to a single tile: 2 images 192x192, 64 -> 32 / 64, 7.7 / 8.3 and 10.1 / 10.8; 256 -> 64 from
    // channels-last features also over one tile each for 3 to 6 waves: 8 images 64x64 13.9 / 12.5)
    if ((10 * s8.per >= ASKED * s12.per && (C > 64 || s12.per > 1)) || (IN_CL && C == 256 && O == 64 && s8.per == 1 && s8.waves > 2 && s8.waves <= 6))
        return launch32_waves<C, O, IN_CL, OUT_CL, WIDE, C == 128 && O == 32 ? 8 : 12>(p, n, B, st, outputs, s12);
    return launch32_waves<C, O, IN_CL, OUT_CL, WIDE, 8>(p, n, B, st, outputs, s8);
}

template <bool IN_CL, bool OUT_CL>
static hipError_t launch32(const ProjectFeature *p, int n, int B, int C, int O, hipStream_t st) {
#define SAPA_PROJECT_CASE(CV, OV) \
    if (C == CV && O == OV) return launch32_co<CV, OV, IN_CL, OUT_CL>(p, n, B, st);
    SAPA_PROJECT_CASE(64, 32) SAPA_PROJECT_CASE(64, 64)
    SAPA_PROJECT_CASE(128, 32) SAPA_PROJECT_CASE(128, 64)
    SAPA_PROJECT_CASE(256, 32) SAPA_PROJECT_CASE(256, 64)
    SAPA_PROJECT_CASE(512, 32)
#undef SAPA_PROJECT_CASE
    return hipErrorNotSupported;
}

template <typename T>
static hipError_t launch_t(const ProjectFeature *p, int n, int B, int C, int O, hipStream_t st) {
#define SAPA_PROJECT_CASE(CV, OV) \
    if (C == CV && O == OV) return launch_co<T, CV, OV>(p, n, B, st);
    SAPA_PROJECT_CASE(64, 32) SAPA_PROJECT_CASE(64, 64)
    SAPA_PROJECT_CASE(128, 32) SAPA_PROJECT_CASE(128, 64) SAPA_PROJECT_CASE(128, 128)
    SAPA_PROJECT_CASE(256, 32) SAPA_PROJECT_CASE(256, 64) SAPA_PROJECT_CASE(256, 128)
    SAPA_PROJECT_CASE(512, 32) SAPA_PROJECT_CASE(512, 64)
#undef SAPA_PROJECT_CASE
    return hipErrorNotSupported;
}

// one output block per 64 outputs (32 where 512 channels' weights leave no room for more)
template <typename T, bool IN_CL, bool OUT_CL>
static hipError_t launch_shared(const ProjectFeature *p, int n, int B, int C, int O, hipStream_t st) {
#define SAPA_SHARED_CASE(CV, OV)                                                                                     \
    if (C == CV) {                                                                                                   \
        if constexpr (sizeof(T) == 4) return launch32_co<CV, OV, IN_CL, OUT_CL, true>(p, n, B, st, O); \
        else if constexpr (IN_CL) return launch_co<T, CV, OV, true>(p, n, B, st, O);                  \
        else return launch16p_co<T, CV, OV, OUT_CL, true>(p, n, B, st, O);                            \
    }
    SAPA_SHARED_CASE(64, 64) SAPA_SHARED_CASE(128, 64) SAPA_SHARED_CASE(256, 64) SAPA_SHARED_CASE(512, 32)
#undef SAPA_SHARED_CASE
    return hipErrorNotSupported;
}

}  // namespace project

// A plain 1x1 convolution: weights w [O, C] and bias [O] (or null) shared by all images, x and out
// in contiguous or channels-last order; C in {64, 128, 256, 512}, O a multiple of 8; what
// project_nhwc_launch / project_nchw_launch require of HW and of pointers holds here too.
hipError_t project_shared_launch(const void *x, const void *w, const void *bias, void *out, int B, int C, int O,
                                 long HW, int x_channels_last, int out_channels_last, int dtype, hipStream_t st) {
    const void *ptrs[3] = {x, w, out};
    for (const void *p : ptrs)
        if ((uintptr_t)p % 16 != 0) return hipErrorNotSupported;
    const ProjectFeature f{x, w, bias, out, HW};
    if (O % 8 != 0 || (x_channels_last && !out_channels_last)) return hipErrorNotSupported;
#define SAPA_SHARED(TV)                                                                                       \
    return x_channels_last ? project::launch_shared<TV, true, true>(&f, 1, B, C, O, st)         \
           : out_channels_last ? project::launch_shared<TV, false, true>(&f, 1, B, C, O, st)    \
                               : project::launch_shared<TV, false, false>(&f, 1, B, C, O, st)
    if (dtype == 0) SAPA_SHARED(float);
    if (dtype == 2) SAPA_SHARED(f16_t);
    if (dtype == 3) SAPA_SHARED(bf16_t);
#undef SAPA_SHARED
    return hipErrorNotSupported;
}

// One projection, or two of the same B, C and O, with per-image weights w [B, O, C] and bias [B, O] or null:
//   x_channels_last: x [B, HW, C] -> out [B, HW, O]; f16 / bf16 / fp32; (C, O) among the instantiated pairs (C in
//     {64, 128, 256, 512}, O in {32, 64, 128}; fp32: those whose three weight planes fit LDS);
//   else x [B, C, HW] (planes) -> out [B, HW, O] (out_channels_last) or [B, O, HW]; the (C, O) pairs of the fp32
//     kernel; fp32: HW a multiple of 4 for a planar result; f16 / bf16: HW a multiple of 8.
// x, w and out aligned to 16 bytes.  hipErrorNotSupported otherwise (of two that take a launch each, the first may have gone
// out then: callers ask project_supported before).
hipError_t project_launch(const ProjectFeature *f, int n, int B, int C, int O, bool x_channels_last, bool out_channels_last,
                          int dtype, hipStream_t st) {
    for (int i = 0; i < n; ++i)
        if (((uintptr_t)f[i].x | (uintptr_t)f[i].w | (uintptr_t)f[i].out) % 16 != 0) return hipErrorNotSupported;
    // Two that together have no more tiles than the chip's waves (2048) go as one launch: the smaller one's latencies
    // lie beside the other's.  Modules, us before and so: bf16, 8 images 16x16, C=256, 35 -> 26 (29 with 2 tiles per wave
    // at least), channels-last 41 -> 36; fp32 45 -> 36, 4 of 24x24 47 -> 40.  Larger ones take a launch each: 16 of 50x84
    // in fp32 102 -> 109 for the two projections, 100x168 in channels-last bf16 176 -> 172 and the operator behind them 3 more.
    const long tile = dtype == 0 ? 32 : x_channels_last ? 16 : 64;
    if (n == 2 && ((f[0].HW + tile - 1) / tile + (f[1].HW + tile - 1) / tile) * B > 2048) {
        const hipError_t e = project_launch(f, 1, B, C, O, x_channels_last, out_channels_last, dtype, st);
        return e == hipSuccess ? project_launch(f + 1, 1, B, C, O, x_channels_last, out_channels_last, dtype, st) : e;
    }
    if (x_channels_last) {
        if (dtype == 0) return project::launch32<true, true>(f, n, B, C, O, st);
        if (dtype == 2) return project::launch_t<f16_t>(f, n, B, C, O, st);
        if (dtype == 3) return project::launch_t<bf16_t>(f, n, B, C, O, st);
        return hipErrorNotSupported;
    }
    if (dtype == 2)
        return out_channels_last ? project::launch16p<f16_t, true>(f, n, B, C, O, st) : project::launch16p<f16_t, false>(f, n, B, C, O, st);
    if (dtype == 3)
        return out_channels_last ? project::launch16p<bf16_t, true>(f, n, B, C, O, st) : project::launch16p<bf16_t, false>(f, n, B, C, O, st);
    if (dtype != 0) return hipErrorNotSupported;
    return out_channels_last ? project::launch32<false, true>(f, n, B, C, O, st) : project::launch32<false, false>(f, n, B, C, O, st);
}

hipError_t project_nhwc_launch(const void *x, const void *w, const void *bias, void *out, int B, int C, int O, long HW,
                               int dtype, hipStream_t st) {
    const ProjectFeature f{x, w, bias, out, HW};
    return project_launch(&f, 1, B, C, O, true, true, dtype, st);
}

hipError_t project_nchw_launch(const void *x, const void *w, const void *bias, void *out, int B, int C, int O, long HW,
                               int out_channels_last, int dtype, hipStream_t st) {
    const ProjectFeature f{x, w, bias, out, HW};
    return project_launch(&f, 1, B, C, O, false, out_channels_last != 0, dtype, st);
}

// Whether project_nhwc_launch (x_channels_last; the result is channels-last then) / project_nchw_launch
// has a kernel for the configuration, pointer alignment aside.
bool project_supported(int C, int O, long HW, bool x_channels_last, bool out_channels_last, int dtype) {
    const bool small_pair = (C == 64 && (O == 32 || O == 64)) || (C == 128 && (O == 32 || O == 64)) ||
                            (C == 256 && (O == 32 || O == 64)) || (C == 512 && O == 32);
    if (dtype == 2 || dtype == 3) {
        if (x_channels_last)
            return out_channels_last && (small_pair || (C == 128 && O == 128) || (C == 256 && O == 128) || (C == 512 && O == 64));
        return small_pair && HW % 8 == 0 && HW * (long)(C > O ? C : O) * 2 < (1L << 31);
    }
    if (dtype != 0 || !small_pair || HW * (long)(C > O ? C : O) * 4 >= (1L << 31)) return false;
    if (x_channels_last) return out_channels_last;
    return out_channels_last || HW % 4 == 0;
}

}  // namespace sapa
