// What the dense-window kernels on the 16-bit matrix instructions share: operand types, the
// matrix instructions by element type, rounding and splitting of fp32 values, transposing LDS reads.
#pragma once
#include "kernels.hpp"

namespace sapa {

namespace wm {

typedef unsigned u32;
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef u32 u32x2 __attribute__((ext_vector_type(2)));
typedef u32 u32x3 __attribute__((ext_vector_type(3)));
typedef u32 u32x4 __attribute__((ext_vector_type(4)));
typedef short s16x4 __attribute__((ext_vector_type(4)));

constexpr u32 OUTSIDE = 0x80000000u;      // past the end of every buffer descriptor: reads zero, stores nothing
constexpr float LOG2E = 1.4426950408889634f;

// Whether the byte offsets inside an image of up to `channels` planes of `plane` bytes are distinct 32-bit
// numbers below OUTSIDE, and those of the last chunk's channels past the image (a chunk has 16), which
// lie outside too, do not come round to its beginning
inline bool offsets_fit(long channels, long plane) {
    return channels * plane < (1L << 31) && (channels + 15) / 16 * 16 * plane <= (1L << 32);
}

template <typename T> struct Mma;
template <> struct Mma<f16_t> {
    typedef _Float16 v4 __attribute__((ext_vector_type(4)));
    typedef _Float16 v8 __attribute__((ext_vector_type(8)));
    static __device__ __forceinline__ f32x4 k16(u32x2 a, u32x2 b, f32x4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x16f16(__builtin_bit_cast(v4, a), __builtin_bit_cast(v4, b), c, 0, 0, 0);
    }
    static __device__ __forceinline__ f32x4 k32(u32x4 a, u32x4 b, f32x4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(v8, a), __builtin_bit_cast(v8, b), c, 0, 0, 0);
    }
};
template <> struct Mma<bf16_t> {
    typedef __bf16 v8 __attribute__((ext_vector_type(8)));
    static __device__ __forceinline__ f32x4 k16(u32x2 a, u32x2 b, f32x4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(s16x4, a), __builtin_bit_cast(s16x4, b), c, 0, 0, 0);
    }
    static __device__ __forceinline__ f32x4 k32(u32x4 a, u32x4 b, f32x4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8, a), __builtin_bit_cast(v8, b), c, 0, 0, 0);
    }
};

template <typename T>
__device__ __forceinline__ u32 pack2(float a, float b) {
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    typedef T tx2 __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(u32, __builtin_convertvector(f32x2{a, b}, tx2));
}

// 8 fp32 values as a 16-bit operand plus the operands of the remainders: N in all
template <typename T, int N>
__device__ __forceinline__ void split8(const float *p, u32x4 (&o)[N]) {
    typedef T tx8 __attribute__((ext_vector_type(8)));
    float r[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) r[k] = p[k];
#pragma unroll
    for (int i = 0; i < N; ++i) {
        o[i] = u32x4{pack2<T>(r[0], r[1]), pack2<T>(r[2], r[3]), pack2<T>(r[4], r[5]), pack2<T>(r[6], r[7])};
        const tx8 h = __builtin_bit_cast(tx8, o[i]);
#pragma unroll
        for (int k = 0; k < 8; ++k) r[k] -= (float)h[k];
    }
}
template <typename T>
__device__ __forceinline__ void split8(const float *p, u32x4 &hi, u32x4 &lo) {
    u32x4 o[2];
    split8<T>(p, o);
    hi = o[0], lo = o[1];
}

// f16 holds a pair of operands to 2^-25 only and nothing beyond 65504, whatever its values' own size: a set
// of values is multiplied by a power of two that takes its largest magnitude m to 2^14 .. 2^15 before
// it is split, and sums of products by its inverse (exact: the pair then holds 23 bits of the largest
// values and 2^-40 of it of the others).  bf16 has fp32's range: 1.
struct Fit {
    float up, down;
};
template <typename T>
__device__ __forceinline__ Fit fit(float m) {
    if constexpr (!__is_same(T, f16_t)) return Fit{1.f, 1.f};
    const u32 b = __builtin_bit_cast(u32, m) >> 23, e = b < 27u ? 27u : b;    // (both factors normal numbers)
    return Fit{__builtin_bit_cast(float, (268u - e) << 23), __builtin_bit_cast(float, (e - 14u) << 23)};
}
// the same in every lane: the largest of the four lane groups' m
__device__ __forceinline__ float over_groups(float m) {
    m = fmaxf(m, __shfl_xor(m, 16));
    return fmaxf(m, __shfl_xor(m, 32));
}

// value k of the operands made by split8
template <typename T, int N>
__device__ __forceinline__ float joined(const u32x4 (&o)[N], int k) {
    typedef T tx8 __attribute__((ext_vector_type(8)));
    float v = (float)__builtin_bit_cast(tx8, o[N - 1])[k];
#pragma unroll
    for (int i = N - 2; i >= 0; --i) v += (float)__builtin_bit_cast(tx8, o[i])[k];
    return v;
}
template <typename T>
__device__ __forceinline__ float joined(u32x4 hi, u32x4 lo, int k) {
    const u32x4 o[2] = {hi, lo};
    return joined<T>(o, k);
}

// a 4 x 4 block of 16-bit values out of LDS, transposed: lane L of a 16-lane block addresses 4
// consecutive values of row L / 4 and receives column L's value of the 4 rows
__device__ __forceinline__ u32x2 read_tr(const u32 *p) {
    return __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                                         (s16x4 __attribute__((address_space(3))) *)p));
}

// Buffer descriptor of `bytes` bytes at p, as the four dwords load_lds takes
__device__ __forceinline__ u32x4 dma_rsrc(const void *p, u32 bytes) {
    const unsigned long long a = (unsigned long long)p;
    return u32x4{(u32)a, (u32)(a >> 32) & 0xffffu, bytes, 0x00020000u};
}

// Direct load of 16 bytes per lane from a buffer into LDS (lane l: the l-th 16-byte piece from LDS byte
// address `at` on, which is wave-uniform).  Written out, because of what the compiler does with its
// builtin: it knows that the instruction writes LDS, and in front of the next transposing LDS read (an
// intrinsic, so without an address it could compare) it waits for every load in flight -- the loads just
// issued for a later chunk among them, which ends all prefetching.  The waits are the kernel's own
// (wait_all_but).  m0 is named as written, so that the compiler, which merges its own settings of m0 where nothing
// writes it between them, sets it again for its own direct loads.  (It warns that m0 is a reserved register, whose value
// is not kept for it: none is in it here.)
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
template <bool NT = false>
__device__ __forceinline__ void load_lds(u32x4 r, u32 at, u32 off) {
#if defined(__HIP_DEVICE_COMPILE__)
    if constexpr (NT)
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen nt lds" ::"s"(at), "v"(off), "s"(r) : "memory", "m0");
    else
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds" ::"s"(at), "v"(off), "s"(r) : "memory", "m0");
#endif
}
#pragma clang diagnostic pop

// LDS byte address of a __shared__ array
__device__ __forceinline__ u32 lds_address(const __attribute__((address_space(3))) u32 *p) { return (u32)(unsigned long long)p; }

// waits until at most `after` vector-memory operations of this wave are outstanding (they retire in
// issue order; the compiler does not track a direct load's LDS write, so the waits are written out)
__device__ __forceinline__ void wait_all_but(int after) {
#if defined(__HIP_DEVICE_COMPILE__)
#define SAPA_WAIT_CASE(N) case N: asm volatile("s_waitcnt vmcnt(" #N ")" ::: "memory"); break;
    switch (after) {
        SAPA_WAIT_CASE(1) SAPA_WAIT_CASE(2) SAPA_WAIT_CASE(3) SAPA_WAIT_CASE(4) SAPA_WAIT_CASE(5) SAPA_WAIT_CASE(6)
        SAPA_WAIT_CASE(7) SAPA_WAIT_CASE(8) SAPA_WAIT_CASE(9) SAPA_WAIT_CASE(10) SAPA_WAIT_CASE(11)
        default: asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); break;
    }
#undef SAPA_WAIT_CASE
#endif
}

// this wave's LDS writes are done; then every wave's (and every wave's landed loads)
__device__ __forceinline__ void lds_barrier() {
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
#endif
}

}  // namespace wm

}  // namespace sapa
