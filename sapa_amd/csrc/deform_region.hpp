// Geometry and helpers of the 16-bit SAPA-D backward (s = 2, sapa_d_region_bwd16.hip): a workgroup owns a
// strip of RPX parents (RW hi-res pixels) of one (image, group) and walks down it by one row of parents a step.
//
// A step's samples lie within RCH cells of their parents (those that do not are handled apart), i.e. in a band of
// BROWS rows of the strip's window of WWX cells per row.  Its dense products run over the blocks of 16 window cells
// that hold the band: NBLK from the one its first cell is in, and a pixel's row of Sim / Wm has an entry per
// cell of those blocks.
#pragma once
#include "deform_tap.hpp"
#include "wm16_common.hpp"

namespace sapa {

namespace dreg {

using wm::f32x4;
using wm::Mma;
using wm::OUTSIDE;
using wm::read_tr;
using wm::u32;
using wm::u32x2;
using wm::u32x4;

constexpr int S = 2;                        // up_factor
constexpr int RCH = 4;                      // window reach around a parent, in low-res cells
constexpr int RPX = 8, RW = RPX * S;        // parents / pixels of a strip along x
constexpr int WWX = RPX + 2 * RCH + 1;      // window cells along x
constexpr int BROWS = 2 * RCH + 2;          // window rows of a step's band
constexpr int NBLK = (BROWS * WWX + 15 + 15) / 16, BC = 16 * NBLK;     // blocks of 16 cells that hold a band, their cells
// dwords per row of Sim / Wm: 20 mod 64, so that the accumulators' rows (4 apart) and the 16 rows of a
// 16-byte operand read start on disjoint groups of banks
constexpr int RS = BC + 20;
static_assert(RS % 64 == 20, "bank layout of the rows");
constexpr float WSCALE = 1073741824.f;      // 2^30: fixed-point scale of Wm

// first cell of the blocks of parent row pr
__device__ __forceinline__ int band_base(int pr) { return pr * WWX / 16 * 16; }

// Whether a 32-bit word holds a 16-bit value that is not finite (its exponent bits are all set)
template <typename T>
__device__ __forceinline__ bool not_finite(u32 x) {
    constexpr u32 EXP = __is_same(T, f16_t) ? 0x7c007c00u : 0x7f807f80u;
    constexpr u32 ONE = __is_same(T, f16_t) ? 0x04000400u : 0x00800080u;
    return ((x & EXP) + ONE) & 0x80008000u;
}
template <typename T>
__device__ __forceinline__ bool not_finite(u32x4 x) {
    return not_finite<T>(x[0]) | not_finite<T>(x[1]) | not_finite<T>(x[2]) | not_finite<T>(x[3]);
}

}  // namespace dreg

}  // namespace sapa
