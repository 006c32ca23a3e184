// Backward of the fused SAPA-B operator for channels-last f16 / bf16 tensors on the 16-bit matrix
// instructions, K = 5, s = 2: the two kernels of sapa_b_bwd16.hip (which states the products and why
// the attention weights are formed again instead of being stored) in the layout of
// sapa_b_nhwc_wm16.hip.  q, grad_q [B,2H,2W,d], key, grad_key [B,H,W,d], value, grad_value [B,H,W,C],
// grad_out [B,2H,2W,C].  (Reference: sapa/sapa/src/cuda/qk_cuda_kernel.cu:101-137,
// av_cuda_kernel.cu:103-148.)
//
// What the layout changes: products that reduce over channels (S, G) read both operands 16 bytes at
// a time; those that reduce over cells or children (grad_q; grad_value, grad_key) take one operand
// through ds_read_tr16_b64 and leave 4 (8) consecutive channels in a lane; every position is a whole
// unit of memory, so tiles have no edge cases, W may be odd, and a halo costs only its own bytes.
//
// Non-finite operands: as there.
//
// Measured: a training step at B=16, C=256, d=64, 100x168 in bf16 0.73 ms (pixel kernel 206 us, cell
// kernel 342) against 1.64 through copies into contiguous order and the chain over K * K tensors; at B=8,
// C=256, d=32, 64x64 in fp16 148 us against 271 (26 + 47 us).  The pixel kernel waits for memory (1.0 GB);
// the cell kernel for LDS and L2: every hi-res value is staged 1.9 times and read by four blocks.
#include "wm16_exact.hpp"

namespace sapa {

namespace cbwm16 {

using namespace wm;

// makes the compiler wait here for a value that is being loaded: behind this kernel's own wait for
// everything in flight it costs nothing, while at the value's first use the loads requested since then
// (which the compiler does not see) would be waited for as well
__device__ __forceinline__ void arrived(u32x4 &v) {
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("" : "+v"(v));
#endif
}

template <typename T> struct Args {
    const T *q, *key, *value, *grad_out;
    float *stats;
    T *grad_q, *grad_key, *grad_value;
    int B, d, C, H, W, tiles_x, tiles_y, ns, nblocks, per_xcd;
};

// ---- per-child gradients ----
// A workgroup of 2 NSW waves owns up to NSW blocks of 4 x 4 parents side by side; waves t and t + NSW
// share block t, 32 of its children each.  Windows of 64 channels in two LDS buffers; q and grad_out go
// from global memory into the operand registers, a chunk ahead.
constexpr int CHK = 64;            // channels per staged chunk = 8 pieces of 16 bytes per cell
constexpr int CELL = CHK / 2;      // dwords per cell
constexpr int NSW = 4;
constexpr int WC = 4 * NSW + 4;    // window cells per row of the tile
constexpr int LOWBUF = 8 * WC * CELL;
constexpr int OSLOT = 16 * CELL;   // dwords of a wave's output slot: 16 children x 64 channels

// dword offset of the 16-byte piece `piece` (0..7) of cell / child `idx` in a [idx][64 channels] array
__device__ __forceinline__ int piece_at(int idx, int piece) { return idx * CELL + ((piece ^ (idx & 7)) << 2); }

// its slow way for the blocks of a tile that are named
template <typename T>
__device__ __attribute__((noinline)) void children_again(Again again) {
    settled();
    const Args<T> a = again.arguments<Args<T>>();
    const int at = (int)(again.workgroup() % 8) * a.per_xcd + (int)(again.workgroup() / 8), n = at / (a.tiles_x * a.tiles_y);
    const int cy = 8 * (at / a.tiles_x % a.tiles_y), cx = 8 * a.ns * (at % a.tiles_x);
    const long lpix = (long)a.H * a.W;
    for (u32 b = 0, blocks = again.of_blocks(); blocks >> b; ++b)
        if (blocks >> b & 1)
            exact_grad_q<T, 128 * NSW>(again.floats(), plane_of<true>(a.q, n, a.d, 4 * lpix), plane_of<true>(a.key, n, a.d, lpix),
                                       plane_of<true>(a.value, n, a.C, lpix), plane_of<true>(a.grad_out, n, a.C, 4 * lpix),
                                       plane_of<true>(a.grad_q, n, a.d, 4 * lpix), a.stats + (2L * a.B + n) * 4 * lpix, a.d, a.C,
                                       a.H, a.W, cy, cx + 8 * (int)b);
}

template <typename T, bool STREAM>
__global__ __launch_bounds__(128 * NSW, 4) void
bwd_pixel_kernel(const Args<T> args) {
    const T *__restrict__ const q = args.q, *__restrict__ const key = args.key, *__restrict__ const value = args.value,
            *__restrict__ const grad_out = args.grad_out;
    T *__restrict__ const grad_q = args.grad_q;
    float *__restrict__ const stats = args.stats;
    const int B = args.B, d = args.d, C = args.C, H = args.H, W = args.W, tiles_x = args.tiles_x, tiles_y = args.tiles_y,
              ns = args.ns, nblocks = args.nblocks, per_xcd = args.per_xcd;
    constexpr int NT = 128 * NSW;
    constexpr int NLP = LOWBUF / 4;                          // 16-byte pieces per window buffer
    constexpr int NLI = (NLP + NT - 1) / NT;                 // direct loads per thread and window, at most
    static_assert(NLP % 64 == 0, "whole direct loads");
    constexpr int STREAM_AUX = STREAM ? 2 : 0;
    constexpr bool SCALED = __is_same(T, f16_t);             // E is brought into the type's range (Fit)
    __shared__ __attribute__((aligned(16))) u32 lds[2 * LOWBUF + 2 * NSW * OSLOT + 4];
    u32 *const non_finite = lds + 2 * LOWBUF + 2 * NSW * OSLOT;          // blocks of the tile with a non-finite result
    const u32 low_at = lds_address((const __attribute__((address_space(3))) u32 *)lds);

    const int logical = (int)(blockIdx.x % 8) * per_xcd + (int)(blockIdx.x / 8);
    if (logical >= nblocks) return;
    const int tx = logical % tiles_x, ty = (logical / tiles_x) % tiles_y, n = logical / (tiles_x * tiles_y);
    const int X0 = tx * 4 * ns, Y0 = ty * 4;                 // first parent of the tile
    const int nsx = (W + 3) / 4;
    const int ns_here = nsx - tx * ns < ns ? nsx - tx * ns : ns;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g = lane >> 4, i16 = lane & 15;
    const int t = wave % NSW, half = wave / NSW;
    const bool active = t < ns_here;
    const long lpix = (long)H * W;

    // piece `slot % 8` of window cell `slot / 8`: its cell of the image, and the channel of the chunk
    u32 cell_low[NLI];
#pragma unroll
    for (int i = 0; i < NLI; ++i) {
        const int slot = i * NT + tid, cell = slot >> 3;
        const int y = Y0 - 2 + cell / WC, x = X0 - 2 + cell % WC;
        const bool ok = (slot < NLP) & (cell % WC < 4 * ns_here + 4) & ((u32)y < (u32)H) & ((u32)x < (u32)W);
        cell_low[i] = ok ? (u32)(y * W + x) : OUTSIDE;
    }
    const int ch_low = 8 * ((tid & 7) ^ ((tid >> 3) & 7));     // (NT / 8 is a multiple of 8: the same for every i)
    const u32x4 rk = dma_rsrc(key + (long)n * d * lpix, (u32)(d * lpix * (long)sizeof(T)));
    const u32x4 rv = dma_rsrc(value + (long)n * C * lpix, (u32)(C * lpix * (long)sizeof(T)));
    const __amdgpu_buffer_rsrc_t rq = __builtin_amdgcn_make_buffer_rsrc(
        (void *)(q + (long)n * d * 4 * lpix), 0, (int)(d * 4 * lpix * (long)sizeof(T)), 0x00020000);
    const __amdgpu_buffer_rsrc_t rg = __builtin_amdgcn_make_buffer_rsrc(
        (void *)(grad_out + (long)n * C * 4 * lpix), 0, (int)(C * 4 * lpix * (long)sizeof(T)), 0x00020000);

    const int nKc = (d + CHK - 1) / CHK, nVc = (C + CHK - 1) / CHK;
    const int ntot = nKc + nVc + (grad_q ? nKc : 0);
    // chunk j: key + q (S), value + grad_out (G), key again (grad_q)
    auto stage = [&](int j) __attribute__((always_inline)) {
        if (j >= ntot) return;
        const bool is_val = j >= nKc && j < nKc + nVc;
        const int cx = is_val ? C : d, c0 = (j < nKc ? j : is_val ? j - nKc : j - nKc - nVc) * CHK;
        const u32x4 r = is_val ? rv : rk;
        const u32 lb = low_at + ((j & 1) * LOWBUF + wave * 256) * 4;
#pragma unroll
        for (int i = 0; i < NLI; ++i)
            if ((i + 1) * NT <= NLP || i * NT + wave * 64 < NLP) {
                const bool ok = (c0 + ch_low < cx) & (cell_low[i] != OUTSIDE);
                load_lds(r, lb + i * NT * 16, ok ? (cell_low[i] * (u32)cx + (u32)(c0 + ch_low)) * (u32)sizeof(T) : OUTSIDE);
            }
    };
    // this lane's child of block nb = 0, 1: row 4 half + 2 nb + i16 / 8, column i16 % 8 of the block's 8 x 8
    const int hW = 2 * W, hH = 2 * H;
    const int cy0 = 2 * Y0 + 4 * half + (i16 >> 3), cx0 = 2 * X0 + 8 * t + (i16 & 7);
    u32 child[2];
#pragma unroll
    for (int nb = 0; nb < 2; ++nb) child[nb] = active && cy0 + 2 * nb < hH && cx0 < hW ? (u32)((cy0 + 2 * nb) * hW + cx0) : OUTSIDE;
    // q / grad_out of chunk j: B operand of reduction step s = channels 32 s + 8 g .. + 7 of the child
    struct Hi {
        u32x4 v[2][2];
    };
    auto fetch = [&](int j, Hi &h) __attribute__((always_inline)) {
        if (j >= nKc + nVc) return;
        const bool is_val = j >= nKc;
        const int cx = is_val ? C : d, c0 = (is_val ? j - nKc : j) * CHK;
#pragma unroll
        for (int nb = 0; nb < 2; ++nb)
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                const int c = c0 + 32 * s + 8 * g;
                const bool ok = (c < cx) & (child[nb] != OUTSIDE);
                const u32 off = ok ? (child[nb] * (u32)cx + (u32)c) * (u32)sizeof(T) : OUTSIDE;
                h.v[nb][s] = is_val ? __builtin_amdgcn_raw_buffer_load_b128(rg, off, 0, STREAM_AUX)
                                    : __builtin_amdgcn_raw_buffer_load_b128(rq, off, 0, STREAM_AUX);
            }
    };
    // Sim[cell][child], 4 x 2 accumulator blocks of 16 x 16: block (mb, nb), lane (g, i16), element v: cell
    // (row 2 mb + g / 2, column 4 (g % 2) + v) of the window, child i16 of block nb
    auto similarity = [&](int j, const Hi &h, f32x4 (&acc)[4][2]) __attribute__((always_inline)) {
        const u32 *kb = lds + (j & 1) * LOWBUF;
#pragma unroll
        for (int s = 0; s < 2; ++s) {
#pragma unroll
            for (int mb = 0; mb < 4; ++mb) {
                const int cell = (2 * mb + (i16 >> 3)) * WC + 4 * t + (i16 & 7);
                const u32x4 a = *(const u32x4 *)(kb + piece_at(cell, 4 * s + g));
#pragma unroll
                for (int nb = 0; nb < 2; ++nb) acc[mb][nb] = Mma<T>::k32(a, h.v[nb][s], acc[mb][nb]);
            }
        }
    };
    auto zero = [](f32x4 (&acc)[4][2]) __attribute__((always_inline)) {
#pragma unroll
        for (int mb = 0; mb < 4; ++mb) acc[mb][0] = acc[mb][1] = f32x4{0.f, 0.f, 0.f, 0.f};
    };
    // chunk j is done with: chunk j + 1 complete for everyone (its windows in LDS, its `hi` in registers),
    // chunk j + 2 requested
    auto next = [&](int j, Hi &hi, Hi &spare) __attribute__((always_inline)) {
        wait_all_but(0);
#pragma unroll
        for (int k = 0; k < 4; ++k) arrived(hi.v[k >> 1][k & 1]);
        lds_barrier();
        stage(j + 2);
        fetch(j + 2, spare);
    };
    f32x4 acc[4][2];
    Hi h0, h1;
    if (tid == 0) *non_finite = 0;
    stage(0);
    fetch(0, h0);
    fetch(1, h1);
    wait_all_but(0);
#pragma unroll
    for (int k = 0; k < 4; ++k) arrived(h0.v[k >> 1][k & 1]), arrived(h1.v[k >> 1][k & 1]);
    lds_barrier();
    stage(1);
    zero(acc);
    int j = 0;
    // (the chunk's hi-res operand is h0 at every turn: h1 moves up)
    for (; j < nKc; ++j) {
        if (active) similarity(j, h0, acc);
        h0 = h1;
        next(j, h0, h1);
    }

    // ---- softmax over each child's 5 x 5 cells ----
    f32x4 p[4][2];
    float mlog[2], inv[2];
    const int px = (i16 & 7) >> 1;
    auto inside = [&](int mb, int nb, int v) __attribute__((always_inline)) {
        return ((u32)(4 * (g & 1) + v - px) <= 4u) & ((u32)(2 * mb + (g >> 1) - (2 * half + nb)) <= 4u);
    };
    if (active) {
        const float NEG_INF = -__builtin_inff();
#pragma unroll
        for (int nb = 0; nb < 2; ++nb) {
            float m = NEG_INF;
#pragma unroll
            for (int mb = 0; mb < 4; ++mb) {
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    p[mb][nb][v] = inside(mb, nb, v) ? acc[mb][nb][v] : NEG_INF;
                    m = fmaxf(m, p[mb][nb][v]);
                }
            }
            m = fmaxf(m, __shfl_xor(m, 16));
            m = fmaxf(m, __shfl_xor(m, 32));
            mlog[nb] = m * LOG2E;
            float sum = 0.f;
#pragma unroll
            for (int mb = 0; mb < 4; ++mb)
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    p[mb][nb][v] = __builtin_amdgcn_exp2f(__builtin_fmaf(p[mb][nb][v], LOG2E, -mlog[nb]));
                    sum += p[mb][nb][v];
                }
            sum += __shfl_xor(sum, 16);
            sum += __shfl_xor(sum, 32);
            inv[nb] = 1.f / sum;
#pragma unroll
            for (int mb = 0; mb < 4; ++mb)
#pragma unroll
                for (int v = 0; v < 4; ++v) p[mb][nb][v] *= inv[nb];
        }
    }

    // ---- gradient of the weights ----
    zero(acc);
    for (; j < nKc + nVc; ++j) {
        if (active) similarity(j, h0, acc);
        h0 = h1;
        next(j, h0, h1);
    }

    // ---- gradient of the logits; what the cell kernel needs to form it again ----
    u32x4 whi[2][2], wlo[2][2];
    NonFinite seen;
    float down[2];              // f16: what the results of this lane's child of block nb are multiplied by
    if (active) {
#pragma unroll
        for (int nb = 0; nb < 2; ++nb) {
            float dsum = 0.f;
#pragma unroll
            for (int mb = 0; mb < 4; ++mb)
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    // (as sapa_b_bwd16.hip has it, without this, the kernel needs 20 registers more than there are:
                    // B=16, C=256, 100x168 in bf16 584 us for both kernels, 545 so)
                    if (!inside(mb, nb, v)) acc[mb][nb][v] = 0.f;
                    dsum = __builtin_fmaf(p[mb][nb][v], acc[mb][nb][v], dsum);
                }
            dsum += __shfl_xor(dsum, 16);
            dsum += __shfl_xor(dsum, 32);
            if (g < 3 && child[nb] != OUTSIDE)
                // planes [3][B, 2H, 2W]: maximum (times log2 e), 1 / sum, D; lanes g = 0, 1, 2 one each
                stats[((long)g * B + n) * 4 * lpix + child[nb]] = g == 0 ? mlog[nb] : g == 1 ? inv[nb] : dsum;
            // reduction step s of the last product covers the cells of blocks mb = 2 s, 2 s + 1
            float e[2][8], m = 0.f;
#pragma unroll
            for (int s = 0; s < 2; ++s)
#pragma unroll
                for (int k = 0; k < 8; ++k) {
                    e[s][k] = p[2 * s + k / 4][nb][k % 4] * (acc[2 * s + k / 4][nb][k % 4] - dsum);
                    if (SCALED) m = fmaxf(m, __builtin_fabsf(e[s][k]));
                }
            if (SCALED) {
                const Fit f = fit<T>(over_groups(m));
                down[nb] = f.down;
#pragma unroll
                for (int k = 0; k < 16; ++k) e[k / 8][k % 8] *= f.up;
            }
#pragma unroll
            for (int s = 0; s < 2; ++s) split8<T>(e[s], whi[nb][s], wlo[nb][s]);
        }
    }

    // ---- grad_q^T[channel][child], per chunk of 64 channels, through this wave's slot ----
    const __amdgpu_buffer_rsrc_t ro = __builtin_amdgcn_make_buffer_rsrc(
        (void *)(grad_q + (long)n * d * 4 * lpix), 0, (int)(d * 4 * lpix * (long)sizeof(T)), 0x00020000);
    u32 *oslot = lds + 2 * LOWBUF + wave * OSLOT;
    for (; j < ntot; ++j) {
        const int c0 = (j - nKc - nVc) * CHK;
        if (active) {
            const u32 *vb = lds + (j & 1) * LOWBUF;
            u32x4 va[4][2];
#pragma unroll
            for (int mk = 0; mk < 4; ++mk)
#pragma unroll
                for (int s = 0; s < 2; ++s) {
                    const int cell = (4 * s + (g >> 1)) * WC + 4 * t + 4 * (g & 1) + (i16 >> 2);
                    const int piece = 2 * mk + ((i16 & 3) >> 1);
                    const u32x2 lo = read_tr(vb + piece_at(cell, piece) + 2 * (i16 & 1));
                    const u32x2 hi = read_tr(vb + piece_at(cell + 2 * WC, piece) + 2 * (i16 & 1));
                    va[mk][s] = u32x4{lo[0], lo[1], hi[0], hi[1]};
                }
#pragma unroll
            for (int nb = 0; nb < 2; ++nb) {
#pragma unroll
                for (int mk = 0; mk < 4; ++mk) {
                    f32x4 o = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int s = 0; s < 2; ++s) {
                        o = Mma<T>::k32(va[mk][s], whi[nb][s], o);
                        o = Mma<T>::k32(va[mk][s], wlo[nb][s], o);
                    }
                    if (nb == 0) seen.see(o);
                    if (SCALED) o *= down[nb];
                    *(u32x2 *)(oslot + piece_at(i16, 2 * mk + (g >> 1)) + 2 * (g & 1)) =
                        u32x2{pack2<T>(o[0], o[1]), pack2<T>(o[2], o[3])};
                }
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    const int pc = lane + 64 * i, ch = c0 + 8 * (pc & 7);
                    const u32x4 o = *(const u32x4 *)(oslot + piece_at(pc >> 3, pc & 7));
                    const int cy = 2 * Y0 + 4 * half + 2 * nb + (pc >> 6), cx = 2 * X0 + 8 * t + ((pc >> 3) & 7);
                    const bool ok = (cy < hH) & (cx < hW) & (ch < d);
                    __builtin_amdgcn_raw_buffer_store_b128(o, ro, ok ? (u32)((cy * hW + cx) * d + ch) * (u32)sizeof(T) : OUTSIDE, 0, STREAM_AUX);
                }
            }
        }
        if (j + 1 < ntot) {
            wait_all_but(0);
            lds_barrier();
            stage(j + 2);
        }
    }

    // ---- blocks with a non-finite result: again, term by term ----
    if (seen.any()) atomicOr(non_finite, 1u << t);
    lds_barrier();
    const u32 blocks = __builtin_amdgcn_readfirstlane(*non_finite);
    if (__builtin_expect(blocks != 0, 0)) children_again<T>(Again(lds, blocks));
}

// ---- per-cell gradients ----
// A workgroup owns 4 x 2 blocks of 4 x 4 cells (which start 2 cells left of / above a multiple of 4) and
// stages the 5 x 3 parent blocks their children lie in, 32 channels (64 bytes) of 24 x 40 children, in
// two LDS buffers; key and value of a wave's own cells go into registers.  Two waves share a block, one
// per row of quadrants: the lower row's wave hands its sums over through LDS, the other adds and stores.
constexpr int TBX = 4, TBY = 2;
constexpr int CNT = 128 * TBX * TBY;
constexpr int CCH = 32;                            // channels per chunk
constexpr int XC = 8 * (TBX + 1), XR = 8 * (TBY + 1);   // staged children per row, rows
constexpr int CHI = XR * XC * CCH / 2;             // dwords per buffer
constexpr int CNH = (CHI / 4 + CNT - 1) / CNT;
constexpr int CPART = 64 * TBX * TBY * 8;          // floats of a chunk's handed-over sums
constexpr int CSTAT = 1024;                        // floats of one stats plane (24 x 40), in whole loads of 4 waves
static_assert(XR * XC <= CSTAT && 2 * CSTAT <= 2 * CPART, "stats planes");
static_assert((2 * CHI + CSTAT + 2 * CPART + 4) * 4 <= 160 * 1024, "LDS");
static_assert(XC % 8 == 0 && CNT % 64 == 0, "piece permutation");

// the slow way of bwd_cell_kernel for the cell blocks of its tile that are named
template <typename T>
__device__ __attribute__((noinline)) void cells_again(Again again) {
    settled();
    const Args<T> a = again.arguments<Args<T>>();
    const int at = (int)(again.workgroup() % 8) * a.per_xcd + (int)(again.workgroup() / 8), n = at / (a.tiles_x * a.tiles_y);
    const int cy = 4 * TBY * (at / a.tiles_x % a.tiles_y) - 2, cx = 4 * TBX * (at % a.tiles_x) - 2;
    const long lpix = (long)a.H * a.W;
    for (u32 b = 0, blocks = again.of_blocks(); blocks >> b; ++b)
        if (blocks >> b & 1)
            exact_grad_cells<T, CNT>(again.floats(), plane_of<true>(a.q, n, a.d, 4 * lpix), plane_of<true>(a.key, n, a.d, lpix),
                                     plane_of<true>(a.value, n, a.C, lpix), plane_of<true>(a.grad_out, n, a.C, 4 * lpix),
                                     a.stats + n * 4 * lpix, (long)a.B * 4 * lpix, plane_of<true>(a.grad_key, n, a.d, lpix),
                                     plane_of<true>(a.grad_value, n, a.C, lpix), a.d, a.C, a.H, a.W, cy + 4 * (int)(b / TBX),
                                     cx + 4 * (int)(b % TBX));
}

template <typename T>
__global__ __launch_bounds__(CNT) void
bwd_cell_kernel(const Args<T> args) {
    const T *__restrict__ const q = args.q, *__restrict__ const key = args.key, *__restrict__ const value = args.value,
            *__restrict__ const grad_out = args.grad_out;
    T *__restrict__ const grad_key = args.grad_key, *__restrict__ const grad_value = args.grad_value;
    const float *__restrict__ const stats = args.stats;
    const int B = args.B, d = args.d, C = args.C, H = args.H, W = args.W, tiles_x = args.tiles_x, tiles_y = args.tiles_y,
              nblocks = args.nblocks, per_xcd = args.per_xcd;
    constexpr bool SCALED = __is_same(T, f16_t);             // A and E are brought into the type's range (Fit)
    __shared__ __attribute__((aligned(16))) u32 lds[2 * CHI + CSTAT + 2 * CPART + 4];
    u32 *const non_finite = lds + 2 * CHI + CSTAT + 2 * CPART;           // cell blocks with a non-finite result
    float *const statbuf = (float *)(lds + 2 * CHI), *const part = statbuf + CSTAT;   // (D; the other planes over `part`)
    const u32 hi_base = lds_address((const __attribute__((address_space(3))) u32 *)lds);

    const int logical = (int)(blockIdx.x % 8) * per_xcd + (int)(blockIdx.x / 8);
    if (logical >= nblocks) return;
    const int tx = logical % tiles_x, ty = (logical / tiles_x) % tiles_y, n = logical / (tiles_x * tiles_y);
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g = lane >> 4, i16 = lane & 15;
    const int blk = wave % (TBX * TBY), qy = wave / (TBX * TBY);
    const int bi = blk % TBX, bj = blk / TBX, I0 = tx * TBX, J0 = ty * TBY;
    const bool active = 4 * (I0 + bi) - 2 < W && 4 * (J0 + bj) - 2 < H;
    const long lpix = (long)H * W;
    const int hW = 2 * W, hH = 2 * H;

    // staged piece slot % 4 of child slot / 4 (pieces XOR-permuted by child / 4: the 16-byte reads of 8
    // neighbouring children touch every bank once)
    u32 pix[CNH];
#pragma unroll
    for (int i = 0; i < CNH; ++i) {
        const int c = (i * CNT + tid) >> 2, cy = 8 * (J0 - 1) + c / XC, cx = 8 * (I0 - 1) + c % XC;
        const bool ok = (c < XR * XC) & ((u32)cy < (u32)hH) & ((u32)cx < (u32)hW);
        pix[i] = ok ? (u32)(cy * hW + cx) : OUTSIDE;
    }
    const int ch_hi = 8 * ((tid & 3) ^ ((tid >> 4) & 3));
    const int nKc = (d + CCH - 1) / CCH, nVc = (C + CCH - 1) / CCH;
    const int ntot = nKc + nVc + (grad_key ? nKc : 0);
    const u32x4 rq = dma_rsrc(q + (long)n * d * 4 * lpix, (u32)(d * 4 * lpix * (long)sizeof(T)));
    const u32x4 rg = dma_rsrc(grad_out + (long)n * C * 4 * lpix, (u32)(C * 4 * lpix * (long)sizeof(T)));
    const __amdgpu_buffer_rsrc_t rk = __builtin_amdgcn_make_buffer_rsrc(
        (void *)(key + (long)n * d * lpix), 0, (int)(d * lpix * (long)sizeof(T)), 0x00020000);
    const __amdgpu_buffer_rsrc_t rv = __builtin_amdgcn_make_buffer_rsrc(
        (void *)(value + (long)n * C * lpix), 0, (int)(C * lpix * (long)sizeof(T)), 0x00020000);

    // chunk j: q + key (S), grad_out + value (G and grad_value), q again (grad_key)
    auto stage = [&](int j) __attribute__((always_inline)) {
        if (j >= ntot) return;
        const bool is_val = j >= nKc && j < nKc + nVc;
        const int cx = is_val ? C : d, c0 = (j < nKc ? j : is_val ? j - nKc : j - nKc - nVc) * CCH;
        const u32 hb = hi_base + ((j & 1) * CHI + wave * 256) * 4;
        const u32x4 r = is_val ? rg : rq;
#pragma unroll
        for (int i = 0; i < CNH; ++i)
            if ((i + 1) * CNT <= CHI / 4 || i * CNT + wave * 64 < CHI / 4) {
                const bool ok = (c0 + ch_hi < cx) & (pix[i] != OUTSIDE);
                load_lds(r, hb + i * CNT * 16, ok ? (pix[i] * (u32)cx + (u32)(c0 + ch_hi)) * (u32)sizeof(T) : OUTSIDE);
            }
    };
    // this lane's cell, and 8 channels of its key / value for chunk j (B operand of the similarity)
    const int cr = i16 >> 2, cc = i16 & 3, ly = 4 * (J0 + bj) - 2 + cr, lx = 4 * (I0 + bi) - 2 + cc;
    const bool cell_in = ((u32)ly < (u32)H) & ((u32)lx < (u32)W);
    const u32 cell = cell_in ? (u32)(ly * W + lx) : OUTSIDE;
    auto fetch = [&](int j) __attribute__((always_inline)) {
        u32x4 v = {0u, 0u, 0u, 0u};
        if (j < nKc + nVc) {
            const bool is_val = j >= nKc;
            const int cx = is_val ? C : d, c = (is_val ? j - nKc : j) * CCH + 8 * g;
            const u32 off = (cell_in & (c < cx)) ? (cell * (u32)cx + (u32)c) * (u32)sizeof(T) : OUTSIDE;
            v = is_val ? __builtin_amdgcn_raw_buffer_load_b128(rv, off, 0, 0) : __builtin_amdgcn_raw_buffer_load_b128(rk, off, 0, 0);
        }
        return v;
    };

    // quadrant (qy, qx): parent block (bj + 1 - qy, bi + 1 - qx) of the staged 3 x 5.  Similarity block
    // (qx, nb): rows = the 16 children of parent row nb, columns = the wave's cells; lane (g, cell i16),
    // element v: child (row 2 nb + g / 2, column 4 (g % 2) + v)
    int sim_at[2], gat_at[2];
#pragma unroll
    for (int qx = 0; qx < 2; ++qx) {
        const int r = 8 * (bj + 1 - qy), x = 8 * (bi + 1 - qx);
        const int cs = (r + (i16 >> 3)) * XC + x + (i16 & 7);
        sim_at[qx] = cs * (CCH / 2) + ((g ^ ((cs >> 2) & 3)) << 2);
        const int cg = (r + (g >> 1)) * XC + x + 4 * (g & 1) + (i16 >> 2);
        gat_at[qx] = cg * (CCH / 2) + (((i16 & 3) ^ ((cg >> 2) & 3)) << 2);
    }
    constexpr int ROW2 = 2 * XC * CCH / 2;                    // dwords of two rows (which keep a child's permutation)
    static_assert((2 * XC / 4) % 4 == 0, "piece permutation");
    auto similarity = [&](int j, u32x4 low, f32x4 (&acc)[2][4]) __attribute__((always_inline)) {
        const u32 *hb = lds + (j & 1) * CHI;
#pragma unroll
        for (int qx = 0; qx < 2; ++qx)
#pragma unroll
            for (int nb = 0; nb < 4; ++nb)
                acc[qx][nb] = Mma<T>::k32(*(const u32x4 *)(hb + sim_at[qx] + nb * ROW2), low, acc[qx][nb]);
    };
    // the gathered sum over this wave's 128 children of 32 channels: reduction step (qx, s) covers parent rows
    // 2 s and 2 s + 1 of the quadrant, in the order the weights are held in.  Transposing read of tile h: lane
    // L of a 16-lane block addresses child L / 4 of the 4, channels 8 (L % 4) + 4 h .. + 3; so element v of
    // result h: channel 8 g + 4 h + v of cell i16
    u32x4 whi[2][2], wlo[2][2];
    Fit f = {1.f, 1.f};         // f16: the factors of this lane's cell
    auto hold = [&](float (&w)[2][2][8]) __attribute__((always_inline)) {
        if (SCALED) {
            float m = 0.f;
#pragma unroll
            for (int k = 0; k < 32; ++k) m = fmaxf(m, __builtin_fabsf(w[k / 16][k / 8 % 2][k % 8]));
            f = fit<T>(over_groups(m));
#pragma unroll
            for (int k = 0; k < 32; ++k) w[k / 16][k / 8 % 2][k % 8] *= f.up;
        }
#pragma unroll
        for (int qx = 0; qx < 2; ++qx)
#pragma unroll
            for (int s = 0; s < 2; ++s) split8<T>(w[qx][s], whi[qx][s], wlo[qx][s]);
    };
    NonFinite seen;
    auto gather = [&](int j, f32x4 (&o)[2]) __attribute__((always_inline)) {
        const u32 *hb = lds + (j & 1) * CHI;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            o[h] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int qx = 0; qx < 2; ++qx)
#pragma unroll
                for (int s = 0; s < 2; ++s) {
                    const u32x2 lo = read_tr(hb + gat_at[qx] + 2 * s * ROW2 + 2 * h), hi = read_tr(hb + gat_at[qx] + (2 * s + 1) * ROW2 + 2 * h);
                    const u32x4 a = u32x4{lo[0], lo[1], hi[0], hi[1]};
                    o[h] = Mma<T>::k32(a, whi[qx][s], o[h]);
                    o[h] = Mma<T>::k32(a, wlo[qx][s], o[h]);
                }
            seen.see(o[h]);
            if (SCALED) o[h] *= f.down;
        }
        if (qy) {
            float *p = part + (j & 1) * CPART + blk * 512 + lane * 4;
            *(f32x4 *)p = o[0];
            *(f32x4 *)(p + 256) = o[1];
        }
    };
    auto store = [&](int j, const f32x4 (&o)[2], __amdgpu_buffer_rsrc_t ro, int cx, int c0) __attribute__((always_inline)) {
        const float *p = part + (j & 1) * CPART + blk * 512 + lane * 4;
        const f32x4 a = o[0] + *(const f32x4 *)p, b = o[1] + *(const f32x4 *)(p + 256);
        const u32x4 v = {pack2<T>(a[0], a[1]), pack2<T>(a[2], a[3]), pack2<T>(b[0], b[1]), pack2<T>(b[2], b[3])};
        const int c = c0 + 8 * g;
        const bool ok = cell_in & (c < cx);
        __builtin_amdgcn_raw_buffer_store_b128(v, ro, ok ? (cell * (u32)cx + (u32)c) * (u32)sizeof(T) : OUTSIDE, 0, 0);
    };

    // the three stats planes of the staged children, straight into LDS.  Zeros outside the image -- and, for
    // an odd W, the statistics of the next row's first two children in a row's last piece: their weights are
    // finite (a child at the row's left end has zeros among its logits: its maximum is not negative) and
    // meet the zeros that are staged as such a child's q and grad_out
    if (wave < 12) {
        const int k = wave / 4, c = (wave % 4 * 64 + lane) * 4, cy = 8 * (J0 - 1) + c / XC, cx = 8 * (I0 - 1) + c % XC;
        const bool ok = (c < XR * XC) & ((u32)cy < (u32)hH) & ((u32)cx < (u32)hW);
        load_lds(dma_rsrc(stats + ((long)((k + 2) % 3) * B + n) * 4 * lpix, (u32)(16 * lpix)),
                 hi_base + (2 * CHI + k * CSTAT + wave % 4 * 256) * 4, ok ? (u32)(cy * hW + cx) * 4u : OUTSIDE);
    }
    auto child_stats = [&](int k, int qx, int nb) __attribute__((always_inline)) {
        return *(const f32x4 *)(statbuf + k * CSTAT + (8 * (bj + 1 - qy) + 2 * nb + (g >> 1)) * XC + 8 * (bi + 1 - qx) + 4 * (g & 1));
    };

    f32x4 acc[2][4];
    auto zero = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int qx = 0; qx < 2; ++qx)
#pragma unroll
            for (int nb = 0; nb < 4; ++nb) acc[qx][nb] = f32x4{0.f, 0.f, 0.f, 0.f};
    };
    zero();
    if (tid == 0) *non_finite = 0;
    stage(0);
    u32x4 l0 = fetch(0), l1 = fetch(1);
    wait_all_but(0);
    arrived(l0);
    arrived(l1);
    lds_barrier();
    stage(1);
    // chunk j is done with: chunk j + 1 complete for everyone, chunk j + 2 requested (stored: behind the
    // loads of chunk j + 1 the wave issued one store)
    auto next = [&](int j, bool stored) __attribute__((always_inline)) {
        wait_all_but(stored ? 1 : 0);
        arrived(l1);
        lds_barrier();
        stage(j + 2);
        l0 = l1;
        l1 = fetch(j + 2);
    };
    int j = 0;
    for (; j < nKc; ++j) {
        if (active) similarity(j, l0, acc);
        next(j, false);
    }

    // ---- the weights of the wave's cells: A = exp2(S log2 e - max) / sum inside a child's window ----
    if (active) {
        float w[2][2][8];
#pragma unroll
        for (int qx = 0; qx < 2; ++qx)
#pragma unroll
            for (int s = 0; s < 2; ++s)
#pragma unroll
                for (int k = 0; k < 2; ++k) {
                    const int nb = 2 * s + k;
                    const f32x4 mlog = child_stats(1, qx, nb), inv = child_stats(2, qx, nb);
                    const bool row_ok = qy ? cr <= nb : cr >= nb;
#pragma unroll
                    for (int v = 0; v < 4; ++v) {
                        const int px = 2 * (g & 1) + (v >> 1);
                        const bool ok = row_ok & (qx ? cc <= px : cc >= px);
                        const float e = __builtin_amdgcn_exp2f(__builtin_fmaf(acc[qx][nb][v], LOG2E, -mlog[v]));
                        w[qx][s][4 * k + v] = ok ? e * inv[v] : 0.f;
                    }
                }
        hold(w);
    }
    lds_barrier();         // (the sums handed over for the first chunks overwrite the stats)

    // ---- G and grad_value ----
    zero();
    f32x4 o[2];
    {
        // (a NULL grad_value: a descriptor of no bytes drops the stores)
        const __amdgpu_buffer_rsrc_t ro = __builtin_amdgcn_make_buffer_rsrc(
            (void *)(grad_value + (long)n * C * lpix), 0, grad_value ? (int)(C * lpix * (long)sizeof(T)) : 0, 0x00020000);
        for (; j < nKc + nVc; ++j) {
            if (active) {
                if (grad_key) similarity(j, l0, acc);
                gather(j, o);
            }
            next(j, active && !qy && j > nKc);
            if (active && !qy) store(j, o, ro, C, (j - nKc) * CCH);
        }
    }

    // ---- E = A (G - D), grad_key ----
    if (grad_key) {
        if (active) {
            float w[2][2][8];
#pragma unroll
            for (int qx = 0; qx < 2; ++qx)
#pragma unroll
                for (int s = 0; s < 2; ++s)
#pragma unroll
                    for (int k = 0; k < 2; ++k) {
                        const int nb = 2 * s + k;
                        const f32x4 dsum = child_stats(0, qx, nb);
#pragma unroll
                        for (int v = 0; v < 4; ++v)
                            w[qx][s][4 * k + v] = joined<T>(whi[qx][s], wlo[qx][s], 4 * k + v) * f.down * (acc[qx][nb][v] - dsum[v]);
                    }
            hold(w);
        }
        const __amdgpu_buffer_rsrc_t ro = __builtin_amdgcn_make_buffer_rsrc(
            (void *)(grad_key + (long)n * d * lpix), 0, (int)(d * lpix * (long)sizeof(T)), 0x00020000);
        for (; j < ntot; ++j) {
            if (active) gather(j, o);
            next(j, active && !qy);
            if (active && !qy) store(j, o, ro, d, (j - nKc - nVc) * CCH);
        }
    }

    // ---- blocks with a non-finite result: again, term by term ----
    if (seen.any()) atomicOr(non_finite, 1u << blk);
    lds_barrier();
    const u32 blocks = __builtin_amdgcn_readfirstlane(*non_finite);
    if (__builtin_expect(blocks != 0, 0)) cells_again<T>(Again(lds, blocks));
}

template <typename T, bool STREAM>
static hipError_t launch(const void *q, const void *key, const void *value, const void *grad_out, float *stats,
                         void *grad_q, void *grad_key, void *grad_value, int B, int d, int C, int H, int W,
                         hipStream_t st) {
    Args<T> args{(const T *)q, (const T *)key, (const T *)value, (const T *)grad_out, stats, (T *)grad_q, (T *)grad_key,
                 (T *)grad_value, B, d, C, H, W, 0, 0, 0, 0, 0};
    // sets the tiles; false: too many
    auto tile = [&](int tiles_x, int tiles_y) {
        const long nb = (long)tiles_x * tiles_y * B;
        args.tiles_x = tiles_x, args.tiles_y = tiles_y, args.nblocks = (int)nb, args.per_xcd = (int)((nb + 7) / 8);
        return nb <= (1L << 30);
    };
    {
        const int nsx = (W + 3) / 4;
        if (!tile((nsx + NSW - 1) / NSW, (H + 3) / 4)) return hipErrorNotSupported;
        args.ns = (nsx + args.tiles_x - 1) / args.tiles_x;    // blocks per tile, balanced over the row
        hipLaunchKernelGGL((bwd_pixel_kernel<T, STREAM>), dim3(args.per_xcd * 8), dim3(128 * NSW), 0, st, args);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    if (!grad_key && !grad_value) return hipSuccess;
    // cell blocks 4 I - 2 .. 4 I + 1 that hold a cell of 0 .. W - 1
    const int nI = (W + 1) / 4 + 1, nJ = (H + 1) / 4 + 1;
    if (!tile((nI + TBX - 1) / TBX, (nJ + TBY - 1) / TBY)) return hipErrorNotSupported;
    hipLaunchKernelGGL((bwd_cell_kernel<T>), dim3(args.per_xcd * 8), dim3(CNT), 0, st, args);
    return hipGetLastError();
}

}  // namespace cbwm16

bool sapa_b_nhwc_bwd16_serves(int d, int C, int H, int W, int K, int s, int dtype) {
    return K == 5 && s == 2 && d % 8 == 0 && C % 8 == 0 && (dtype == 2 || dtype == 3) &&
           (long)(d > C ? d : C) * H * W * 8 < (1L << 31);
}

// Gradients of the fused operator (any of them may be NULL) for channels-last tensors; f16 / bf16,
// K = 5, s = 2, d and C multiples of 8, tensors aligned to 16 bytes, every image of every tensor below
// 2 GiB; stats: 3 floats per output pixel.  hipErrorNotSupported otherwise (nothing is launched then).
hipError_t sapa_b_nhwc_bwd16_launch(const void *q, const void *key, const void *value, const void *grad_out,
                                    void *stats, void *grad_q, void *grad_key, void *grad_value, int B, int d,
                                    int C, int H, int W, int K, int s, int dtype, hipStream_t st) {
    if (!sapa_b_nhwc_bwd16_serves(d, C, H, W, K, s, dtype)) return hipErrorNotSupported;
    if (((uintptr_t)q | (uintptr_t)key | (uintptr_t)value | (uintptr_t)grad_out | (uintptr_t)stats | (uintptr_t)grad_q |
         (uintptr_t)grad_key | (uintptr_t)grad_value) % 16 != 0)
        return hipErrorNotSupported;
    const bool stream = 2L * ((long)B * H * W * (5L * d + 5L * C)) > (256L << 20);
    float *f = (float *)stats;
    if (dtype == 2)
        return stream ? cbwm16::launch<f16_t, true>(q, key, value, grad_out, f, grad_q, grad_key, grad_value, B, d, C, H, W, st)
                      : cbwm16::launch<f16_t, false>(q, key, value, grad_out, f, grad_q, grad_key, grad_value, B, d, C, H, W, st);
    return stream ? cbwm16::launch<bf16_t, true>(q, key, value, grad_out, f, grad_q, grad_key, grad_value, B, d, C, H, W, st)
                  : cbwm16::launch<bf16_t, false>(q, key, value, grad_out, f, grad_q, grad_key, grad_value, B, d, C, H, W, st);
}

}  // namespace sapa
