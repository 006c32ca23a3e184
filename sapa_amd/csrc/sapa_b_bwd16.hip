// Backward of the fused SAPA-B operator for contiguous (NCHW) f16 / bf16 tensors on the 16-bit
// matrix instructions, K = 5, s = 2: all three gradients from the four operands in two kernels,
// nothing of size K * K ever in memory.
//
//   S = q . key, A = softmax(S), G = grad_out . value  (over a child's 5 x 5 cells)
//   D = sum_cells A * G,  E = A * (G - D)
//   grad_q[child]    = sum_cells E * key[cell]           bwd_pixel_kernel
//   grad_value[cell] = sum_children A * grad_out[child]  bwd_cell_kernel
//   grad_key[cell]   = sum_children E * q[child]         bwd_cell_kernel
//
// (reference: sapa/sapa/src/cuda/qk_cuda_kernel.cu:101-137 and av_cuda_kernel.cu:103-148, whose
// atomicAdd per product becomes a sum in registers here.)  As in the forward kernel
// (sapa_b_wmat16.hip) the products are written densely over blocks of 4 x 4 parents and 8 x 8
// cells, of which a child uses 25.
//
// bwd_pixel_kernel works on blocks of 4 x 4 parents (64 children) as the forward kernel does and
// leaves three numbers per child behind: the softmax's maximum and 1 / sum, and D.  With those a
// second kernel can form A and E for any (child, cell) pair from one dot product each, so
// bwd_cell_kernel turns the assignment round: a wave owns 4 x 4 cells and gathers over the 256
// children of the 8 x 8 parents around them, recomputing S and G for its cells only (a quarter
// of a window) while it passes over grad_out once for both G and grad_value.  The alternative, A
// and E written by the first kernel and read by the second, moves 2 x 100 values per parent
// (430 MB each way at B=16, 100x168 in fp32) for the 2 x 29 % more matrix work that this costs.
//
// Operands: A and E enter the products as a 16-bit value plus a 16-bit remainder (f16: of values brought
// into its range, see Fit) and, with odd W, a second remainder: calls with even W have had pairs since these
// kernels serve them, those with odd W had fp32 weights before.  Everything else is exact in 16 bits; sums are fp32.
//
// What a non-finite operand does to the products' cells and children outside a window is mended behind them
// (wm16_exact.hpp): the masked logits are selected, so that the maximum and 1 / sum are the child's own
// whatever lies around; D, the gradients of a block's queries and of its cells are formed again where
// one of them is not finite.
//
// Measured (B=16, C=256, d=64, 100x168, bf16): pixel kernel 295 us, cell kernel 429 us, a training step
// 970 us against 1211 for the chain over K * K tensors (similarity and its softmax backward 274 us,
// grad_q 92, grad_value and grad_key by vector fmas 544, the weights 86).  Odd W: key and value are copied into rows
// of an even number of cells first (direct loads begin on dwords); B=16, 100x167 1593 -> 1193 us for a step (1166 with
// pairs), of which the copies 98 and the cell kernel 526 (hi-res pieces across cache lines, results moved by half a
// dword; of pairs 503, and 560 with a 2-byte store per result); B=4, C=512, d=32, 97x165 911 -> 543; B=8, d=64, 51x83
// 409 -> 242, with 100 for a forward pass that aggregates with fp32 weights (175 with pairs and the one-launch forward).
// The third operand costs the cell kernel 8 registers spilled in bf16, 16 in fp16.
#include "wm16_exact.hpp"

namespace sapa {

namespace bwm16 {

using namespace wm;

constexpr int CHK = 16;            // channels per staged chunk
constexpr int WROWS = 8;           // window rows = child rows of a block row

template <typename T> struct Args {
    const T *q, *key, *value, *grad_out;
    float *stats;
    T *grad_q, *grad_key, *grad_value;
    // the key and value that the products read, in rows of `low_w` (even) cells: the tensors, or copies with a
    // cell more per row where W is odd -- direct loads begin on dwords
    const T *key_rows, *value_rows;
    int B, d, C, H, W, low_w, tiles_x, tiles_y, ns, nblocks, per_xcd;
};

// Rows of w 16-bit cells -> rows of w + 1 (w odd), the added cell 0; two tensors in one launch.  A thread moves 4
// dwords of a row, from the dword before where the row begins in the middle of one (B=16, d=64, C=256,
// 100x167: 98 us = 3.5 TB/s; 131 with a thread per dword).
__global__ __launch_bounds__(256) void
pad_rows_kernel(const unsigned short *__restrict__ a, const unsigned short *__restrict__ b, u32 *__restrict__ pa,
                u32 *__restrict__ pb, long rows_a, long rows_b, int w) {
    const unsigned short *const src = blockIdx.y ? b : a;
    u32 *const dst = blockIdx.y ? pb : pa;
    const u32 per_row = (u32)(w + 1) / 2, pieces = (per_row + 3) / 4;
    const long n = (blockIdx.y ? rows_b : rows_a) * pieces;
    for (long i = blockIdx.x * 256L + threadIdx.x; i < n; i += gridDim.x * 256L) {
        const long row = i < (1L << 31) ? (long)((u32)i / pieces) : i / pieces;
        const u32 x = 4 * (u32)(i - row * pieces);           // first dword
        const unsigned short *const p = src + row * w + 2 * x;
        u32 *const o = dst + row * per_row + x;
        const bool half = (uintptr_t)p % 4 != 0;
        // (a tensor may begin in the middle of a dword: nothing in front of it is read)
        if (x + 4 < per_row && !(half && i == 0)) {
            // (cells 2 x .. 2 x + 7 and one more are the row's own)
            typedef u32x4 __attribute__((aligned(4))) u32x4_a4;
            const u32 *const q = (const u32 *)(p - half);
            const u32x4 v = *(const u32x4_a4 *)q;
            const u32 next = half ? q[4] : 0u;
            *(u32x4_a4 *)o = half ? u32x4{__builtin_amdgcn_alignbit(v[1], v[0], 16), __builtin_amdgcn_alignbit(v[2], v[1], 16),
                                          __builtin_amdgcn_alignbit(v[3], v[2], 16), __builtin_amdgcn_alignbit(next, v[3], 16)}
                                  : v;
        } else {
            for (u32 k = 0; k < 4 && k < per_row - x; ++k) o[k] = p[2 * k] | (2 * (x + k) + 1 < (u32)w ? (u32)p[2 * k + 1] << 16 : 0u);
        }
    }
}

// Operands that hold A and E: two, with odd rows three, i.e. all 24 bits of them
constexpr int pieces_of(bool odd) { return odd ? 3 : 2; }

// position of the 16-byte piece of row r, channel ch in the swizzled tile of bwd_pixel_kernel
__device__ __forceinline__ int swz(int ch, int r) { return ((ch & 7) << 1) | ((r + (ch >> 3)) & 1); }

// the slow way of bwd_pixel_kernel for the blocks of its tile that are named
template <typename T, int NT>
__device__ __attribute__((noinline)) void children_again(Again again) {
    settled();
    const Args<T> a = again.arguments<Args<T>>();
    const int at = (int)(again.workgroup() % 8) * a.per_xcd + (int)(again.workgroup() / 8), n = at / (a.tiles_x * a.tiles_y);
    const int cy = 8 * (at / a.tiles_x % a.tiles_y), cx = 8 * a.ns * (at % a.tiles_x);
    const long lpix = (long)a.H * a.W;
    for (u32 b = 0, blocks = again.of_blocks(); blocks >> b; ++b)
        if (blocks >> b & 1)
            exact_grad_q<T, NT>(again.floats(), plane_of<false>(a.q, n, a.d, 4 * lpix), plane_of<false>(a.key, n, a.d, lpix),
                                plane_of<false>(a.value, n, a.C, lpix), plane_of<false>(a.grad_out, n, a.C, 4 * lpix),
                                plane_of<false>(a.grad_q, n, a.d, 4 * lpix), a.stats + (2L * a.B + n) * 4 * lpix, a.d, a.C, a.H, a.W,
                                cy, cx + 8 * (int)b);
}

// ---- per-child gradients ----
// A workgroup of 2 NSW waves owns up to NSW blocks side by side; waves t and t + NSW share block t,
// the upper / lower 32 of its children each (with all 64 a wave would hold 128 accumulators and
// weights, and half as many waves would be resident).  Chunks of 16 channels: key + q (S), value +
// grad_out (G), key again (grad_q), in a ring of three buffers, the next two in flight.
// ODD: an odd W
template <typename T, int NSW, bool STREAM, bool ODD>
__global__ __launch_bounds__(128 * NSW) void
bwd_pixel_kernel(const Args<T> args) {
    const T *__restrict__ const q = args.q, *__restrict__ const key = args.key_rows, *__restrict__ const value = args.value_rows,
            *__restrict__ const grad_out = args.grad_out;
    T *__restrict__ const grad_q = args.grad_q;
    float *__restrict__ const stats = args.stats;
    const int B = args.B, d = args.d, C = args.C, H = args.H, W = args.W, tiles_x = args.tiles_x, tiles_y = args.tiles_y,
              ns = args.ns, nblocks = args.nblocks, per_xcd = args.per_xcd;
    constexpr int NT = 128 * NSW;
    constexpr bool SCALED = __is_same(T, f16_t);             // E is brought into the type's range (Fit)
    constexpr int NP = pieces_of(ODD);
    constexpr int NBUF = 3;
    constexpr int LROW = (4 * NSW + 4 + 7) / 8 * 4;          // dwords per staged window row: whole pieces of 8 cells
    constexpr int LOWBUF = WROWS * CHK * LROW;               // dwords per low-res buffer
    constexpr int NLP = LOWBUF / 4;                          // 16-byte pieces per low-res buffer
    constexpr int HIROW = 8 * NSW / 2;                       // dwords per hi-res tile row
    constexpr int HICH = WROWS * HIROW;                      // dwords per channel of the tile
    constexpr int HIBUF = CHK * HICH;                        // dwords per hi-res buffer
    constexpr int NPC = NSW;                                 // 16-byte pieces per tile row
    static_assert(HIBUF == 4 * NT && NLP % 64 == 0 && NLP <= NT, "one direct load per thread and buffer");

    __shared__ __attribute__((aligned(16))) u32 lds[NBUF * (LOWBUF + HIBUF) + 4];
    u32 *const lowbuf = lds, *const hibuf = lds + NBUF * LOWBUF, *const non_finite = lds + NBUF * (LOWBUF + HIBUF);
    const u32 low_at = lds_address((const __attribute__((address_space(3))) u32 *)lds), hi_base = low_at + NBUF * LOWBUF * 4;

    const int logical = (int)(blockIdx.x % 8) * per_xcd + (int)(blockIdx.x / 8);
    if (logical >= nblocks) return;
    const int tx = logical % tiles_x, ty = (logical / tiles_x) % tiles_y, n = logical / (tiles_x * tiles_y);
    const int X0 = tx * 4 * ns, Y0 = ty * 4;                 // first parent of the tile
    const int nsx = (W + 3) / 4;
    const int ns_here = nsx - tx * ns < ns ? nsx - tx * ns : ns;

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int t = wave % NSW, half = wave / NSW;              // block of the tile, half of its children
    const int g = lane >> 4, i16 = lane & 15;
    const long lpix = (long)H * W;
    const int low_w = ODD ? args.low_w : W;
    const long lowpix = (long)H * low_w;
    const u32 lplane = (u32)(lowpix * sizeof(T)), hplane = (u32)(4 * lpix * sizeof(T));

    // direct-load offsets inside one image, without the chunk's first channel; the low-res pieces as
    // in sapa_b_wmat16.hip (a piece that runs over an end of its row brings the neighbouring row's
    // cells; the one that starts before the image reads as zeros and is patched)
    u32 off_low, off_hi;
    int short_piece;           // W % 4 != 0: dwords of a row's last 16-byte piece (the rest is the next row's), else 0
    int patch_slot = -1;
    {
        const int slot = tid, rc = slot / (LROW / 4), pc = slot % (LROW / 4);
        const int r = rc / CHK, ch = rc % CHK;
        const int y = Y0 - 2 + r, x = X0 - 2 + 8 * pc;
        const bool ok = slot < NLP && 8 * pc < 4 * ns_here + 4 && y >= 0 && y < H && x < W;
        off_low = ok ? (u32)(ch * lowpix + (long)y * low_w + x) * (u32)sizeof(T) : OUTSIDE;
        if (ok && x < 0 && y == 0 && ch == 0) patch_slot = slot;
    }
    {
        const int slot = tid, ch = slot / (WROWS * NPC), r = (slot / NPC) % WROWS;
        const int pc = (slot % NPC) ^ (swz(ch, r) & (NPC - 1));
        const int cy = 2 * Y0 + r, cx = 2 * X0 + 8 * pc;
        const bool ok = pc < ns_here && cy < 2 * H && cx < 2 * W;
        off_hi = ok ? (u32)(ch * 4 * lpix + (long)cy * 2 * W + cx) * (u32)sizeof(T) : OUTSIDE;
        short_piece = ok && cx + 8 > 2 * W ? W - cx / 2 : 0;
    }

    const int nKc = (d + CHK - 1) / CHK, nVc = (C + CHK - 1) / CHK;
    const int ntot = nKc + nVc + (grad_q ? nKc : 0);
    const u32x4 rq = dma_rsrc(q + (long)n * d * 4 * lpix, d * hplane);
    const u32x4 rk = dma_rsrc(key + (long)n * d * lowpix, d * lplane);
    const u32x4 rv = dma_rsrc(value + (long)n * C * lowpix, C * lplane);
    const u32x4 rg = dma_rsrc(grad_out + (long)n * C * 4 * lpix, C * hplane);

    // phase of chunk j: 0 = key + q, 1 = value + grad_out, 2 = key
    auto loads_of = [&](int j) __attribute__((always_inline)) {
        return j < ntot ? (wave * 64 < NLP ? 1 : 0) + (j < nKc + nVc ? 1 : 0) : 0;
    };
    auto stage = [&](int j) __attribute__((always_inline)) {
        if (j >= ntot) return;
        const bool is_val = j >= nKc && j < nKc + nVc;
        const u32 c0 = (u32)((j < nKc ? j : is_val ? j - nKc : j - nKc - nVc) * CHK);
        const int buf = j % NBUF;
        if (wave * 64 < NLP) load_lds(is_val ? rv : rk, low_at + (buf * LOWBUF + wave * 256) * 4, off_low + c0 * lplane);
        if (j < nKc + nVc) load_lds<STREAM>(is_val ? rg : rq, hi_base + (buf * HIBUF + wave * 256) * 4, off_hi + c0 * hplane);
    };
    // loads of this wave that may be outstanding when chunk j + 1 is wanted: those of the chunks after it
    auto later = [&](int j) __attribute__((always_inline)) {
        int k = 0;
#pragma unroll
        for (int i = 1; i < NBUF; ++i) k += loads_of(j + i);
        return k;
    };
    // the 6 cells of the piece that has no address (first channel of a tensor, tile at the image's
    // upper left corner)
    auto patch_low = [&](int j) __attribute__((always_inline)) {
        if (tx == 0 && ty == 0 && patch_slot >= 0 && (j == 0 || j == nKc || j == nKc + nVc) && j < ntot) {
            const u32 *src = (const u32 *)(j == nKc ? value + (long)n * C * lowpix : key + (long)n * d * lowpix);
            u32 *dst = lowbuf + (j % NBUF) * LOWBUF + patch_slot * 4;
#pragma unroll
            for (int k = 1; k < 4; ++k) dst[k] = src[k - 1];
        }
    };

    const bool row_tail = (W & 3) != 0 && X0 + 4 * ns_here > W;      // workgroup-uniform
    const bool active = t < ns_here;

    if (tid == 0) *non_finite = 0;          // blocks of the tile with a non-finite result
    stage(0);
    stage(1);
    for (int j = 2; j < NBUF; ++j) stage(j);
    wait_all_but(later(0));
    patch_low(0);
    lds_barrier();

    // Sim[cell][child], 4 x 2 accumulator blocks of 16 x 16: block (mb, nb), lane (g, i16), element v:
    // cell (row 2 mb + g / 2, column 4 (g % 2) + v) of the window, child (row 2 (2 half + nb) + i16 / 8,
    // column i16 % 8) of the block's 8 x 8 children
    auto zero = [](f32x4 (&acc)[4][2]) __attribute__((always_inline)) {
#pragma unroll
        for (int mb = 0; mb < 4; ++mb) acc[mb][0] = acc[mb][1] = f32x4{0.f, 0.f, 0.f, 0.f};
    };
    const int tch = 4 * g + (i16 >> 2), trow = (i16 & 3) >> 1, tcol = i16 & 1;
    auto similarity = [&](int j, f32x4 (&acc)[4][2]) __attribute__((always_inline)) {
        const u32 *kb = lowbuf + (j % NBUF) * LOWBUF, *qb = hibuf + (j % NBUF) * HIBUF;
        u32x2 a[4], b[2];
#pragma unroll
        for (int mb = 0; mb < 4; ++mb)
            a[mb] = read_tr(kb + ((2 * mb + trow) * CHK + tch) * LROW + 2 * t + 2 * tcol);
#pragma unroll
        for (int nb = 0; nb < 2; ++nb) {
            const int r = 2 * (2 * half + nb) + trow;
            b[nb] = read_tr(qb + tch * HICH + r * HIROW + ((t ^ (swz(tch, r) & (NPC - 1))) << 2) + 2 * tcol);
        }
#pragma unroll
        for (int mb = 0; mb < 4; ++mb)
#pragma unroll
            for (int nb = 0; nb < 2; ++nb) acc[mb][nb] = Mma<T>::k16(a[mb], b[nb], acc[mb][nb]);
    };
    // chunk j is done with: chunk j + 1 complete for everyone, chunk j + 3 requested
    auto next = [&](int j) __attribute__((always_inline)) {
        wait_all_but(later(j + 1) - loads_of(j + NBUF));
        patch_low(j + 1);
        lds_barrier();
        stage(j + NBUF);
    };

    f32x4 acc[4][2];
    zero(acc);
    for (int j = 0; j < nKc; ++j) {
        if (active) similarity(j, acc);
        next(j);
    }

    // ---- softmax over each child's 5 x 5 cells ----
    // element v of every block is window column 4 (g % 2) + v; columns outside the image hold the
    // neighbouring row's cells: their logit is 0 and their weight may as well be 0
    bool cell_outside[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) cell_outside[v] = (u32)(X0 + 4 * t - 2 + 4 * (g & 1) + v) >= (u32)W;
    const bool at_row_end = X0 + 4 * t - 2 < 0 || X0 + 4 * t + 5 >= W;      // wave-uniform
    auto clear_outside = [&](f32x4 (&x)[4][2]) __attribute__((always_inline)) {
        if (at_row_end) {
#pragma unroll
            for (int mb = 0; mb < 4; ++mb)
#pragma unroll
                for (int nb = 0; nb < 2; ++nb)
#pragma unroll
                    for (int v = 0; v < 4; ++v)
                        if (cell_outside[v]) x[mb][nb][v] = 0.f;
        }
    };
    f32x4 p[4][2];
    float mlog[2], inv[2];
    // whether element v of block (mb, nb) lies in its child's window: parent row 2 half + nb and column px take
    // window rows and columns from theirs on, 5 of each
    const int px = (i16 & 7) >> 1;
    auto inside = [&](int mb, int nb, int v) __attribute__((always_inline)) {
        return ((u32)(4 * (g & 1) + v - px) <= 4u) & ((u32)(2 * mb + (g >> 1) - (2 * half + nb)) <= 4u);
    };
    if (active) {
        clear_outside(acc);
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
        clear_outside(p);
    }

    // ---- gradient of the weights ----
    zero(acc);
    for (int j = nKc; j < nKc + nVc; ++j) {
        if (active) similarity(j, acc);
        next(j);
    }

    // ---- gradient of the logits; what the cell kernel needs to form it again ----
    u32x4 we[2][2][NP];
    NonFinite seen;
    float down[2][4];           // f16: what the results of child 4 g + v of block nb are multiplied by
    if (active) {
        clear_outside(acc);
#pragma unroll
        for (int nb = 0; nb < 2; ++nb) {
            float dsum = 0.f;
#pragma unroll
            for (int mb = 0; mb < 4; ++mb)
#pragma unroll
                for (int v = 0; v < 4; ++v) dsum = __builtin_fmaf(p[mb][nb][v], acc[mb][nb][v], dsum);
            dsum += __shfl_xor(dsum, 16);
            dsum += __shfl_xor(dsum, 32);
            seen.see(dsum);
            const int cy = 2 * Y0 + 2 * (2 * half + nb) + (i16 >> 3), cx = 2 * X0 + 8 * t + (i16 & 7);
            if (g < 3 && cy < 2 * H && cx < 2 * W) {
                // planes [3][B, 2H, 2W]: maximum (times log2 e), 1 / sum, D; lanes g = 0, 1, 2 one each
                const long plane = (long)B * 4 * lpix;
                stats[g * plane + (long)n * 4 * lpix + (long)cy * 2 * W + cx] = g == 0 ? mlog[nb] : g == 1 ? inv[nb] : dsum;
            }
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
#pragma unroll
                for (int v = 0; v < 4; ++v) down[nb][v] = __shfl(f.down, 4 * g + v);
#pragma unroll
                for (int k = 0; k < 16; ++k) e[k / 8][k % 8] *= f.up;
            }
#pragma unroll
            for (int s = 0; s < 2; ++s) split8<T>(e[s], we[nb][s]);
        }
    }

    // ---- grad_q[child][channel], per chunk of 16 channels, through the hi-res tile ----
    const __amdgpu_buffer_rsrc_t ro = __builtin_amdgcn_make_buffer_rsrc(
        (void *)(grad_q + (long)n * d * 4 * lpix), 0, (int)(d * hplane), 0x00020000);
    for (int j = nKc + nVc; j < ntot; ++j) {
        const u32 c0 = (u32)((j - nKc - nVc) * CHK);
        u32 *ob = hibuf + (j % NBUF) * HIBUF;                    // no loads into this ring any more
        if (active) {
            const u32 *vb = lowbuf + (j % NBUF) * LOWBUF;
            u32x4 b[2];
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                const u32 *pp = vb + ((4 * s + (g >> 1)) * CHK + i16) * LROW + 2 * t + 2 * (g & 1);
                const u32x2 lo = *(const u32x2 *)pp, hi = *(const u32x2 *)(pp + 2 * CHK * LROW);
                b[s] = u32x4{lo[0], lo[1], hi[0], hi[1]};
            }
#pragma unroll
            for (int nb = 0; nb < 2; ++nb) {
                f32x4 o = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int s = 0; s < 2; ++s)
#pragma unroll
                    for (int i = 0; i < NP; ++i) o = Mma<T>::k32(we[nb][s][i], b[s], o);
                // (a key that is not finite makes its channel's results so for every child of the block)
                if (nb == 0) seen.see(o[0]);
                if (SCALED) {
#pragma unroll
                    for (int v = 0; v < 4; ++v) o[v] *= down[nb][v];
                }
                // element v: child (row 2 (2 half + nb) + g / 2, column 4 (g % 2) + v), channel c0 + i16
                const int r = 2 * (2 * half + nb) + (g >> 1);
                *(u32x2 *)(ob + i16 * HICH + r * HIROW + ((t ^ (swz(i16, r) & (NPC - 1))) << 2) + 2 * (g & 1)) =
                    u32x2{pack2<T>(o[0], o[1]), pack2<T>(o[2], o[3])};
            }
        }
        // chunk j + 1 was requested before the last store and chunk j + 2
        wait_all_but(0);
        patch_low(j + 1);
        lds_barrier();
        const u32x4 o = *(const u32x4 *)(ob + tid * 4);
        u32 off = off_hi + c0 * hplane;
        if (row_tail && short_piece) {
            if (ODD) {
#pragma unroll
                for (int k = 0; k < 3; ++k)
                    if (k < short_piece) __builtin_amdgcn_raw_buffer_store_b32(o[k], ro, off + 4 * k, 0, 0);
            } else {
                __builtin_amdgcn_raw_buffer_store_b64(u32x2{o[0], o[1]}, ro, off, 0, 0);
            }
            off = OUTSIDE;
        }
        __builtin_amdgcn_raw_buffer_store_b128(o, ro, off, 0, STREAM ? 2 : 0);
        stage(j + NBUF);
    }

    // ---- blocks with a non-finite result: again, term by term ----
    if (seen.any()) atomicOr(non_finite, 1u << t);
    lds_barrier();
    const u32 blocks = __builtin_amdgcn_readfirstlane(*non_finite);
    if (__builtin_expect(blocks != 0, 0)) children_again<T, NT>(Again(lds, blocks));
}

// ---- per-cell gradients ----
// A workgroup owns TBX blocks of 4 x 4 cells side by side; blocks start 2 cells left of / above a
// multiple of 4, so that the 8 x 8 parents a block gathers over are 2 x 2 whole parent blocks
// (quadrants): the workgroup stages 2 x (TBX + 1) parent blocks = 16 hi-res rows of 144 bytes per
// channel.  Two waves share a block, one per row of quadrants; their halves of the sums meet in LDS
// on the way out.  Wide and flat, because what bounds the kernel is the number of cache-line requests
// the hi-res rows take (2 x 2 blocks per workgroup: 2.3 times the requests, 645 us; results stored
// 8 bytes per lane straight from the registers: 200 us of that).
// LDS of a chunk of 16 channels, three in a ring: hi-res tile [16][16 rows][9 pieces of 16 bytes], rows
// XOR-permuted and pieces rotated by the channel so that the transposing reads and the 8-byte reads
// below spread over all banks; cells [16][4 rows][4 pieces].
constexpr int TBX = 8;                     // cell blocks per workgroup
constexpr int CNT = 128 * TBX;             // threads
constexpr int CBUF = 3;
constexpr int CPC = TBX + 1;               // pieces per hi-res row
constexpr int CROW = 4 * CPC;              // dwords per hi-res row
constexpr int CHICH = 16 * CROW;           // dwords per channel of the hi-res tile
constexpr int CHI = CHK * CHICH;           // dwords per hi-res buffer
constexpr int CLROW = 2 * TBX;             // dwords per cell row
constexpr int CLOW = CHK * 4 * CLROW;      // dwords per cell buffer
constexpr int CNH = CHI / 4 / CNT;         // whole rounds of hi-res direct loads
constexpr int COUT = CHK * 4 * 4 * TBX;    // floats of one half of a chunk's results
constexpr int CNL = CLOW / 256;            // waves that a round over a chunk's cells takes
static_assert(CHI / 4 == CNH * CNT + 256 && CLOW % 256 == 0, "waves 0 .. 3 load the rest of the tile, waves 4 .. the cells");
constexpr int CSTAT = 5 * 256;             // floats of one stats plane: 16 rows of 8 CPC, in whole loads of 5 waves
static_assert(TBX == 8 && 16 * 8 * CPC <= CSTAT && 2 * CSTAT <= 4 * COUT, "stats planes");
static_assert((CBUF * (CHI + CLOW) + CSTAT + 4 * COUT + 4) * 4 <= 160 * 1024, "LDS");

// dword of piece `pc` of hi-res row r, channel ch
__device__ __forceinline__ int hi_at(int ch, int r, int pc) {
    return ch * CHICH + (r ^ (((ch & 3) << 1) | ((ch >> 3) & 1))) * CROW + ((pc + ((ch >> 2) & 1)) % CPC) * 4;
}

// float of the 4 cells `bi` of (channel, cell row) in a half of a chunk's results: rows of 4 TBX floats
// begin on two banks only, so the pieces are XOR-permuted by the channel and every other row by its
// upper bit: the 16 channels of a lane group write to 16 different bank quads (unpermuted, 16 lanes on
// one: B=16, C=256, 100x168 in bf16 460 -> 433 us)
__device__ __forceinline__ int out_at(int ch, int row, int bi) {
    return ((ch * 4 + row) ^ ((ch >> 3) & 1)) * 4 * TBX + 4 * (bi ^ (ch & 7));
}

// the slow way of bwd_cell_kernel for the cell blocks of its tile that are named
template <typename T>
__device__ __attribute__((noinline)) void cells_again(Again again) {
    settled();
    const Args<T> a = again.arguments<Args<T>>();
    const int at = (int)(again.workgroup() % 8) * a.per_xcd + (int)(again.workgroup() / 8), n = at / (a.tiles_x * a.tiles_y);
    const int cy = 4 * (at / a.tiles_x % a.tiles_y) - 2, cx = 4 * TBX * (at % a.tiles_x) - 2;
    const long lpix = (long)a.H * a.W;
    for (u32 b = 0, blocks = again.of_blocks(); blocks >> b; ++b)
        if (blocks >> b & 1)
            exact_grad_cells<T, CNT>(again.floats(), plane_of<false>(a.q, n, a.d, 4 * lpix), plane_of<false>(a.key, n, a.d, lpix),
                                     plane_of<false>(a.value, n, a.C, lpix), plane_of<false>(a.grad_out, n, a.C, 4 * lpix),
                                     a.stats + n * 4 * lpix, (long)a.B * 4 * lpix, plane_of<false>(a.grad_key, n, a.d, lpix),
                                     plane_of<false>(a.grad_value, n, a.C, lpix), a.d, a.C, a.H, a.W, cy, cx + 4 * (int)b);
}

// ODD: an odd W
template <typename T, bool ODD>
__global__ __launch_bounds__(CNT) void
bwd_cell_kernel(const Args<T> args) {
    const T *__restrict__ const q = args.q, *__restrict__ const key = args.key_rows, *__restrict__ const value = args.value_rows,
            *__restrict__ const grad_out = args.grad_out;
    T *__restrict__ const grad_key = args.grad_key, *__restrict__ const grad_value = args.grad_value;
    const float *__restrict__ const stats = args.stats;
    const int B = args.B, d = args.d, C = args.C, H = args.H, W = args.W, tiles_x = args.tiles_x, tiles_y = args.tiles_y,
              nblocks = args.nblocks, per_xcd = args.per_xcd;
    constexpr bool SCALED = __is_same(T, f16_t);             // A and E are brought into the type's range (Fit)
    constexpr int NP = pieces_of(ODD);
    __shared__ __attribute__((aligned(16))) u32 lds[CBUF * (CHI + CLOW) + CSTAT + 4 * COUT + 4];
    u32 *const hibuf = lds, *const lowbuf = lds + CBUF * CHI;
    const u32 hi_base = lds_address((const __attribute__((address_space(3))) u32 *)lds), low_at = hi_base + CBUF * CHI * 4;
    // D in front, the other stats planes over the results [chunk % 2][half][16][4 rows][4 TBX cells]
    float *const statbuf = (float *)(lowbuf + CBUF * CLOW), *const outbuf = statbuf + CSTAT;
    const u32 stat_at = low_at + CBUF * CLOW * 4;
    u32 *const non_finite = (u32 *)(outbuf + 4 * COUT);       // cell blocks with a non-finite result

    const int logical = (int)(blockIdx.x % 8) * per_xcd + (int)(blockIdx.x / 8);
    if (logical >= nblocks) return;
    const int tx = logical % tiles_x, J = (logical / tiles_x) % tiles_y, n = logical / (tiles_x * tiles_y);
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g = lane >> 4, i16 = lane & 15;
    const int bi = wave % TBX, qy = wave / TBX;               // this wave's cell block, its row of quadrants
    const int I0 = tx * TBX;
    const bool active = 4 * (I0 + bi) - 2 < W;
    const long lpix = (long)H * W;
    const int low_w = ODD ? args.low_w : W;
    const long lowpix = (long)H * low_w;
    const u32 lplane = (u32)(lowpix * sizeof(T)), hplane = (u32)(4 * lpix * sizeof(T));

    // direct-load offsets inside one image, without the chunk's first channel
    u32 off_hi[CNH + 1];
#pragma unroll
    for (int i = 0; i < CNH + 1; ++i) {
        const int slot = i * CNT + tid, ch = slot / (16 * CPC) % CHK;
        const int r = (slot / CPC) % 16 ^ (((ch & 3) << 1) | ((ch >> 3) & 1)), pc = (slot % CPC + CPC - ((ch >> 2) & 1)) % CPC;
        const int cy = 8 * (J - 1) + r, cx = 8 * (I0 - 1 + pc);
        const bool ok = ((u32)cy < (u32)(2 * H)) & ((u32)cx < (u32)(2 * W));
        off_hi[i] = ok ? (u32)(ch * 4 * lpix + (long)cy * 2 * W + cx) * (u32)sizeof(T) : OUTSIDE;
    }
    // cells (waves 4 .. 7) and results (waves 0 .. 3): piece [channel][row][x] of 8 cells.  A piece that
    // runs over an end of its row brings / would overwrite the neighbouring row's cells: read it is
    // harmless (they belong to columns that are not stored), results are stored dword by dword there.
    // The piece 2 cells before the image's first has no address: zeros, and patched.
    const int lslot = tid & (64 * CNL - 1), lch = lslot / (2 * TBX), ly = 4 * J - 2 + (lslot / (TBX / 2)) % 4, lx = 4 * I0 - 2 + 8 * (lslot % (TBX / 2));
    const bool lrow = ((u32)ly < (u32)H) & (lx < W);
    const u32 off_low = lrow ? (u32)(lch * lowpix + (long)ly * low_w + lx) * (u32)sizeof(T) : OUTSIDE;
    const bool patch = lx < 0 && ly == 0 && lch == 0 && wave >= 4 && wave < 4 + CNL;
    const bool ragged = I0 == 0 || 4 * I0 - 2 + 4 * TBX > W;  // workgroup-uniform

    const int nKc = (d + CHK - 1) / CHK, nVc = (C + CHK - 1) / CHK;
    const int ntot = nKc + nVc + (grad_key ? nKc : 0);
    const u32x4 rq = dma_rsrc(q + (long)n * d * 4 * lpix, d * hplane);
    const u32x4 rk = dma_rsrc(key + (long)n * d * lowpix, d * lplane);
    const u32x4 rv = dma_rsrc(value + (long)n * C * lowpix, C * lplane);
    const u32x4 rg = dma_rsrc(grad_out + (long)n * C * 4 * lpix, C * hplane);

    // chunk j: q + key (S), grad_out + value (G and grad_value), q again (grad_key)
    auto loads_of = [&](int j) __attribute__((always_inline)) {
        return j < ntot ? CNH + (wave < 4 || (wave < 4 + CNL && j < nKc + nVc) ? 1 : 0) : 0;
    };
    auto stage = [&](int j) __attribute__((always_inline)) {
        if (j >= ntot) return;
        const bool is_val = j >= nKc && j < nKc + nVc;
        const u32 c0 = (u32)((j < nKc ? j : is_val ? j - nKc : j - nKc - nVc) * CHK);
        const u32 hb = hi_base + (j % CBUF * CHI + wave * 256) * 4;
        const u32x4 rh = is_val ? rg : rq;
#pragma unroll
        for (int i = 0; i < CNH; ++i) load_lds(rh, hb + i * CNT * 16, off_hi[i] + c0 * hplane);
        if (wave < 4) load_lds(rh, hb + CNH * CNT * 16, off_hi[CNH] + c0 * hplane);
        else if (wave < 4 + CNL && j < nKc + nVc)
            load_lds(is_val ? rv : rk, low_at + (j % CBUF * CLOW + (wave - 4) * 256) * 4, off_low + c0 * lplane);
    };

    // quadrant (qy, qx): parent block (1 - qy, bi + 1 - qx) of the staged 2 x 9.
    // A similarity block (qx, nb) has the 16 children of parent row nb (hi-res rows 2 nb, 2 nb + 1) as
    // rows and the wave's 16 cells as columns: lane (g, cell i16), element v: child (row 2 nb + g / 2,
    // column 4 (g % 2) + v).  (The row permutation turns nb into nb ^ (channel % 4): a lane base per nb.)
    const int tch = 4 * g + (i16 >> 2), trow = (i16 & 3) >> 1, tcol = i16 & 1;
    int sim_at[2][4], gat_at[2][4];
#pragma unroll
    for (int qx = 0; qx < 2; ++qx)
#pragma unroll
        for (int nb = 0; nb < 4; ++nb) {
            sim_at[qx][nb] = hi_at(tch, 8 * (1 - qy) + 2 * nb + trow, bi + 1 - qx) + 2 * tcol;
            gat_at[qx][nb] = hi_at(i16, 8 * (1 - qy) + 2 * nb + (g >> 1), bi + 1 - qx) + 2 * (g & 1);
        }
    auto similarity = [&](int j, f32x4 (&acc)[2][4]) __attribute__((always_inline)) {
        const u32 *hb = hibuf + j % CBUF * CHI, *lb = lowbuf + j % CBUF * CLOW;
        const u32x2 b = read_tr(lb + (tch * 4 + (i16 & 3)) * CLROW + 2 * bi);
#pragma unroll
        for (int qx = 0; qx < 2; ++qx)
#pragma unroll
            for (int nb = 0; nb < 4; ++nb) acc[qx][nb] = Mma<T>::k16(read_tr(hb + sim_at[qx][nb]), b, acc[qx][nb]);
    };
    // the gathered sum over this wave's 128 children of 16 channels: reduction step (qx, s) covers parent
    // rows 2 s and 2 s + 1 of the quadrant, in the order the weights are held in; element v of the
    // result: cell (row g, column v), channel i16
    u32x4 wp[2][2][NP];
    Fit f = {1.f, 1.f};         // f16: the factors of this lane's cell, the results' of cells (g, v)
    float down[4];
    auto hold = [&](float (&w)[2][2][8]) __attribute__((always_inline)) {
        if (SCALED) {
            float m = 0.f;
#pragma unroll
            for (int k = 0; k < 32; ++k) m = fmaxf(m, __builtin_fabsf(w[k / 16][k / 8 % 2][k % 8]));
            f = fit<T>(over_groups(m));
#pragma unroll
            for (int v = 0; v < 4; ++v) down[v] = __shfl(f.down, 4 * g + v);
#pragma unroll
            for (int k = 0; k < 32; ++k) w[k / 16][k / 8 % 2][k % 8] *= f.up;
        }
#pragma unroll
        for (int qx = 0; qx < 2; ++qx)
#pragma unroll
            for (int s = 0; s < 2; ++s) split8<T>(w[qx][s], wp[qx][s]);
    };
    NonFinite seen;
    auto gather = [&](int j) __attribute__((always_inline)) {
        const u32 *hb = hibuf + j % CBUF * CHI;
        f32x4 o = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int qx = 0; qx < 2; ++qx)
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                const u32x2 lo = *(const u32x2 *)(hb + gat_at[qx][2 * s]), hi = *(const u32x2 *)(hb + gat_at[qx][2 * s + 1]);
                const u32x4 b = u32x4{lo[0], lo[1], hi[0], hi[1]};
#pragma unroll
                for (int i = 0; i < NP; ++i) o = Mma<T>::k32(wp[qx][s][i], b, o);
            }
        // (what is not finite in a child makes its channel's results so for every cell of the block)
        seen.see(o[0]);
        if (SCALED) {
#pragma unroll
            for (int v = 0; v < 4; ++v) o[v] *= down[v];
        }
        *(f32x4 *)(outbuf + (2 * (j & 1) + qy) * COUT + out_at(i16, g, bi)) = o;
    };
    // the chunk's results, complete after the barrier
    const int out0 = out_at(lch, (lslot / (TBX / 2)) % 4, 2 * (lslot % (TBX / 2))), out1 = out_at(lch, (lslot / (TBX / 2)) % 4, 2 * (lslot % (TBX / 2)) + 1);
    auto store = [&](int j, __amdgpu_buffer_rsrc_t ro, u32 c0) __attribute__((always_inline)) {
        if (wave >= CNL) return;
        const float *p0 = outbuf + 2 * (j & 1) * COUT + out0, *p1 = outbuf + 2 * (j & 1) * COUT + out1;
        const f32x4 a = *(const f32x4 *)p0 + *(const f32x4 *)(p0 + COUT), b = *(const f32x4 *)p1 + *(const f32x4 *)(p1 + COUT);
        const u32x4 o = {pack2<T>(a[0], a[1]), pack2<T>(a[2], a[3]), pack2<T>(b[0], b[1]), pack2<T>(b[2], b[3])};
        const u32 off = (u32)((c0 + (u32)lch) * (u32)lpix + ly * W + lx) * (u32)sizeof(T);
        if (ODD) {
            // A row that begins in the middle of a dword takes its pieces half a dword to the left: the
            // last cell of the piece before (the lane before's), then this one's first seven; the first cells
            // of the tile's row and the last one before a piece that is not whole by themselves.  Pieces
            // over an end of the image's row: cell by cell.
            const int pc = lslot % (TBX / 2);
            const u32 before = (u32)__shfl_up((int)o[3], 1);
            const bool here = lrow & (lx >= 0) & (lx + 8 <= W), next_whole = (pc < TBX / 2 - 1) & (lx + 16 <= W);
            const bool whole = here & ((pc > 0) | next_whole), half = ((((c0 + (u32)lch) & 1) * (u32)(lpix & 1) + (u32)(ly & 1)) & 1) != 0;
            const u32x4 left = {__builtin_amdgcn_alignbit(o[0], before, 16), __builtin_amdgcn_alignbit(o[1], o[0], 16),
                                __builtin_amdgcn_alignbit(o[2], o[1], 16), __builtin_amdgcn_alignbit(o[3], o[2], 16)};
            const bool first = half & (pc == 0), last = half & !next_whole;
            __builtin_amdgcn_raw_buffer_store_b128(half ? left : o, ro, whole & !first ? half ? off - 2 : off : OUTSIDE, 0, 0);
            __builtin_amdgcn_raw_buffer_store_b96(u32x3{left[1], left[2], left[3]}, ro, whole & first ? off + 2 : OUTSIDE, 0, 0);
            __builtin_amdgcn_raw_buffer_store_b16((unsigned short)(first ? o[0] : o[3] >> 16), ro,
                                                  whole & first ? off : whole & last ? off + 14 : OUTSIDE, 0, 0);
            if (ragged) {
#pragma unroll
                for (int k = 0; k < 8; ++k)
                    __builtin_amdgcn_raw_buffer_store_b16((unsigned short)(o[k / 2] >> (16 * (k & 1))), ro,
                                                          lrow & !whole & ((u32)(lx + k) < (u32)W) ? off + 2 * k : OUTSIDE, 0, 0);
            }
        } else if (!ragged) {
            __builtin_amdgcn_raw_buffer_store_b128(o, ro, lrow ? off : OUTSIDE, 0, 0);
        } else {
#pragma unroll
            for (int k = 0; k < 4; ++k)
                __builtin_amdgcn_raw_buffer_store_b32(o[k], ro, (lrow & ((u32)(lx + 2 * k) < (u32)W)) ? off + 4 * k : OUTSIDE, 0, 0);
        }
    };
    // chunk j + 1 complete for everyone (outs: how many chunks' results have been stored; those of the last
    // CBUF - 1 chunks and the loads of the chunks after j + 1 were issued behind its loads), chunk
    // j + CBUF requested
    auto next = [&](int j, int outs) __attribute__((always_inline)) {
        if (outs > CBUF - 1) outs = CBUF - 1;
        int after = wave < CNL ? outs * (ODD ? ragged ? 11 : 3 : ragged ? 4 : 1) : 0;
#pragma unroll
        for (int i = 2; i < CBUF; ++i) after += loads_of(j + i);
        // (odd rows store more often than wait_all_but counts, whose every further case costs all its callers:
        // 1 us of 165; to wait for more than is needed is safe)
        if (ODD && after > 11) asm volatile("s_waitcnt vmcnt(11)" ::: "memory");
        else wait_all_but(after);
        if (patch && (j + 1 == 0 || j + 1 == nKc)) {
            const u32 *src = (const u32 *)(j + 1 == 0 ? key + (long)n * d * lowpix : value + (long)n * C * lowpix);
            u32 *dst = lowbuf + (j + 1) % CBUF * CLOW + lslot * 4;
#pragma unroll
            for (int k = 1; k < 4; ++k) dst[k] = src[k - 1];
        }
        lds_barrier();
        stage(j + CBUF);
    };

    // The three stats planes of the staged children, [16 rows][72] each, loaded straight into LDS in
    // front of everything else (fetched into registers between the products they cost a memory latency
    // each, with nothing else to run meanwhile): the wait for chunk 0 covers them, however few chunks
    // there are.  Zeros outside the image.  The first two planes lie where results will go later.
    if (wave < 15) {
        const int k = wave / 5, slot = wave % 5 * 64 + lane, r = slot / (2 * CPC);
        const int cy = 8 * (J - 1) + r, cx = 8 * (I0 - 1) + slot % (2 * CPC) * 4;
        const bool ok = ((u32)cy < (u32)(2 * H)) & ((u32)cx < (u32)(2 * W)) & (r < 16);
        load_lds(dma_rsrc(stats + ((long)((k + 2) % 3) * B + n) * 4 * lpix, (u32)(16 * lpix)), stat_at + (k * CSTAT + wave % 5 * 256) * 4,
                 ok ? (u32)(cy * 2 * W + cx) * 4u : OUTSIDE);
    }
    if (tid == 0) *non_finite = 0;
#pragma unroll
    for (int j = 0; j < CBUF - 1; ++j) stage(j);
    next(-1, 0);

    // this lane's 4 children of block (qx, nb)
    auto child_stats = [&](int k, int qx, int nb) __attribute__((always_inline)) {
        return *(const f32x4 *)(statbuf + k * CSTAT + (8 * (1 - qy) + 2 * nb + (g >> 1)) * 8 * CPC + 8 * (bi + 1 - qx) + 4 * (g & 1));
    };
    const int cr = i16 >> 2, cc = i16 & 3;
    const bool cell_in = (u32)(4 * (I0 + bi) - 2 + cc) < (u32)W;

    f32x4 acc[2][4];
#pragma unroll
    for (int qx = 0; qx < 2; ++qx)
#pragma unroll
        for (int nb = 0; nb < 4; ++nb) acc[qx][nb] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int j = 0; j < nKc; ++j) {
        if (active) similarity(j, acc);
        next(j, 0);
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
                        // (a child or a cell beside the image is one of a neighbouring row's, whose products
                        // no maximum bounds: it must not count, whatever it is)
                        const int px = 2 * (g & 1) + (v >> 1);
                        const bool ok = row_ok & (qx ? cc <= px : cc >= px) & (4 * (I0 + bi - qx) + px < W) & cell_in;
                        const float e = __builtin_amdgcn_exp2f(__builtin_fmaf(acc[qx][nb][v], LOG2E, -mlog[v]));
                        w[qx][s][4 * k + v] = ok ? e * inv[v] : 0.f;
                    }
                }
        hold(w);
    }

    lds_barrier();         // (the results of the first chunk overwrite the stats)

    // ---- G and grad_value ----
#pragma unroll
    for (int qx = 0; qx < 2; ++qx)
#pragma unroll
        for (int nb = 0; nb < 4; ++nb) acc[qx][nb] = f32x4{0.f, 0.f, 0.f, 0.f};
    {
        // (a NULL grad_value: a descriptor of no bytes drops the stores)
        const __amdgpu_buffer_rsrc_t ro = __builtin_amdgcn_make_buffer_rsrc(
            (void *)(grad_value + (long)n * C * lpix), 0, grad_value ? (int)(C * lpix * sizeof(T)) : 0, 0x00020000);
        for (int j = nKc; j < nKc + nVc; ++j) {
            if (active) {
                if (grad_key) similarity(j, acc);
                gather(j);
            }
            next(j, j - nKc);
            store(j, ro, (u32)((j - nKc) * CHK));
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
                            w[qx][s][4 * k + v] = joined<T>(wp[qx][s], 4 * k + v) * f.down * (acc[qx][nb][v] - dsum[v]);
                    }
            hold(w);
        }
        const __amdgpu_buffer_rsrc_t ro = __builtin_amdgcn_make_buffer_rsrc(
            (void *)(grad_key + (long)n * d * lpix), 0, (int)(d * lpix * sizeof(T)), 0x00020000);
        for (int j = nKc + nVc; j < ntot; ++j) {
            if (active) gather(j);
            next(j, j - nKc);
            store(j, ro, (u32)((j - nKc - nVc) * CHK));
        }
    }

    // ---- blocks with a non-finite result: again, term by term ----
    if (seen.any()) atomicOr(non_finite, 1u << bi);
    lds_barrier();
    const u32 blocks = __builtin_amdgcn_readfirstlane(*non_finite);
    if (__builtin_expect(blocks != 0, 0)) cells_again<T>(Again(lds, blocks));
}

static long align256(long x) { return (x + 255) / 256 * 256; }
static long stats_bytes(int B, int H, int W) { return 48L * B * H * W; }
static long padded_bytes(int B, int channels, int H, int W) { return 2L * B * channels * H * (W + 1); }

template <typename T, bool STREAM>
static hipError_t launch(const void *q, const void *key, const void *value, const void *grad_out, float *stats,
                         void *grad_q, void *grad_key, void *grad_value, int B, int d, int C, int H, int W,
                         hipStream_t st) {
    constexpr int NSW = 8;
    const bool odd = W % 2 != 0;
    const void *key_rows = key, *value_rows = value;
    if (odd) {
        u32 *const pk = (u32 *)((char *)stats + align256(stats_bytes(B, H, W)));
        u32 *const pv = (u32 *)((char *)pk + align256(padded_bytes(B, d, H, W)));
        const long most = (long)B * (d > C ? d : C) * H * (((W + 1) / 2 + 3) / 4);
        const long blocks = (most + 255) / 256;
        hipLaunchKernelGGL(pad_rows_kernel, dim3((unsigned)(blocks < 4096 ? blocks : 4096), 2), dim3(256), 0, st,
                           (const unsigned short *)key, (const unsigned short *)value, pk, pv, (long)B * d * H, (long)B * C * H, W);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
        key_rows = pk, value_rows = pv;
    }
    Args<T> args{(const T *)q, (const T *)key, (const T *)value, (const T *)grad_out, stats, (T *)grad_q, (T *)grad_key,
                 (T *)grad_value, (const T *)key_rows, (const T *)value_rows, B, d, C, H, W, W + (odd ? 1 : 0), 0, 0, 0, 0, 0};
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
        if (odd) hipLaunchKernelGGL((bwd_pixel_kernel<T, NSW, false, true>), dim3(args.per_xcd * 8), dim3(128 * NSW), 0, st, args);
        else hipLaunchKernelGGL((bwd_pixel_kernel<T, NSW, STREAM, false>), dim3(args.per_xcd * 8), dim3(128 * NSW), 0, st, args);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    if (!grad_key && !grad_value) return hipSuccess;
    // cell blocks 4 I - 2 .. 4 I + 1 that hold a cell of 0 .. W - 1
    const int nI = (W + 1) / 4 + 1, nJ = (H + 1) / 4 + 1;
    if (!tile((nI + TBX - 1) / TBX, nJ)) return hipErrorNotSupported;
    if (odd) hipLaunchKernelGGL((bwd_cell_kernel<T, true>), dim3(args.per_xcd * 8), dim3(CNT), 0, st, args);
    else hipLaunchKernelGGL((bwd_cell_kernel<T, false>), dim3(args.per_xcd * 8), dim3(CNT), 0, st, args);
    return hipGetLastError();
}

}  // namespace bwm16

// Gradients of the fused operator (any of them may be NULL); f16 / bf16, K = 5, s = 2, W >= 16, low-res tensors
// 4-byte (W odd: 2-byte) and high-res tensors 16-byte aligned, every image of every tensor below 2 GiB.
// Scratch (`scratch` bytes at stats): 3 floats per output pixel and, where W is odd, padded copies of key and
// value.
// hipErrorNotSupported otherwise (nothing is launched then).
bool sapa_b_bwd16_serves(int d, int C, int H, int W, int K, int s, int dtype) {
    return K == 5 && s == 2 && W >= 16 && (dtype == 2 || dtype == 3) &&
           wm::offsets_fit(d > C ? d : C, (long)H * (W + W % 2) * 8);
}

long sapa_b_bwd16_workspace(int B, int d, int C, int H, int W) {
    using namespace bwm16;
    return W % 2 == 0 ? stats_bytes(B, H, W)
                      : align256(stats_bytes(B, H, W)) + align256(padded_bytes(B, d, H, W)) + padded_bytes(B, C, H, W);
}

hipError_t sapa_b_bwd16_launch(const void *q, const void *key, const void *value, const void *grad_out, void *stats,
                               void *grad_q, void *grad_key, void *grad_value, int B, int d, int C, int H, int W,
                               int K, int s, int dtype, hipStream_t st, long scratch) {
    if (!sapa_b_bwd16_serves(d, C, H, W, K, s, dtype) || scratch < sapa_b_bwd16_workspace(B, d, C, H, W))
        return hipErrorNotSupported;
    if (((uintptr_t)key | (uintptr_t)value | (uintptr_t)grad_key | (uintptr_t)grad_value) % (W % 2 ? 2 : 4) != 0 ||
        ((uintptr_t)q | (uintptr_t)grad_out | (uintptr_t)grad_q | (uintptr_t)stats) % 16 != 0)
        return hipErrorNotSupported;
    // Beyond the 256 MB memory-side cache the pixel kernel's hi-res traffic is non-temporal, as the
    // forward kernel's -- where the rows of a tile of 8 blocks are whole 128-byte lines (W a multiple
    // of 32); else two workgroups use parts of a line and the caches serve the second (both gradient
    // kernels, B=16, C=256, d=64, bf16: 96x160 621 us streamed, 643 not; 100x168 728 and 710; 168x100
    // 802 and 765).
    const bool stream = W % 32 == 0 && 2L * ((long)B * H * W * (5L * d + 5L * C)) > (256L << 20);
    float *f = (float *)stats;
    if (dtype == 2)
        return stream ? bwm16::launch<f16_t, true>(q, key, value, grad_out, f, grad_q, grad_key, grad_value, B, d, C, H, W, st)
                      : bwm16::launch<f16_t, false>(q, key, value, grad_out, f, grad_q, grad_key, grad_value, B, d, C, H, W, st);
    return stream ? bwm16::launch<bf16_t, true>(q, key, value, grad_out, f, grad_q, grad_key, grad_value, B, d, C, H, W, st)
                  : bwm16::launch<bf16_t, false>(q, key, value, grad_out, f, grad_q, grad_key, grad_value, B, d, C, H, W, st);
}

}  // namespace sapa
