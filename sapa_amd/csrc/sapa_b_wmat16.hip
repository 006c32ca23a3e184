// Fused SAPA-B forward (qk -> softmax -> av) for contiguous (NCHW) f16 / bf16 tensors on the
// 16-bit matrix instructions; written out for K = 5, s = 2, other windows at the kernel.
//
// The 16 parents of a 4 x 4 block share one 8 x 8 window of low-res cells (block + halo of 2),
// and their 64 children need, each, 25 of those 64 cells.  Written over the whole window the two
// products are dense and small enough for the matrix pipe to do them many times over:
//
//   Sim[cell][child]  = sum_c key[c][cell] * q[c][child]            64 x 64 x d
//   P[child][cell]    = softmax over the child's 5 x 5 cells of Sim, 0 on the window's other cells
//   out[child][ch]    = sum_cell P[child][cell] * value[ch][cell]    64 x C x 64
//
// (reference: sapa/sapa/src/cuda/qk_cuda_kernel.cu:55-66, av_cuda_kernel.cu:52-66 and the
// softmax between them in sapa_base.py:38-40; the zero padding of the reference is the zero a
// cell outside the image holds here).  A wave owns one block; a workgroup of NSW waves owns up to
// NSW blocks side by side, so that the rows it writes are up to 8 * NSW children long.
//
// Layouts follow the tensors: NCHW planes are contiguous along x, which is the M / N index of
// every operand here, while the matrix instructions want the reduction index contiguous in a
// lane.  For the logits both operands reduce over channels: ds_read_tr16_b64 transposes 4
// channels x 16 positions on the way out of LDS.  For the aggregation the reduction runs over
// cells, which the value window holds contiguously (two 8-byte reads per operand), and the
// softmax result is already one lane per child with its cells in registers -- the accumulator
// layout of the first product is the A-operand layout of the second, so the weights never leave
// the registers.  They enter the product as a 16-bit value plus a 16-bit remainder (two
// instructions), the sums are fp32: the result is within half a 16-bit spacing of the exact one.
// (bf16: 16 significant bits of a weight.  Against 64 bits the results are off by 1.7e-3 in bf16 and 2.1e-4 in
// fp16, one rounding, as with weights in fp32; a third piece needs 32 registers more than there are.)
// (f16, which holds a pair to 2^-25 only, takes them times 2^15: small weights keep their bits.)
// The 4 x 4 output blocks go back through LDS so that global stores are 16 bytes per lane along
// whole tile rows.
//
// All global -> LDS traffic is direct (buffer loads with the LDS modifier, 16 bytes per lane); an
// offset of 2^31 is outside every descriptor and reads as zero, which is the zero padding above
// and below the image.  A window row starts 2 cells left of its block, so its 16-byte pieces are
// only 4-byte aligned in memory and the first / last of a row run over the row's ends: what they
// bring from the neighbouring row is put right in the registers (logit 0, weight 0 for a cell left
// of x = 0 or right of x = W - 1).  The q / output tile is stored with its 16-byte pieces
// XOR-swizzled so that transposing reads, accumulator writes and the linear store pass are all
// free of 4-way bank conflicts without padding.
//
// Masked cells still enter both products; what a non-finite value does there is mended behind the
// aggregation (wm16_exact.hpp).
#include "wm16_exact.hpp"

namespace sapa {

namespace wm16 {

using namespace wm;

constexpr int CHK = 16;            // channels per staged chunk
constexpr int WROWS = 8;           // window rows = child rows of a block row

// position of the 16-byte piece `pc` of row r, channel ch in the swizzled q / output tile
__device__ __forceinline__ int swz(int ch, int r) { return ((ch & 7) << 1) | ((r + (ch >> 3)) & 1); }

// STREAM: q loads and output stores are non-temporal -- each byte passes once and must not push the
// low-res windows, which neighbouring tiles re-read, out of the caches (fused FPN-large bf16, 860 MB:
// 271 -> 213 us; at a quarter of the size, where everything fits the memory-side cache, 50 -> 58 us:
// the launcher decides by size)
//
// (K, S) other than (5, 2) take the same blocks of 8 x 8 children and 8 x 8 cells, of PB = 8 / S
// parents a side: (7, 4) uses all 64 cells of a window, (5, 4) and (3, 2) 36.  Windows of
// neighbouring blocks start PB cells apart, which the transposing reads (4 cells, 8-byte aligned)
// cannot follow in a shared row, so every block has a piece of 8 cells of its own per row (OWN): a
// low-res cell is staged 8 / PB times, out of the caches, for S * S outputs.  Measured in bf16 against
// the one-parent-per-block matrix kernel on fp32 operands, which these windows took before: K=7, s=4,
// B=4, C=512, d=64, 64x64 250 -> 69 us (4.7 TB/s: memory), B=16, C=256, 50x84 756 -> 309 us (rows
// of 672 bytes: split cache lines); K=5, s=4 165 -> 66 and 480 -> 263 us; K=3, s=2 57 -> 27 and
// 132 -> 52 us; one image 16x16 33 -> 12, 20 -> 15 and 15 -> 15 us.
//
// HALF: images of the key or of the value of an odd number of elements (a kernel of its own: what it
// takes in registers costs the others up to 10 % -- K=3, s=2, B=16, C=256, 50x84 in bf16 83 -> 91 us)
//
// DEEP: three buffers of each kind instead of two, requests two chunks ahead and stores waited for two chunks later
template <typename T, int K, int S, int NSW, bool STREAM, bool ODD, bool HALF, bool DEEP>
__global__ __launch_bounds__(64 * NSW, 4) void
sapa_b_wmat16_kernel(const T *__restrict__ q, const T *__restrict__ key, const T *__restrict__ value,
                     T *__restrict__ out, int d, int C, int H, int W, int tiles_x, int tiles_y, int ns,
                     int nslices, int slice_chunks, int nblocks, int per_xcd) {
    constexpr int NT = 64 * NSW;
    constexpr int PB = 8 / S, R = (K - 1) / 2, SS = S * S;
    constexpr bool OWN = !(K == 5 && S == 2);
    static_assert(PB + K - 1 <= 8 && S * PB == 8, "a block's window");
    static_assert(!OWN || ODD, "pieces of a block's own come through registers");
    static_assert(!HALF || ODD, "half a dword comes through registers");
    // dwords per staged window row: whole pieces of 8 cells (OWN: one per block; a piece of padding
    // keeps the rows of the 16 channels on different banks)
    constexpr int LROW = OWN ? 4 * NSW + 4 : (4 * NSW + 4 + 7) / 8 * 4;
    constexpr int LPC = OWN ? NSW : LROW / 4;                // pieces per row
    constexpr int BSTEP = OWN ? 4 : 2;                       // dwords from a block's window to the next one's
    constexpr int LOWBUF = WROWS * CHK * LROW;               // dwords per low-res buffer
    constexpr int NLP = WROWS * CHK * LPC;                   // 16-byte pieces per low-res buffer
    constexpr int NLI = (NLP + NT - 1) / NT;                 // 16-byte direct loads per thread and window, at most
    constexpr int HIROW = 8 * NSW / 2;                       // dwords per q / output tile row
    constexpr int HICH = WROWS * HIROW;                      // dwords per channel of the tile
    constexpr int HIBUF = CHK * HICH;                        // dwords per q / output buffer
    constexpr int NHI = HIBUF / 4 / NT;                      // 16-byte pieces per thread and tile
    static_assert(HIBUF % (4 * NT) == 0 && NLP % 64 == 0, "whole direct loads");
    static_assert(OWN || 4 * NSW + 4 <= 2 * LROW, "window row");
    static_assert(NSW == 16 || NSW == 8, "piece swizzle");
    constexpr int NPC = 2 * NSW / 2;                         // 16-byte pieces per tile row = NSW

    // buffers of each kind, one chunk per buffer
    static_assert(!DEEP || (STREAM && !ODD), "three buffers: streamed tensors");
    constexpr int NB = DEEP ? 3 : 2;
    // (of two by the lowest bit: a signed remainder in the kernels whose registers spill cost K=7, s=4, B=4, C=512, 64x64
    // in bf16 68.1 -> 68.7 us)
    auto ring = [](int j) { return NB == 2 ? j & 1 : j % NB; };
    __shared__ __attribute__((aligned(16))) u32 lds[NB * (LOWBUF + HIBUF) + 4];
    u32 *const lowbuf = lds, *const hibuf = lds + NB * LOWBUF;
    const u32 low_at = lds_address((const __attribute__((address_space(3))) u32 *)lds), hi_base = low_at + NB * LOWBUF * 4;
    // blocks of the tile with a non-finite result (in the same array: with a variable of its own the
    // compiler waits for direct loads in other places, 258 -> 268 us at FPN-large)
    u32 *const non_finite = lds + NB * (LOWBUF + HIBUF);

    const int logical = (int)(blockIdx.x % 8) * per_xcd + (int)(blockIdx.x / 8);
    if (logical >= nblocks) return;
    int tile = logical, vbase = 0;                           // first value chunk
    if (nslices > 1) tile = logical / nslices, vbase = (logical - tile * nslices) * slice_chunks;
    const int tx = tile % tiles_x, ty = (tile / tiles_x) % tiles_y, n = tile / (tiles_x * tiles_y);
    const int X0 = tx * PB * ns, Y0 = ty * PB;               // first parent of the tile
    const int nsx = (W + PB - 1) / PB;
    const int ns_here = nsx - tx * ns < ns ? nsx - tx * ns : ns;

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g = lane >> 4, i16 = lane & 15;
    const long lpix = (long)H * W;
    const u32 lplane = (u32)(lpix * sizeof(T)), hplane = SS * lplane;

    // direct-load offsets inside one image, without the chunk's first channel.  A low-res piece is
    // 8 cells from x = X0 - 2 + 8 pc on: 4-byte aligned, and where it runs over an end of its row it
    // brings the neighbouring row's cells (zeros past the tensor's end) -- the cells left of x = 0
    // and right of x = W - 1 are put right in the registers below (cell_outside).  Only the piece
    // that starts 2 cells before the image's first has no address: it reads as zeros and its 6
    // cells are fetched apart (patch_low).
    u32 off_low[NLI], off_hi[NHI];
    bool low_odd[NLI];         // ODD: the piece starts in the middle of a dword
    int tail_children[NHI];    // children of its row in a row's last 16-byte piece (the rest is the next row's), else 8
    int patch_slot = -1;
#pragma unroll
    for (int i = 0; i < NLI; ++i) {
        const int slot = i * NT + tid, rc = slot / LPC, pc = slot % LPC;
        const int r = rc / CHK, ch = rc % CHK;
        const int y = Y0 - R + r, x = X0 - R + (OWN ? PB : 8) * pc;
        const bool ok = slot < NLP && (OWN ? pc < ns_here : 8 * pc < 4 * ns_here + 4) && y >= 0 && y < H && x < W;
        low_odd[i] = ODD && ((ch * lpix + (long)y * W + x) & 1);
        off_low[i] = ok ? (u32)(ch * lpix + (long)y * W + x - low_odd[i]) * (u32)sizeof(T) : OUTSIDE;
        if (ok && x < 0 && y == 0 && ch == 0) patch_slot = slot;
    }
#pragma unroll
    for (int i = 0; i < NHI; ++i) {
        const int slot = i * NT + tid, ch = slot / (WROWS * NPC), r = (slot / NPC) % WROWS;
        const int pc = (slot % NPC) ^ (swz(ch, r) & (NPC - 1));
        const int cy = S * Y0 + r, cx = S * X0 + 8 * pc;
        const bool ok = pc < ns_here && cy < S * H && cx < S * W;
        off_hi[i] = ok ? (u32)(ch * SS * lpix + (long)cy * S * W + cx) * (u32)sizeof(T) : OUTSIDE;
        tail_children[i] = ok && cx + 8 > S * W ? S * W - cx : 8;
    }

    const int nKc = (d + CHK - 1) / CHK, allV = (C + CHK - 1) / CHK;
    const int nVc = allV - vbase < slice_chunks ? allV - vbase : slice_chunks, ntot = nKc + nVc;
    // (HALF: an image ends with half a dword, which lies outside: nothing behind a tensor is read, and
    // low_end puts that element in its place)
    const __amdgpu_buffer_rsrc_t rk = __builtin_amdgcn_make_buffer_rsrc(
        (void *)(key + (long)n * d * lpix), 0, (int)(HALF ? d * lplane & ~3u : d * lplane), 0x00020000);
    const __amdgpu_buffer_rsrc_t rv = __builtin_amdgcn_make_buffer_rsrc(
        (void *)(value + (long)n * C * lpix), 0, (int)(HALF ? C * lplane & ~3u : C * lplane), 0x00020000);
    const __amdgpu_buffer_rsrc_t ro = __builtin_amdgcn_make_buffer_rsrc(
        (void *)(out + (long)n * C * SS * lpix), 0, (int)(C * hplane), 0x00020000);

    (void)rk, (void)rv;
    // Chunk j is the key + q channels 16 j .. for j < nKc and the value channels 16 (j - nKc) ..
    // after; it lives in buffer j % NB and is requested NB chunks ahead, as soon as every wave is
    // done with that buffer.  A channel past the tensor's last lies past the descriptor: zeros.
    const u32x4 dq = dma_rsrc(q + (long)n * d * SS * lpix, d * hplane);
    const u32x4 dk = dma_rsrc(key + (long)n * d * lpix, d * lplane);
    const u32x4 dv = dma_rsrc(value + (long)n * C * lpix, C * lplane);
    auto stage_low = [&](u32x4 r, u32 c0, int buf) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < NLI; ++i)
            if ((i + 1) * NT <= NLP || i * NT + wave * 64 < NLP)
                load_lds(r, low_at + (buf * LOWBUF + wave * 256 + i * NT * 4) * 4, off_low[i] + c0 * lplane);
    };
    auto stage_q = [&](u32 c0, int buf) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < NHI; ++i) load_lds<STREAM>(dq, hi_base + (buf * HIBUF + wave * 256 + i * NT * 4) * 4, off_hi[i] + c0 * hplane);
    };
    // operations that this wave issues for chunk j
    auto loads_of = [&](int j) __attribute__((always_inline)) {
        return j < ntot ? (ODD ? 0 : (NLP - wave * 64 + NT - 1) / NT) + (j < nKc ? NHI : 0) : 0;
    };
    auto stage = [&](int j) __attribute__((always_inline)) {
        if (j < nKc) {
            if (!ODD) stage_low(dk, (u32)(j * CHK), ring(j));
            stage_q((u32)(j * CHK), ring(j));
        } else if (!ODD && j < ntot) {
            stage_low(dv, (u32)((j - nKc + vbase) * CHK), ring(j));
        }
    };
    // ODD: an odd W puts every other row of a low-res plane in the middle of a dword, where direct loads
    // cannot start.  The pieces of chunk j come through registers instead, from the dword before, and are
    // moved by half a dword on their way into LDS: requested before chunk j - 1 is computed on, written
    // behind it.
    u32x4 low_reg[ODD ? NLI : 1];
    u32 low_next[ODD ? NLI : 1];
    auto low_load = [&](int j) __attribute__((always_inline)) {
        if (!ODD || j >= ntot) return;
        const u32 c0 = (u32)((j < nKc ? j : j - nKc + vbase) * CHK);
        const __amdgpu_buffer_rsrc_t r = j < nKc ? rk : rv;
#pragma unroll
        for (int i = 0; i < NLI; ++i) {
            u32 off = off_low[i] + c0 * lplane;
            // (OWN: the piece without an address: the tensor's first cells, put in place by low_commit)
            if (OWN && c0 == 0 && patch_slot == i * NT + tid) off = 0;
            low_reg[i] = __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0);
            low_next[i] = __builtin_amdgcn_raw_buffer_load_b32(r, off + 16, 0, 0);
        }
    };
    auto low_commit = [&](int j) __attribute__((always_inline)) {
        if (!ODD || j >= ntot) return;
#pragma unroll
        for (int i = 0; i < NLI; ++i) {
            const int slot = i * NT + tid;
            const u32x4 v = low_reg[i];
            u32x4 m = v;
            if (low_odd[i])
                m = u32x4{__builtin_amdgcn_alignbyte(v[1], v[0], 2), __builtin_amdgcn_alignbyte(v[2], v[1], 2),
                          __builtin_amdgcn_alignbyte(v[3], v[2], 2), __builtin_amdgcn_alignbyte(low_next[i], v[3], 2)};
            if (OWN && patch_slot == slot && (j == 0 || (j == nKc && vbase == 0)))
                // moved up by R cells (R = 3: by 1 in the second block's piece)
                m = R == 2 ? u32x4{0u, v[0], v[1], v[2]}
                    : R == 1 || slot % LPC == 1
                        ? u32x4{v[0] << 16, __builtin_amdgcn_alignbyte(v[1], v[0], 2),
                                __builtin_amdgcn_alignbyte(v[2], v[1], 2), __builtin_amdgcn_alignbyte(v[3], v[2], 2)}
                        : u32x4{0u, v[0] << 16, __builtin_amdgcn_alignbyte(v[1], v[0], 2),
                                __builtin_amdgcn_alignbyte(v[2], v[1], 2)};
            const int at = OWN ? slot / LPC * LROW + slot % LPC * 4 : slot * 4;
            if (NLP % NT == 0 || slot < NLP) *(u32x4 *)(lowbuf + ring(j) * LOWBUF + at) = m;
        }
    };
    // behind low_commit(j), by the wave that wrote the piece: the last element of an image of an odd number
    auto low_end = [&](int j) __attribute__((always_inline)) {
        const int c0 = (j < nKc ? j : j - nKc + vbase) * CHK, nch = j < nKc ? d : C;
        if (!HALF || j >= ntot || c0 + CHK < nch || !(nch & lpix & 1)) return;
        const T last = (j < nKc ? key : value)[((long)n + 1) * nch * lpix - 1];
#pragma unroll
        for (int i = 0; i < NLI; ++i) {
            const int slot = i * NT + tid, at = OWN ? slot / LPC * LROW + slot % LPC * 4 : slot * 4;
            const u32 e = (u32)((long)(nch - c0) * lpix) - 1u - (u32)(((int)off_low[i] >> 1) + (low_odd[i] ? 1 : 0));
            if (e < 8u) ((T *)(lowbuf + ring(j) * LOWBUF + at))[e] = last;
        }
    };
    // chunk jn (the first of the keys or of the values) has landed in this wave's slots: the 6
    // cells of the piece that has no address (first row of the image's first channel, tile at the
    // left edge)
    auto patch_low = [&](int jn) __attribute__((always_inline)) {
        if (!OWN && tx == 0 && ty == 0 && patch_slot >= 0 && (jn < nKc || vbase == 0)) {
            const __amdgpu_buffer_rsrc_t r = jn < nKc ? rk : rv;
            u32 *dst = lowbuf + ring(jn) * LOWBUF + patch_slot * 4;
#pragma unroll
            for (int k = 1; k < 4; ++k) dst[k] = __builtin_amdgcn_raw_buffer_load_b32(r, 4 * (k - 1), 0, 0);
        }
    };
    const bool row_tail = W % PB != 0 && X0 + PB * ns_here > W;      // wave-uniform
    const bool active = wave < ns_here;
    const int t = wave;                                       // this wave's block of the tile

    if (tid == 0) *non_finite = 0;
    low_load(0);
    low_commit(0);
    low_end(0);
    stage(0);
    stage(1);
    if (NB > 2) stage(2);
    // chunk 0: all but the loads of the chunks after it
    wait_all_but(ODD ? 0 : loads_of(1) + (NB > 2 ? loads_of(2) : 0));
    patch_low(0);
    lds_barrier();

    // ---- logits: Sim[cell][child], 4 x 4 accumulator blocks of 16 x 16 ----
    // block (mb, nb), lane (g, i16), element v: cell (row 2 mb + g / 2, column 4 (g % 2) + v) of the
    // window, child (row 2 nb + i16 / 8, column i16 % 8) of the block's 8 x 8 children
    f32x4 sim[4][4];
#pragma unroll
    for (int mb = 0; mb < 4; ++mb)
#pragma unroll
        for (int nb = 0; nb < 4; ++nb) sim[mb][nb] = f32x4{0.f, 0.f, 0.f, 0.f};
    // transposing reads: lane (g, L = i16) addresses channel 4 g + L / 4, the 4 positions of group
    // L % 4 of the 16 (row (L % 4) / 2 of the pair, columns 4 (L % 2) ..)
    const int tch = 4 * g + (i16 >> 2), trow = (i16 & 3) >> 1, tcol = i16 & 1;
    for (int j = 0; j < nKc; ++j) {
        low_load(j + 1);
        if (active) {
            const u32 *kb = lowbuf + ring(j) * LOWBUF, *qb = hibuf + ring(j) * HIBUF;
            u32x2 a[4], b[4];
#pragma unroll
            for (int mb = 0; mb < 4; ++mb)
                a[mb] = read_tr(kb + ((2 * mb + trow) * CHK + tch) * LROW + BSTEP * t + 2 * tcol);
#pragma unroll
            for (int nb = 0; nb < 4; ++nb) {
                const int r = 2 * nb + trow;
                b[nb] = read_tr(qb + tch * HICH + r * HIROW + ((t ^ (swz(tch, r) & (NPC - 1))) << 2) + 2 * tcol);
            }
#pragma unroll
            for (int mb = 0; mb < 4; ++mb)
#pragma unroll
                for (int nb = 0; nb < 4; ++nb) sim[mb][nb] = Mma<T>::k16(a[mb], b[nb], sim[mb][nb]);
        }
        low_commit(j + 1);
        low_end(j + 1);
        // chunk j + 1: all but the loads of a chunk requested since
        wait_all_but(NB > 2 ? loads_of(j + 2) : 0);
        if (j + 1 == nKc) patch_low(nKc);
        lds_barrier();
        stage(j + NB);
    }

    // ---- softmax over each child's 5 x 5 cells; the weights as A operands of the aggregation ----
    // reduction step s of the aggregation covers the cells of blocks mb = 2 s, 2 s + 1; lane
    // (g, child) holds 4 + 4 of its 32
    u32x4 whi[4][2], wlo[4][2];
    constexpr float UP = __is_same(T, f16_t) ? 32768.f : 1.f;
    if (active) {
        // element v of every block is window column 4 (g % 2) + v.  Outside the image the key is zero
        // (logit 0) and so is the value (the weight may as well be 0): only the waves at a row's
        // ends have such columns.
        bool cell_outside[4];
#pragma unroll
        for (int v = 0; v < 4; ++v) cell_outside[v] = (u32)(X0 + PB * t - R + 4 * (g & 1) + v) >= (u32)W;
        const bool at_row_end = X0 + PB * t - R < 0 || X0 + PB * t - R + 7 >= W;      // wave-uniform
        if (at_row_end) {
#pragma unroll
            for (int mb = 0; mb < 4; ++mb)
#pragma unroll
                for (int nb = 0; nb < 4; ++nb)
#pragma unroll
                    for (int v = 0; v < 4; ++v)
                        if (cell_outside[v]) sim[mb][nb][v] = 0.f;
        }
        // a child of parent column px takes window columns px .. px + K - 1: -inf for the others
        const int px = (i16 & 7) / S;
        const float NEG_INF = -__builtin_inff(), LOG2E = 1.4426950408889634f;
        bool col_in[4];
#pragma unroll
        for (int v = 0; v < 4; ++v) col_in[v] = (u32)(4 * (g & 1) + v - px) < (u32)K;
#pragma unroll
        for (int nb = 0; nb < 4; ++nb) {
            // child row 2 nb + i16 / 8 -> parent row pr: window rows pr .. pr + K - 1.  Block mb holds
            // rows 2 mb (lanes g < 2) and 2 mb + 1: all, some or none of its lanes take part
            const int pr = 2 * nb / S;
            float x[4][4], m = NEG_INF;
#pragma unroll
            for (int mb = 0; mb < 4; ++mb) {
                const bool lo_in = 2 * mb >= pr && 2 * mb < pr + K, hi_in = 2 * mb + 1 >= pr && 2 * mb + 1 < pr + K;
                if (!lo_in && !hi_in) continue;
                const bool row_in = (g >> 1) ? hi_in : lo_in;
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    x[mb][v] = (col_in[v] & row_in) ? sim[mb][nb][v] : NEG_INF;
                    m = fmaxf(m, x[mb][v]);
                }
            }
            m = fmaxf(m, __shfl_xor(m, 16));
            m = fmaxf(m, __shfl_xor(m, 32));
            // exp(x - m) as 2^(x log2 e - m log2 e); a masked cell gives 2^-inf = 0
            const float mneg = -m * LOG2E;
            float e[4][4], sum = 0.f;
#pragma unroll
            for (int mb = 0; mb < 4; ++mb) {
                const bool lo_in = 2 * mb >= pr && 2 * mb < pr + K, hi_in = 2 * mb + 1 >= pr && 2 * mb + 1 < pr + K;
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    e[mb][v] = lo_in || hi_in ? __builtin_amdgcn_exp2f(__builtin_fmaf(x[mb][v], LOG2E, mneg)) : 0.f;
                    if (lo_in || hi_in) sum += e[mb][v];
                }
            }
            sum += __shfl_xor(sum, 16);
            sum += __shfl_xor(sum, 32);
            const float inv = UP / sum;
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                float p[8];
#pragma unroll
                for (int k = 0; k < 8; ++k) p[k] = e[2 * s + k / 4][k % 4] * inv;
                if (at_row_end) {
#pragma unroll
                    for (int k = 0; k < 8; ++k)
                        if (cell_outside[k % 4]) p[k] = 0.f;
                }
                typedef T tx8 __attribute__((ext_vector_type(8)));
                whi[nb][s] = u32x4{pack2<T>(p[0], p[1]), pack2<T>(p[2], p[3]), pack2<T>(p[4], p[5]), pack2<T>(p[6], p[7])};
                const tx8 hi = __builtin_bit_cast(tx8, whi[nb][s]);
#pragma unroll
                for (int k = 0; k < 8; ++k) p[k] -= (float)hi[k];
                wlo[nb][s] = u32x4{pack2<T>(p[0], p[1]), pack2<T>(p[2], p[3]), pack2<T>(p[4], p[5]), pack2<T>(p[6], p[7])};
            }
        }
    }

    // ---- aggregation: out[child][channel], per chunk of 16 channels ----
    NonFinite seen;
    for (int j = nKc; j < ntot; ++j) {
        const u32 c0 = (u32)((j - nKc + vbase) * CHK);
        u32 *ob = hibuf + (j & 1) * HIBUF;                      // no loads into this ring any more
        low_load(j + 1);
        if (active) {
            const u32 *vb = lowbuf + ring(j) * LOWBUF;
            // B operand of step s: lane (g, channel i16) holds the cells of rows 4 s + g / 2 and
            // 4 s + 2 + g / 2, columns 4 (g % 2) .. + 3 -- the order the weights are held in
            u32x4 b[2];
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                const u32 *p = vb + ((4 * s + (g >> 1)) * CHK + i16) * LROW + BSTEP * t + 2 * (g & 1);
                const u32x2 lo = *(const u32x2 *)p, hi = *(const u32x2 *)(p + 2 * CHK * LROW);
                b[s] = u32x4{lo[0], lo[1], hi[0], hi[1]};
            }
#pragma unroll
            for (int nb = 0; nb < 4; ++nb) {
                f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int s = 0; s < 2; ++s) {
                    acc = Mma<T>::k32(whi[nb][s], b[s], acc);
                    acc = Mma<T>::k32(wlo[nb][s], b[s], acc);
                }
                // (a value that is not finite makes its channel's results so for every child of the block)
                if (nb == 0) seen.see(acc[0]);
                if (UP != 1.f) acc *= 1.f / UP;
                // element v: child (row 2 nb + g / 2, column 4 (g % 2) + v), channel c0 + i16
                const int r = 2 * nb + (g >> 1);
                *(u32x2 *)(ob + i16 * HICH + r * HIROW + ((t ^ (swz(i16, r) & (NPC - 1))) << 2) + 2 * (g & 1)) =
                    u32x2{pack2<T>(acc[0], acc[1]), pack2<T>(acc[2], acc[3])};
                // (no register to spare: with the products of several nb in flight the loop goes through scratch
                // memory; K=7, s=4, B=4, C=512, 64x64 in bf16 71.2 us, 69.1 so)
                if (OWN) __builtin_amdgcn_sched_barrier(0);
            }
        }
        low_commit(j + 1);
        low_end(j + 1);
        // chunk j + 1: all but the stores of chunk j - 1 (at least NHI) and the loads requested behind them
        wait_all_but(NB > 2 ? loads_of(j + 2) + (j > nKc ? NHI : 0) : 0);
        lds_barrier();
        // the tile's 16 channels x 8 rows, 16 bytes per lane, right after the barrier that completes
        // them (sending them behind the next chunk's matrix instructions measured slower); a piece
        // outside the tensor (ragged tile, channel past the last) lies outside the descriptor and
        // is dropped
#pragma unroll
        for (int i = 0; i < NHI; ++i) {
            const u32x4 o = *(const u32x4 *)(ob + (i * NT + tid) * 4);
            u32 off = off_hi[i] + c0 * hplane;
            if (row_tail && tail_children[i] < 8) {
                if (S == 4 || !ODD) {
                    __builtin_amdgcn_raw_buffer_store_b64(u32x2{o[0], o[1]}, ro, off, 0, 0);
                } else {
#pragma unroll
                    for (int k = 0; k < 3; ++k)
                        if (2 * k < tail_children[i]) __builtin_amdgcn_raw_buffer_store_b32(o[k], ro, off + 4 * k, 0, 0);
                }
                off = OUTSIDE;
            }
            if constexpr (STREAM) __builtin_amdgcn_raw_buffer_store_b128(o, ro, off, 0, 2);
            else __builtin_amdgcn_raw_buffer_store_b128(o, ro, off, 0, 0);
        }
        // (the next request behind the stores: 208 us at FPN-large against 216 with the loads first)
        if (!ODD && j + NB < ntot) stage_low(dv, (u32)((j + NB - nKc + vbase) * CHK), ring(j));
    }

    // ---- blocks with a non-finite result: again, term by term ----
    if (seen.any()) atomicOr(non_finite, 1u << t);
    lds_barrier();
    const u32 blocks = __builtin_amdgcn_readfirstlane(*non_finite);
    if (__builtin_expect(blocks != 0, 0)) {
        settled();
        const int c_hi = (vbase + nVc) * CHK < C ? (vbase + nVc) * CHK : C;
        for (int b = 0; b < ns_here; ++b)
            if (blocks >> b & 1)
                exact_children<T, K, S, NT>((float *)lds, plane_of<false>(q, n, d, SS * lpix), plane_of<false>(key, n, d, lpix),
                                            plane_of<false>(value, n, C, lpix), plane_of<false>(out, n, C, SS * lpix), d,
                                            vbase * CHK, c_hi, H, W, S * Y0, S * X0 + 8 * b);
    }
}

template <typename T, int K, int S, int NSW, bool STREAM, bool ODD, bool HALF = false, bool DEEP = false>
static hipError_t launch_geom(const void *q, const void *key, const void *value, void *out, int B, int d,
                              int C, int H, int W, hipStream_t st) {
    constexpr int PB = 8 / S;
    const int nsx = (W + PB - 1) / PB;
    const int tiles_x = (nsx + NSW - 1) / NSW, tiles_y = (H + PB - 1) / PB;
    const int ns = (nsx + tiles_x - 1) / tiles_x;             // blocks per tile, balanced over the row
    const long tiles = (long)tiles_x * tiles_y * B;
    // Fewer tiles than CUs: a workgroup's time is a chain of one step per 16 channels, so the value
    // channels are split over several workgroups per tile, each forming the weights again, up to one
    // workgroup per CU (B=8, C=256, d=32, bf16, 16x16: 12.5 us unsplit, 8.0 / 7.3 / 8.9 with up to 128 /
    // 256 / 512 workgroups; 32x32: 16.6, 12.6 / 11.1 / 13.2; B=2, d=64, 50x84: 18.7, 18.4 / 13.6 / 14.8)
    const int allV = (C + CHK - 1) / CHK;
    long want = 256 / tiles;
    // ... and from 129 tiles, each CU with room for two workgroups of 8 blocks, in three slices where those are still
    // resident at once and many enough channels share a tile's weights (bf16, d=64, one slice / two / three: 4 images 50x84,
    // 156 tiles, 256 channels 21.6 / 20.6 / 18.6 us, 512 of them 51x83 53.2 / 47.4 / 44.5; K=7, s=4, 160 tiles 31.5 / 27.2
    // / 25.6; but 128 channels, d=32, 160 tiles 13.7 / 14.9 / 14.4, and 224 or 234 tiles 19.8 / 18.9 / 24.5, 29.9 / 32.0
    // / 37.9)
    if (NSW == 8 && tiles > 128 && 3 * tiles <= 512 && allV >= 16) want = 3;
    want = want < 1 ? 1 : want > allV ? allV : want;
    const int slice_chunks = (int)((allV + want - 1) / want), nslices = (allV + slice_chunks - 1) / slice_chunks;
    const long nb = tiles * nslices;
    if (nb > (1L << 30)) return hipErrorNotSupported;
    const int per_xcd = (int)((nb + 7) / 8);
    hipLaunchKernelGGL((sapa_b_wmat16_kernel<T, K, S, NSW, STREAM, ODD, HALF, DEEP>), dim3(per_xcd * 8), dim3(64 * NSW), 0, st, (const T *)q,
                       (const T *)key, (const T *)value, (T *)out, d, C, H, W, tiles_x, tiles_y, ns,
                       nslices, slice_chunks, (int)nb, per_xcd);
    return hipGetLastError();
}

}  // namespace wm16

// Fused forward only; f16 / bf16, (K, s) = (5, 2), (7, 4), (5, 4) or (3, 2), W >= 4, low-res tensors 4-byte and
// high-res tensors 16-byte aligned, every image of every tensor below 2 GiB (32-bit offsets
// inside an image); hipErrorNotSupported otherwise.
hipError_t sapa_b_wmat16_launch(int mode, const void *q, const void *key, const void *value, void *out, int B,
                                int d, int C, int H, int W, int K, int s, int dtype, hipStream_t st) {
    const bool k5s2 = K == 5 && s == 2, k7s4 = K == 7 && s == 4, k5s4 = K == 5 && s == 4, k3s2 = K == 3 && s == 2;
    if (mode != TILED_FUSED || !(k5s2 || k7s4 || k5s4 || k3s2) || W < 4) return hipErrorNotSupported;
    if (dtype != 2 && dtype != 3) return hipErrorNotSupported;
    if (!wm::offsets_fit(d > C ? d : C, (long)H * W * s * s * 2)) return hipErrorNotSupported;
    if (((uintptr_t)key | (uintptr_t)value) % 4 != 0 || ((uintptr_t)q | (uintptr_t)out) % 16 != 0)
        return hipErrorNotSupported;
    // bytes read and written once; beyond the 256 MB memory-side cache they are streamed, in tiles of
    // up to 16 blocks (longer rows per store); what fits the cache takes tiles of 8 blocks, two
    // workgroups per CU (FPN 25x42 at B=16: 24 -> 19 us, SegFormer 64x64 at B=8: 25 -> 20 us).  The
    // arithmetic of a child does not depend on the tiling: results are the same bit for bit.  An odd W
    // (low-res rows through registers) has tiles of 8 blocks only: with 16 the registers do not suffice
    // (B=16, C=256, d=64, 42x25: 24 us, by vector fmas 65; 100x167: 289 us against 451; rows below 16
    // cells, 13x13 at B=8: 9 us against 19 on the one-block-per-parent matrix kernel).
    const long bytes = 2L * ((long)B * H * W * (1L + s * s) * ((long)d + C));
    const bool stream = bytes > (256L << 20);
    // Three buffers where the bytes are well beyond that cache and the chain of chunks is long enough for them (d=64 in
    // bf16, three sets of tensors in turn, two buffers / three, us per call: C=256, 16 images 100x168, 820 MiB, 257 / 247,
    // 10 of them, 513, 156 / 153, 16 of 96x96, 450, 134 / 126; but 8 of 100x168, 410, 118 / 122, 32 of 50x84, 410, 119 / 128,
    // 3 of them with C=512, 277, 67 / 73; chains of 10 chunks, d=32, C=128: 16 images, 410 MiB, 123 / 133, 32, 820, 273 / 275,
    // of 6 348 / 363.  One set again and again, partly from the cache: 16 of 100x168 215 / 220)
    const bool deep = bytes > (432L << 20) && (d + wm16::CHK - 1) / wm16::CHK + (C + wm16::CHK - 1) / wm16::CHK >= 16;
    const bool odd = W % 2 != 0, half = ((d | C) & H & W & 1) != 0;
    // Other windows: streamed only where a tile's rows are whole 128-byte lines (s W a multiple of 64);
    // else parts of a line are written by two workgroups, and the caches put them together
    // (K=7, s=4, bf16: B=4, C=512, 64x64: 69 us streamed, 114 not; B=16, C=256, 50x84: 386 and 309)
    const bool lines = stream && s * W % 64 == 0;
#define SAPA_WM16_OWN(T, KV, SV)                                                                                 \
    if (K == KV && s == SV)                                                                                      \
        return half    ? wm16::launch_geom<T, KV, SV, 8, false, true, true>(q, key, value, out, B, d, C, H, W, st)  \
               : lines ? wm16::launch_geom<T, KV, SV, 8, true, true>(q, key, value, out, B, d, C, H, W, st)       \
                      : wm16::launch_geom<T, KV, SV, 8, false, true>(q, key, value, out, B, d, C, H, W, st);
#define SAPA_WM16_CASE(T)                                                                                       \
    SAPA_WM16_OWN(T, 7, 4) SAPA_WM16_OWN(T, 5, 4) SAPA_WM16_OWN(T, 3, 2)                                         \
    return half     ? wm16::launch_geom<T, 5, 2, 8, false, true, true>(q, key, value, out, B, d, C, H, W, st)    \
           : odd    ? wm16::launch_geom<T, 5, 2, 8, false, true>(q, key, value, out, B, d, C, H, W, st)          \
           : deep   ? wm16::launch_geom<T, 5, 2, 16, true, false, false, true>(q, key, value, out, B, d, C, H, W, st) \
           : stream ? wm16::launch_geom<T, 5, 2, 16, true, false>(q, key, value, out, B, d, C, H, W, st)         \
                    : wm16::launch_geom<T, 5, 2, 8, false, false>(q, key, value, out, B, d, C, H, W, st)
    if (dtype == 2) {
        SAPA_WM16_CASE(f16_t);
    }
    SAPA_WM16_CASE(bf16_t);
#undef SAPA_WM16_CASE
#undef SAPA_WM16_OWN
}

}  // namespace sapa
