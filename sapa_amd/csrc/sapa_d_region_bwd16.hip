// Backward of the fused SAPA-D operator for f16 / bf16 tensors and up_factor 2, all four gradients from
// one pass over the samples:
//
//   att = softmax_p(sampled key . q) (recomputed)      gat[p] = grad_out . sampled value
//   gl[p] = att[p] (gat[p] - sum att gat)              grad_offset from the four corners' products
//   grad_query = sum_p gl[p] sampled key               grad_value, grad_key: the samples' scatters
//
// (the chain of deformsapa/deformsapa/src/cuda/deform_qk_cuda_kernel.cu:70-137 and
// deform_av_cuda_kernel.cu:70-137 with autograd's softmax backward between them).  A workgroup owns a
// strip of 8 parents (16 hi-res pixels) by some rows of parents of one (image, group) and walks down it in
// steps of one row of parents (32 pixels), with the key and value window of the step's samples in LDS:
//
//   A  Sim[pixel][cell] = q . key, G'[pixel][cell] = grad_out . value over the step's band of cells
//   B  per (pixel, point): logit, gat and both position derivatives from four entries of Sim and of G';
//      softmax and its backward across the lanes; the pixel's rows then become Wv (att x corner
//      weights) and Wg (gl x corner weights): integers, added with LDS atomics -- exact in any order
//   C  grad_query = Wg . key;  grad_value[cell] += Wv^T . grad_out and grad_key[cell] += Wg^T . q, whose
//      sums stay in registers until the band has passed their cell and are then added to fp32 buffers
//
// The chain before (sapa_d_bwdmat.hip, then sapa_d_scatter.hip twice; they still serve fp32, other
// factors and wider groups) went over the samples three times, kept att and gl in memory between them,
// multiplied widened values on the fp32 matrix instructions, and brought a window of 121 / 289 cells in for
// 16 / 256 pixels.  Strips bring a row of 17 cells in for 32 pixels and add each cell's sums once per
// strip, not once per 16 x 16 pixels (a form of this kernel on such squares, windows whole in LDS: 9 us
// per square in front of its first step, 115 us of 665 for the additions).
//
// Measured (B=8, C=256, 4 groups, d=32, 64x64 -> 128x128, bf16): this kernel 427 us with 25 points and 351 with 9, a
// training step 656 and 536, by the chain before 1016 and 800; C=128, 90x121, 9 points, channels-last 2600 -> 1712.  What bounds it is
// the chain of a step's three phases, each behind a barrier with the 16 waves that one CU's LDS holds (timed apart
// in a form of 470 us, whose 60 for memory are no more waited for: A 35, B 150, C 175, barriers 50): 54 % of the vector instructions that it could
// issue, a tenth of the matrix rate, 1 TB/s.
//
// Numerics: products of 16-bit values are exact in fp32, sums are fp32.  The integers (30 bits of a row's
// largest possible sum; Wg's scaled by a power of two per pixel) enter the products as three 16-bit
// operands, which hold all 24 bits of an fp32 number (in fp16 down to 2^-40 of the largest: for grad_key's sum over
// pixels a cell's weights are scaled to the largest of the step).  Points outside the band, every point of a pixel with operands or
// gradients that are not finite, and grad_query's terms where the key window holds a non-finite
// value are added one by one: a dense product would spread 0 * inf.
#include <utility>

#include "deform_region.hpp"
#include "kernels.hpp"

namespace sapa {

namespace dreg {

constexpr int NTB = 1024;                   // threads: 16 waves
// Window cells in LDS, by their number in the column's whole window (parent row 0's first) modulo RING: the blocks of 16
// cells that a pixel's sums are formed over are the same however the rows are split into segments.  A step's blocks reach up to two
// rows beyond its band; while its products are formed the row behind those comes in: nothing is read
// while it is written, and whether a row holds values that are not finite is known before a block reaches it.
constexpr int RING = 256, AHEAD = BROWS + 2;
static_assert(RING % 16 == 0 && RING >= 15 + (AHEAD + 1) * WWX && BC <= AHEAD * WWX, "no row comes in over one in use");
constexpr int CG = 64, DP = 32;             // value / key channels of a group, at most
constexpr int NVB = CG / 16, NKB = DP / 16;
// elements per window cell: 20 / 36 dwords, so that the 16 cells of an operand read fall on disjoint
// groups of banks, as do the rows of 32 bytes of a transposing read
constexpr int KSB = DP + 8, VSB = CG + 8;
// The step's 32 pixels: position 8 j + 4 a + b is pixel 4 j + b of row a, so that a load of 4 pixels of a
// plane is one piece in LDS and the 8 pixels of a lane of a matrix operand are 16 contiguous bytes
constexpr int PXS = 40;                     // elements per channel of the q / grad_out tile (20 dwords)
constexpr int OFS = 36;                     // elements per plane of the offsets' tile
constexpr int GQS = 36;                     // floats per channel of the grad_query tile

template <typename T>
struct BwdArgs {
    const T *grad_out, *q, *key, *value, *offset;
    T *grad_q, *grad_offset;                // may be null
    float *grad_key, *grad_value;           // channels-last fp32, accumulated into; may be null
    int Cq, C, H, W, P, G, strips_x, segments, rows, nblocks, per_xcd;
};

// 8 fp32 values as 16-bit operands that sum up to them
constexpr int PIECES = 3;
template <typename T>
__device__ __forceinline__ void pieces8(float (&f)[8], u32x4 (&p)[PIECES]) {
    typedef T tx8 __attribute__((ext_vector_type(8)));
#pragma unroll
    for (int i = 0; i < PIECES; ++i) {
        p[i] = u32x4{wm::pack2<T>(f[0], f[1]), wm::pack2<T>(f[2], f[3]), wm::pack2<T>(f[4], f[5]), wm::pack2<T>(f[6], f[7])};
        if (i + 1 < PIECES) {
            const tx8 h = __builtin_bit_cast(tx8, p[i]);
#pragma unroll
            for (int k = 0; k < 8; ++k) f[k] -= (float)h[k];
        }
    }
}

template <typename T>
__global__ void __launch_bounds__(NTB) __attribute__((amdgpu_waves_per_eu(4, 4)))
deform_bwd_region16_kernel(const BwdArgs<T> A) {
    __shared__ __attribute__((aligned(16))) T Kl[RING * KSB];           // key window [cell][channel]
    __shared__ __attribute__((aligned(16))) T Vl[RING * VSB];           // value window
    __shared__ __attribute__((aligned(16))) u32 Sl[32 * RS];            // Sim (fp32), then Wv
    __shared__ __attribute__((aligned(16))) u32 Gl[32 * RS];            // G' (fp32), then Wg
    __shared__ __attribute__((aligned(16))) T Ql[2][DP * PXS];          // q [channel][position], two steps in turn
    __shared__ __attribute__((aligned(16))) T Dl[2][CG * PXS];          // grad_out
    __shared__ __attribute__((aligned(16))) T Of[2][64 * OFS];          // offsets [plane][position], then their gradients
    __shared__ __attribute__((aligned(16))) float GQ[2][DP * GQS];      // grad_query, the two halves of the cells apart
    __shared__ __attribute__((aligned(16))) int ex[32];                 // a pixel's Wg is scaled by 2^(30 - ex)
    __shared__ u32 badpx[2];                // positions whose q or grad_out holds a value that is not finite
    __shared__ int kbad, fb_flag;           // the key window holds one; some point adds to grad_query by itself

    const int logical = (int)(blockIdx.x % 8) * A.per_xcd + (int)(blockIdx.x / 8);
    if (logical >= A.nblocks) return;
    const int rx = logical % A.strips_x, seg = (logical / A.strips_x) % A.segments;
    const int rest = logical / (A.strips_x * A.segments);
    const int g = rest % A.G, n = rest / A.G;

    const int H = A.H, W = A.W, P = A.P, Cq = A.Cq, C = A.C;
    const int hW = W * S, d = Cq / A.G, cg = C / A.G;
    const int p0 = seg * A.rows;                        // first row of parents
    const int nstep = H - p0 < A.rows ? H - p0 : A.rows;
    const int c00 = p0 * WWX;                           // number of the segment's first window cell
    const int x0 = rx * RW, wy0 = p0 - RCH, wx0 = rx * RPX - RCH;
    const long hpl = (long)H * W * (S * S);
    const bool two_k = cg > 32;                                         // G' in two contraction steps
    const bool want_q = A.grad_q != nullptr, want_o = A.grad_offset != nullptr;
    const bool want_k = A.grad_key != nullptr, want_v = A.grad_value != nullptr;
    // first planes of the group in the hi-res tensors
    const long dplane = (long)n * C + g * cg, qplane = (long)n * Cq + g * d, oplane = 2L * P * ((long)n * A.G + g);
    // The arguments, read again where they are used: the pointers of all tensors and their descriptors kept over
    // the whole loop do not fit the scalar registers (a fifth of all vector instructions then moved them
    // back from vector registers).
    auto args = [&]() __attribute__((always_inline)) {
#if defined(__HIP_DEVICE_COMPILE__)
        const auto *k = (const __attribute__((address_space(4))) BwdArgs<T> *)__builtin_amdgcn_kernarg_segment_ptr();
        asm volatile("" : "+s"(k));
        return k;
#else
        return &A;
#endif
    };
    auto rsrc = [](const void *p, long bytes) __attribute__((always_inline)) {
        return __builtin_amdgcn_make_buffer_rsrc((void *)p, 0, (int)bytes, 0x00020000);
    };

    // What a step needs from memory, fetched a step ahead, by wave: 0 .. 7 grad_out and the offsets, 8 .. 11 q
    // (a thread takes 4 pixels of a channel plane -- channel t / 8 of the kind, row (t / 4) % 2, pixels
    // 4 (t % 4) .. + 3), 12 .. 15 the window row that comes in (a thread: a piece of 16 bytes of a cell,
    // 4 of the key and 8 of the value).  Byte offsets of the first step and of image row 0; what lies
    // outside begins past the descriptor.
    const int t = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int uj = t & 3, ua = (t >> 2) & 1;
    const bool hires = wave < 12, isq = wave >= 8;
    const int uch = hires ? (t >> 3) - (isq ? 64 : 0) : 0, upos = 8 * uj + 4 * ua;
    const int piece = t - 768, pwl = piece / 12, pu = piece % 12, pc8 = 8 * (pu < 4 ? pu : pu - 4);
    const __amdgpu_buffer_rsrc_t rsa =
        !hires ? rsrc(A.key + (long)n * H * W * Cq, (long)H * W * Cq * 2)
               : isq ? rsrc(A.q + qplane * hpl, d * hpl * 2) : rsrc(A.grad_out + dplane * hpl, cg * hpl * 2);
    const __amdgpu_buffer_rsrc_t rsb = !hires ? rsrc(A.value + (long)n * H * W * C, (long)H * W * C * 2)
                                              : rsrc(A.offset + oplane * hpl, 2L * P * hpl * 2);
    u32 offa = OUTSIDE, offb = OUTSIDE;
    if (hires) {
        if (x0 + 4 * uj < hW) {
            const u32 at = (u32)((((long)2 * p0 + ua) * hW + x0 + 4 * uj) * 2);
            if (uch < (isq ? d : cg)) offa = (u32)uch * (u32)(hpl * 2) + at;
            if (!isq && uch < 2 * P) offb = (u32)uch * (u32)(hpl * 2) + at;
        }
    } else if (pwl < WWX && wx0 + pwl >= 0 && wx0 + pwl < W) {
        if (pu < 4 && pc8 < d) offa = (u32)(((wx0 + pwl) * Cq + g * d + pc8) * 2);
        if (pu >= 4 && pc8 < cg) offb = (u32)(((wx0 + pwl) * C + g * cg + pc8) * 2);
    }
    // (columns behind a row's end are the next row's)
    const bool tail = hires && x0 + 4 * uj + 2 >= hW;
    // A step's loads as they leave them.  Whatever joins two of them or moves one waits for it, and is done where they
    // are put into LDS; and all waves issue the same two loads, of which those of pixels use half, or registers
    // would be moved where the branches meet (each step waited for its own requests then, and for the stores
    // of the step before: the kernel 454 us, 426 so).
    struct Fetched {
        u32x4 a, b;                 // pixels, offsets; or a piece of the key, of the value (one of them zeros)
    };
    auto put_piece = [&](int row, u32x4 v) __attribute__((always_inline)) {
        const int at = (int)((u32)((p0 + row) * WWX + pwl) % RING);
        if (pu < 4) {
            *(u32x4 *)(Kl + at * KSB + pc8) = v;
            if (not_finite<T>(v)) kbad = 1;
        } else {
            *(u32x4 *)(Vl + at * VSB + pc8) = v;
        }
    };
    auto fetch = [&](int step, Fetched &f) __attribute__((always_inline)) {
        // (pixels: all of the offset in the lane's part, which the descriptor's check is made for dword by dword: where
        // a row ends two pixels into a piece, the tensor's last one runs over its end)
        const u32 lane_part = hires ? (u32)(step * 4 * hW) : 0u;
        const int gy = step + AHEAD - 1 < nstep + 2 * RCH + 1 ? wy0 + step + AHEAD - 1 : -1;
        const bool ok = hires ? step < nstep : gy >= 0 && gy < H;
        const u32 row = !hires && ok ? (u32)(gy * W) * 2u : 0u;  // (no row beside the image is ever an offset)
        f.a = __builtin_amdgcn_raw_buffer_load_b128(rsa, ok ? offa + lane_part : OUTSIDE, row * (u32)Cq, 0);
        f.b = __builtin_amdgcn_raw_buffer_load_b128(rsb, ok ? offb + lane_part : OUTSIDE, row * (u32)C, 0);
    };
    auto put = [&](int step, const Fetched &f) __attribute__((always_inline)) {
        const int buf = step & 1;
        if (hires) {
            const u32 hr[2] = {f.a[0], tail ? 0u : f.a[1]};
            if (!isq) {
                *(u32x2 *)(Dl[buf] + uch * PXS + upos) = u32x2{hr[0], hr[1]};
                *(u32x2 *)(Of[buf] + uch * OFS + upos) = u32x2{f.b[0], f.b[1]};
            } else {
                *(u32x2 *)(Ql[buf] + uch * PXS + upos) = u32x2{hr[0], hr[1]};
            }
            if (not_finite<T>(hr[0]) | not_finite<T>(hr[1])) {
                u32 m = 0;
#pragma unroll
                for (int e = 0; e < 4; ++e) m |= not_finite<T>((hr[e >> 1] >> (16 * (e & 1))) & 0xffffu) ? 1u << e : 0u;
                atomicOr(&badpx[buf], m << upos);
            }
        } else if (pwl < WWX) {
            put_piece(step + AHEAD - 1, u32x4{f.a[0] | f.b[0], f.a[1] | f.b[1], f.a[2] | f.b[2], f.a[3] | f.b[3]});
        }
    };

    // ---- the first step's band and the rows its blocks reach into; the rest of the ring is cleared
    if (t == 0) {
        badpx[0] = badpx[1] = 0u;
        kbad = 0;
        fb_flag = 0;
    }
    for (int i = AHEAD * WWX * (KSB / 8) + t; i < RING * (KSB / 8); i += NTB)
        ((u32x4 *)Kl)[(c00 + i / (KSB / 8)) % RING * (KSB / 8) + i % (KSB / 8)] = u32x4{0u, 0u, 0u, 0u};
    for (int i = AHEAD * WWX * (VSB / 8) + t; i < RING * (VSB / 8); i += NTB)
        ((u32x4 *)Vl)[(c00 + i / (VSB / 8)) % RING * (VSB / 8) + i % (VSB / 8)] = u32x4{0u, 0u, 0u, 0u};
    {
        const __amdgpu_buffer_rsrc_t kr = rsrc(A.key + (long)n * H * W * Cq, (long)H * W * Cq * 2);
        const __amdgpu_buffer_rsrc_t vr = rsrc(A.value + (long)n * H * W * C, (long)H * W * C * 2);
        constexpr int NPC = AHEAD * WWX, NK = (NPC * 4 + NTB - 1) / NTB, NV = (NPC * 8 + NTB - 1) / NTB;
        auto cell_pix = [&](int cell) __attribute__((always_inline)) {
            const int wr = cell / WWX, gy = wy0 + wr, gx = wx0 + cell % WWX;
            return cell < NPC && wr < nstep + 2 * RCH + 1 && gy >= 0 && gy < H && gx >= 0 && gx < W ? gy * W + gx : -1;
        };
        u32x4 kw[NK], vw[NV];
#pragma unroll
        for (int i = 0; i < NK; ++i) {
            const int u = i * NTB + t, cp = cell_pix(u >> 2), c8 = 8 * (u & 3);
            kw[i] = __builtin_amdgcn_raw_buffer_load_b128(kr, cp >= 0 && c8 < d ? (u32)((cp * Cq + g * d + c8) * 2) : OUTSIDE, 0, 0);
        }
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            const int u = i * NTB + t, cp = cell_pix(u >> 3), c8 = 8 * (u & 7);
            vw[i] = __builtin_amdgcn_raw_buffer_load_b128(vr, cp >= 0 && c8 < cg ? (u32)((cp * C + g * cg + c8) * 2) : OUTSIDE, 0, 0);
        }
        Fetched f;
        if (hires) fetch(0, f);
        __syncthreads();            // (the flags are clear)
        bool bad = false;
#pragma unroll
        for (int i = 0; i < NK; ++i) {
            const int u = i * NTB + t;
            bad |= not_finite<T>(kw[i]);
            if (u < NPC * 4) *(u32x4 *)(Kl + (c00 + (u >> 2)) % RING * KSB + 8 * (u & 3)) = kw[i];
        }
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            const int u = i * NTB + t;
            if (u < NPC * 8) *(u32x4 *)(Vl + (c00 + (u >> 3)) % RING * VSB + 8 * (u & 7)) = vw[i];
        }
        if (bad) kbad = 1;
        if (hires) put(0, f);
    }
    __syncthreads();

    const int lane = t & 63;
    // (the matrix view of the lanes is made anew in each phase: the addresses derived from it would be kept over the
    // whole loop, in registers that are not there)
    auto view = [&](int &mi, int &mk) __attribute__((always_inline)) {
        int l = lane;
        asm volatile("" : "+v"(l));
        mi = l & 15;
        mk = l >> 4;
    };
    // per-sample view: P <= 16 -> 16 lanes per pixel in the first 8 waves, else 32 lanes
    const bool narrow = P <= 16;
    const int pt = narrow ? (lane & 15) : (lane & 31);
    const int pos = narrow ? 4 * wave + (lane >> 4) : 2 * wave + (lane >> 5);
    const int px_x = x0 + 4 * (pos >> 3) + (pos & 3);
    // the sums of this wave's cell block, which is `mine` until the band has passed it, then mine + 16
    f32x4 Dv[NVB], Dk[NKB];
    int mine = band_base(p0) / 16 + ((wave - band_base(p0) / 16) & 15);
    auto clear = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int nb = 0; nb < NVB; ++nb) Dv[nb] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int nb = 0; nb < NKB; ++nb) Dk[nb] = f32x4{0.f, 0.f, 0.f, 0.f};
    };
    clear();
    // a power of two
    auto pow2 = [](int e) __attribute__((always_inline)) { return __builtin_ldexpf(1.f, e); };
    constexpr bool F16 = __is_same(T, f16_t);
    // Wv (and a row of Wg) enters its products times 2^WEXP: in fp16 as large as the type holds; bf16 has fp32's
    // range, and sums times 2^30 would leave it above 2^97
    constexpr int WEXP = F16 ? 15 : 0;
    constexpr float WIN = F16 ? 1.f / 32768.f : 1.f / 1073741824.f;

    // ... added to the gradients: lanes along 16 channels of a cell
    auto flush = [&]() __attribute__((always_inline)) {
        const auto *const a = args();
        float *const gv = a->grad_value + (long)n * H * W * C, *const gk = a->grad_key + (long)n * H * W * Cq;
        int lane_o = lane;
        asm volatile("" : "+v"(lane_o));
        const int ch = lane_o & 15;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int cell = 16 * mine + 4 * (lane_o >> 4) + r;       // of the column's window
            const int gy = cell / WWX - RCH, gx = wx0 + cell % WWX, pix = gy * W + gx;
            if (gy < 0 || gy >= H || gx < 0 || gx >= W) continue;
            if (want_v) {
#pragma unroll
                for (int nb = 0; nb < NVB; ++nb) {
                    const float v = Dv[nb][r] * pow2(-WEXP);
                    if (16 * nb + ch < cg && v != 0.f) unsafeAtomicAdd(gv + (pix * C + g * cg + 16 * nb + ch), v);
                }
            }
            if (want_k) {
#pragma unroll
                for (int nb = 0; nb < NKB; ++nb) {
                    const float v = Dk[nb][r];
                    if (16 * nb + ch < d && v != 0.f) unsafeAtomicAdd(gk + (pix * Cq + g * d + 16 * nb + ch), v);
                }
            }
        }
    };

    for (int step = 0; step < nstep; ++step) {
        const int buf = step & 1;
        Fetched next;
        fetch(step + 1, next);
        const int base = band_base(p0 + step), cb0 = base / 16;
        const bool exact_q = kbad != 0;

        // ---- A: wave = (16 positions, blocks of cells)
        {
            const int pxb = wave & 1;
            int mi, mk;
            view(mi, mk);
            union { u32x2 h[2]; u32x4 u; } aq, ad[2];
            const T *qt = Ql[buf] + (8 * mk + (mi >> 2)) * PXS + 16 * pxb + 4 * (mi & 3);
            const T *dt = Dl[buf] + (8 * mk + (mi >> 2)) * PXS + 16 * pxb + 4 * (mi & 3);
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                aq.h[h] = read_tr((const u32 *)(qt + 4 * h * PXS));
                ad[0].h[h] = read_tr((const u32 *)(dt + 4 * h * PXS));
                ad[1].h[h] = read_tr((const u32 *)(dt + (32 + 4 * h) * PXS));
            }
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const int cb = (wave >> 1) + 8 * i;
                if (cb >= NBLK) break;
                const int row = (int)((u32)(base + 16 * cb) % RING) + mi;
                const T *kp = Kl + row * KSB + 8 * mk, *vp = Vl + row * VSB + 8 * mk;
                const f32x4 sim = Mma<T>::k32(aq.u, *(const u32x4 *)kp, f32x4{0.f, 0.f, 0.f, 0.f});
                f32x4 gp = Mma<T>::k32(ad[0].u, *(const u32x4 *)vp, f32x4{0.f, 0.f, 0.f, 0.f});
                if (two_k) gp = Mma<T>::k32(ad[1].u, *(const u32x4 *)(vp + 32), gp);
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int at = (16 * pxb + 4 * mk + r) * RS + 16 * cb + mi;
                    ((float *)Sl)[at] = sim[r];
                    ((float *)Gl)[at] = gp[r];
                }
            }
        }
        __syncthreads();

        // ---- B (a pixel's rows are touched by its own lanes only, all in one wave, whose LDS operations
        // run in program order: gathers, the rows cleared, the adds -- no barrier between)
        bool fbq = false;               // this point adds to grad_query by itself
        float gl = 0.f, kh = 0.f, kw = 0.f;
        auto sample = [&](auto nl) __attribute__((always_inline)) {
            constexpr int NL = decltype(nl)::value;
            const bool live = (px_x < hW) & (pt < P);   // (both rows of a parent lie in the image)
            T *const op = Of[buf] + 2 * pt * OFS + pos;
            kw = (float)(px_x >> 1) + (float)op[0];
            kh = (float)(p0 + step) + (float)op[OFS];
            const bool guard = (kh > -1.f) & (kh < (float)H) & (kw > -1.f) & (kw < (float)W);
            const float fh = floor_(kh), fw = floor_(kw);
            const int hl = (int)fh + RCH, wl = (int)fw - wx0;       // of the column's window
            const bool in = live & guard & ((u32)(hl - (p0 + step)) <= (u32)(BROWS - 2)) & ((u32)wl <= (u32)(WWX - 2));
            const bool out = live & guard & !in;
            const float lh = kh - fh, lw = kw - fw, hh = 1.f - lh, hw = 1.f - lw;
            const bool use = in | out;
            const float w1 = use ? hh * hw : 0.f, w2 = use ? hh * lw : 0.f, w3 = use ? lh * hw : 0.f, w4 = use ? lh * lw : 0.f;
            const int cell = in ? hl * WWX + wl - base : 0;
            u32 *const srow = Sl + pos * RS, *const grow = Gl + pos * RS;
            float s1 = 0.f, s2 = 0.f, s3 = 0.f, s4 = 0.f, v1 = 0.f, v2 = 0.f, v3 = 0.f, v4 = 0.f;
            if (in) {
                const float *sp = (const float *)srow + cell, *gp = (const float *)grow + cell;
                s1 = sp[0], s2 = sp[1], s3 = sp[WWX], s4 = sp[WWX + 1];
                v1 = gp[0], v2 = gp[1], v3 = gp[WWX], v4 = gp[WWX + 1];
            }
            // (rare paths set up what they need from opaque copies, or it would be kept for them throughout)
            auto rare = [&](Tap<float> &tp, int &px) __attribute__((always_inline)) {
                float fkh = kh, fkw = kw;
                px = (2 * (p0 + step) + (pos >> 2 & 1)) * hW + px_x;
                asm volatile("" : "+v"(fkh), "+v"(fkw), "+v"(px));
                tp = Tap<float>{};
                tap_setup(fkh, fkw, H, W, tp);
            };
            if (__builtin_amdgcn_ballot_w64(out) != 0) {
                if (out) {
                    // the same eight products straight from global memory
                    Tap<float> tp;
                    int px;
                    rare(tp, px);
                    const auto *const a = args();
                    const T *kp = a->key + (long)n * H * W * Cq + g * d;
                    const T *qp = a->q + qplane * hpl + px;
                    for (int c = 0; c < d; ++c) {
                        const float z = (float)qp[c * hpl];
                        s1 = fma_(tp.m1 ? (float)kp[(long)tp.i1 * Cq + c] : 0.f, z, s1);
                        s2 = fma_(tp.m2 ? (float)kp[(long)tp.i2 * Cq + c] : 0.f, z, s2);
                        s3 = fma_(tp.m3 ? (float)kp[(long)tp.i3 * Cq + c] : 0.f, z, s3);
                        s4 = fma_(tp.m4 ? (float)kp[(long)tp.i4 * Cq + c] : 0.f, z, s4);
                    }
                    const T *vp = a->value + (long)n * H * W * C + g * cg;
                    const T *gp = a->grad_out + dplane * hpl + px;
                    for (int c = 0; c < cg; ++c) {
                        const float z = (float)gp[c * hpl];
                        v1 = fma_(tp.m1 ? (float)vp[(long)tp.i1 * C + c] : 0.f, z, v1);
                        v2 = fma_(tp.m2 ? (float)vp[(long)tp.i2 * C + c] : 0.f, z, v2);
                        v3 = fma_(tp.m3 ? (float)vp[(long)tp.i3 * C + c] : 0.f, z, v3);
                        v4 = fma_(tp.m4 ? (float)vp[(long)tp.i4 * C + c] : 0.f, z, v4);
                    }
                }
            }
            float lg = w1 * s1;
            lg = fma_(w2, s2, lg);
            lg = fma_(w3, s3, lg);
            lg = fma_(w4, s4, lg);
            // softmax over the pixel's points = the lanes pt < P of its group of NL lanes
            const float mx = reduce_lanes<true, NL>(pt < P ? lg : -__builtin_huge_valf());
            const float e = pt < P ? exp_(lg - mx) : 0.f;
            const float sum = reduce_lanes<false, NL>(e);
            float rs = __builtin_amdgcn_rcpf(sum);
            rs = fma_(fma_(-sum, rs, 1.f), rs, rs);
            const float att = e * rs;
            // its backward: gat = grad of the weight, gl = grad of the logit
            float gat = w1 * v1;
            gat = fma_(w2, v2, gat);
            gat = fma_(w3, v3, gat);
            gat = fma_(w4, v4, gat);
            const float dot = reduce_lanes<false, NL>(pt < P ? att * gat : 0.f);
            gl = pt < P ? att * (gat - dot) : 0.f;
            const float l1 = reduce_lanes<false, NL>(in ? __builtin_fabsf(gl) : 0.f);
            if (want_o && live) {
                // d / d(kw) and d / d(kh) of w1 x1 + w2 x2 + w3 x3 + w4 x4 (deform_qk_cuda_kernel.cu:98-133), of
                // the aggregation with the weight and of the logit with its gradient
                float gw = 0.f, gh = 0.f;
                if (use) {
                    const float dvw = -hh * v1 + hh * v2 - lh * v3 + lh * v4;
                    const float dvh = -hw * v1 - lw * v2 + hw * v3 + lw * v4;
                    const float dsw = -hh * s1 + hh * s2 - lh * s3 + lh * s4;
                    const float dsh = -hw * s1 - lw * s2 + hw * s3 + lw * s4;
                    gw = fma_(gl, dsw, att * dvw);
                    gh = fma_(gl, dsh, att * dvh);
                }
                op[0] = (T)gw;
                op[OFS] = (T)gh;
            }
            // the pixel's terms one by one: operands, weights or gradients that are not finite
            const bool slow = ((badpx[buf] >> pos & 1u) != 0u) | !(l1 < __builtin_huge_valf()) | (att != att);
            const bool direct = live & guard & (!in | slow);
            fbq = direct | (live & guard & exact_q);
            // the rows become Wv and Wg: cleared, then the corners' shares.  Wg's scale: |sum of any subset of a
            // row's entries| <= l1 < 2^e2
            int e2 = 0;
            (void)__builtin_frexpf(l1, &e2);
            if (pt == 0) ex[pos] = (l1 > 0.f) & !slow ? e2 : -126;
#pragma unroll
            for (int i = 0; i < (BC / 4 + NL - 1) / NL; ++i)
                if (i * NL + pt < BC / 4) {
                    *(u32x4 *)(srow + 4 * (i * NL + pt)) = u32x4{0u, 0u, 0u, 0u};
                    *(u32x4 *)(grow + 4 * (i * NL + pt)) = u32x4{0u, 0u, 0u, 0u};
                }
            if (in & !slow) {
                int *sp = (int *)srow + cell, *gp = (int *)grow + cell;
                const float sv = att * WSCALE, sg = __builtin_ldexpf(gl, 30 - e2);
                auto add = [](int *p, float v) __attribute__((always_inline)) {
                    __hip_atomic_fetch_add(p, (int)__builtin_rintf(v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                };
                add(sp, sv * w1);
                add(sp + 1, sv * w2);
                add(sp + WWX, sv * w3);
                add(sp + WWX + 1, sv * w4);
                add(gp, sg * w1);
                add(gp + 1, sg * w2);
                add(gp + WWX, sg * w3);
                add(gp + WWX + 1, sg * w4);
            }
            if (__builtin_amdgcn_ballot_w64(direct) != 0) {
                if (direct) {
                    // the reference's own way: one float atomic per term
                    Tap<float> tp;
                    int px;
                    rare(tp, px);
                    auto scatter = [&](const T *hi, float *low, int nch, int all, float sc) __attribute__((always_inline)) {
                        for (int c = 0; c < nch; ++c) {
                            const float tv = (float)hi[c * hpl] * sc;
                            if (tp.m1) unsafeAtomicAdd(low + (long)tp.i1 * all + c, tp.w1 * tv);
                            if (tp.m2) unsafeAtomicAdd(low + (long)tp.i2 * all + c, tp.w2 * tv);
                            if (tp.m3) unsafeAtomicAdd(low + (long)tp.i3 * all + c, tp.w3 * tv);
                            if (tp.m4) unsafeAtomicAdd(low + (long)tp.i4 * all + c, tp.w4 * tv);
                        }
                    };
                    const auto *const a = args();
                    if (want_v)
                        scatter(a->grad_out + dplane * hpl + px, a->grad_value + (long)n * H * W * C + g * cg, cg, C, att);
                    if (want_k)
                        scatter(a->q + qplane * hpl + px, a->grad_key + (long)n * H * W * Cq + g * d, d, Cq, gl);
                }
            }
            if (fbq) fb_flag = 1;
        };
        if (!narrow) sample(std::integral_constant<int, 32>{});
        else if (wave < 8) sample(std::integral_constant<int, 16>{});
        if (threadIdx.x == 0) badpx[buf ^ 1] = 0u;
        __syncthreads();

        // ---- C
        const bool any_fb = fb_flag != 0;
        const u32 bad = badpx[buf];
        int mi, mk;
        view(mi, mk);
        const int role = (wave - cb0) & 15;
        if (role < NBLK) {
            // the wave's cell block: sums over the step's 32 positions
            u32 z[4];                   // (rare: the 16-bit values of pixels that are not finite become 0)
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const u32 m = bad >> (8 * mk + 2 * k);
                z[k] = (m & 1u ? 0u : 0xffffu) | (m & 2u ? 0u : 0xffff0000u);
            }
            auto operand = [&](const T *p) __attribute__((always_inline)) {
                u32x4 b = *(const u32x4 *)p;
                if (bad != 0u) b = u32x4{b[0] & z[0], b[1] & z[1], b[2] & z[2], b[3] & z[3]};
                return b;
            };
            if (cb0 + role != mine) {
                flush();
                clear();
                mine = cb0 + role;
            }
            {
                if (want_v) {
                    const int *sp = (const int *)Sl + 8 * mk * RS + 16 * role + mi;
                    float f[8];
#pragma unroll
                    for (int k = 0; k < 8; ++k) f[k] = (float)sp[k * RS] * WIN;
                    u32x4 a[PIECES];
                    pieces8<T>(f, a);
                    // (two blocks of channels at a time: four do not fit the registers)
#pragma unroll
                    for (int nb = 0; nb < NVB; nb += 2) {
                        if (16 * nb >= cg) break;
                        const u32x4 b0 = operand(Dl[buf] + (16 * nb + mi) * PXS + 8 * mk);
                        const u32x4 b1 = operand(Dl[buf] + (16 * nb + 16 + mi) * PXS + 8 * mk);
#pragma unroll
                        for (int i = PIECES - 1; i >= 0; --i) {
                            Dv[nb] = Mma<T>::k32(a[i], b0, Dv[nb]);
                            Dv[nb + 1] = Mma<T>::k32(a[i], b1, Dv[nb + 1]);
                        }
                    }
                }
                if (want_k) {
                    const int *gp = (const int *)Gl + 8 * mk * RS + 16 * role + mi;
                    float f[8], down[4];
#pragma unroll
                    for (int k = 0; k < 8; ++k) f[k] = __builtin_ldexpf((float)gp[k * RS], ex[8 * mk + k] - 30);
                    if (F16) {
                        // (lanes of one mi hold the cell's 32 weights)
                        float m = 0.f;
#pragma unroll
                        for (int k = 0; k < 8; ++k) m = fmaxf(m, __builtin_fabsf(f[k]));
                        const wm::Fit fit = wm::fit<T>(wm::over_groups(m));
#pragma unroll
                        for (int k = 0; k < 8; ++k) f[k] *= fit.up;
#pragma unroll
                        for (int r = 0; r < 4; ++r) down[r] = __shfl(fit.down, 4 * mk + r);
                    }
                    u32x4 a[PIECES];
                    pieces8<T>(f, a);
#pragma unroll
                    for (int nb = 0; nb < NKB; ++nb) {
                        if (16 * nb >= d) break;
                        const u32x4 b = operand(Ql[buf] + (16 * nb + mi) * PXS + 8 * mk);
                        f32x4 acc = F16 ? f32x4{0.f, 0.f, 0.f, 0.f} : Dk[nb];
#pragma unroll
                        for (int i = PIECES - 1; i >= 0; --i) acc = Mma<T>::k32(a[i], b, acc);
                        if (F16) {
#pragma unroll
                            for (int r = 0; r < 4; ++r) acc[r] = fma_(acc[r], down[r], Dk[nb][r]);
                        }
                        Dk[nb] = acc;
                    }
                }
            }
        } else if (want_q) {
            // grad_query: wave = (16 positions, half of the band's cells)
            const int pxb = role & 1, kq = (role >> 1) & 1;
            f32x4 acc[NKB];
#pragma unroll
            for (int nb = 0; nb < NKB; ++nb) acc[nb] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int i = 0; i < BC / 64; ++i) {
                const int ks = kq * (BC / 64) + i;
                const u32x4 *ap = (const u32x4 *)(Gl + (16 * pxb + mi) * RS + 32 * ks + 8 * mk);
                const u32x4 w0 = ap[0], w1 = ap[1];
                float f[8];
#pragma unroll
                for (int k = 0; k < 8; ++k) f[k] = (float)(int)(k < 4 ? w0[k] : w1[k - 4]) * WIN;
                u32x4 a[PIECES];
                pieces8<T>(f, a);
                const T *kt = Kl + ((u32)(base + 32 * ks + 8 * mk) % RING + (mi >> 2)) * KSB + 4 * (mi & 3);
#pragma unroll
                for (int nb = 0; nb < NKB; ++nb) {
                    union { u32x2 h[2]; u32x4 u; } b;
                    b.h[0] = read_tr((const u32 *)(kt + 16 * nb));
                    b.h[1] = read_tr((const u32 *)(kt + 16 * nb + 4 * KSB));
#pragma unroll
                    for (int j = PIECES - 1; j >= 0; --j) acc[nb] = Mma<T>::k32(a[j], b.u, acc[nb]);
                }
            }
#pragma unroll
            for (int nb = 0; nb < NKB; ++nb) {
                f32x4 o;
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    o[r] = exact_q ? 0.f : __builtin_ldexpf(acc[nb][r], ex[16 * pxb + 4 * mk + r] - WEXP);
                *(f32x4 *)(GQ[kq] + (16 * nb + mi) * GQS + 16 * pxb + 4 * mk) = o;
            }
        }
        // (4 pixels of a plane per thread, where its offsets and its q came from)
        auto store = [&](const T *p, long bytes, u32 off, u32x2 v) __attribute__((always_inline)) {
            const __amdgpu_buffer_rsrc_t r = rsrc(p, bytes);
            const u32 at = off + (u32)(step * 4 * hW);
            if (hW % 4 == 0) {
                __builtin_amdgcn_raw_buffer_store_b64(v, r, off == OUTSIDE ? OUTSIDE : at, 0, 0);
            } else {            // (rows are even)
                __builtin_amdgcn_raw_buffer_store_b32(v[0], r, off == OUTSIDE ? OUTSIDE : at, 0, 0);
                __builtin_amdgcn_raw_buffer_store_b32(v[1], r, off == OUTSIDE || tail ? OUTSIDE : at + 4, 0, 0);
            }
        };
        // (the store behind the loads that it does not wait for)
        put(step + 1, next);
        if (want_o && wave < 8)
            store(args()->grad_offset + oplane * hpl, 2L * P * hpl * 2, offb, *(const u32x2 *)(Of[buf] + uch * OFS + upos));
        __syncthreads();
        if (any_fb) {
            if (fbq && want_q) {
                float fkh = kh, fkw = kw;
                asm volatile("" : "+v"(fkh), "+v"(fkw));
                Tap<float> tp = {};
                tap_setup(fkh, fkw, H, W, tp);
                const T *kp = args()->key + (long)n * H * W * Cq + g * d;
                for (int c = 0; c < d; ++c) {
                    const float k1 = tp.m1 ? (float)kp[(long)tp.i1 * Cq + c] : 0.f;
                    const float k2 = tp.m2 ? (float)kp[(long)tp.i2 * Cq + c] : 0.f;
                    const float k3 = tp.m3 ? (float)kp[(long)tp.i3 * Cq + c] : 0.f;
                    const float k4 = tp.m4 ? (float)kp[(long)tp.i4 * Cq + c] : 0.f;
                    float v = tp.w1 * k1;
                    v = fma_(tp.w2, k2, v);
                    v = fma_(tp.w3, k3, v);
                    v = fma_(tp.w4, k4, v);
                    __hip_atomic_fetch_add(GQ[0] + c * GQS + pos, gl * v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                }
            }
            if (threadIdx.x == 0) fb_flag = 0;
            __syncthreads();
        }
        if (want_q && isq && hires) {
            const f32x4 a = *(const f32x4 *)(GQ[0] + uch * GQS + upos), b = *(const f32x4 *)(GQ[1] + uch * GQS + upos);
            store(args()->grad_q + qplane * hpl, d * hpl * 2, offa,
                  u32x2{wm::pack2<T>(a[0] + b[0], a[1] + b[1]), wm::pack2<T>(a[2] + b[2], a[3] + b[3])});
        }
    }
    flush();
}

template <typename T>
static hipError_t launch_bwd(const void *grad_out, const void *q, const void *key, const void *value, const void *offset,
                             void *grad_q, void *grad_offset, float *grad_key, float *grad_value, int B, int Cq, int C,
                             int H, int W, int P, int G, hipStream_t st) {
    const int strips_x = (W + RPX - 1) / RPX;
    const long columns = (long)strips_x * G * B;
    // A workgroup fills a CU and walks down a strip of parent rows; its first band and the window rows beyond
    // its own cost about as much as 4 steps.  As many segments per column as make the whole shortest.
    constexpr int CUS = 256, OVER = 4;
    int segments = 1;
    long best = -1;
    for (int k = 1; k <= H && (k == 1 || columns * (k - 1) < 4 * CUS); ++k) {
        const int rows = (H + k - 1) / k;
        const long time = (columns * ((H + rows - 1) / rows) + CUS - 1) / CUS * (rows + OVER);
        if (best < 0 || time < best) best = time, segments = k;
    }
    const int rows = (H + segments - 1) / segments;
    segments = (H + rows - 1) / rows;
    const long nb = columns * segments;
    const int per_xcd = (int)((nb + 7) / 8);
    const BwdArgs<T> a = {(const T *)grad_out, (const T *)q, (const T *)key, (const T *)value, (const T *)offset,
                          (T *)grad_q, (T *)grad_offset, grad_key, grad_value, Cq, C, H, W, P, G, strips_x, segments, rows,
                          (int)nb, per_xcd};
    hipLaunchKernelGGL(deform_bwd_region16_kernel<T>, dim3(per_xcd * 8), dim3(NTB), 0, st, a);
    return hipGetLastError();
}

}  // namespace dreg

// f16 / bf16 tensors, s = 2, up to 32 points, groups of whole 16-byte pieces with at most 32 query / key and
// 64 value channels.
bool deform_bwd_region16_serves(int B, int Cq, int C, int H, int W, int P, int s, int G, int dtype) {
    if ((dtype != 2 && dtype != 3) || s != 2 || P < 1 || P > 32) return false;
    if (G <= 0 || Cq % G != 0 || C % G != 0) return false;
    const int d = Cq / G, cg = C / G;
    if (d % 8 != 0 || d > 32 || cg % 8 != 0 || cg > 64) return false;
    const long plane = (long)H * W * 2, hpl = plane * 4;
    // workgroups; one image's key / value, a group's planes of the hi-res tensors, in bytes
    return (long)B * G * ((W + dreg::RPX - 1) / dreg::RPX) * H <= (1L << 30) && plane * Cq < (1L << 31) && plane * C < (1L << 31) && 64 * hpl < (1L << 31);
}

// key_cl, value_cl: channels-last copies, aligned to 16 bytes; grad_key, grad_value: fp32 [B, H, W, channels],
// accumulated into; any gradient may be null.  The hi-res tensors begin on dwords.
hipError_t deform_bwd_region16_launch(const void *grad_out, const void *q, const void *key_cl, const void *value_cl,
                                      const void *offset, void *grad_q, void *grad_offset, float *grad_key,
                                      float *grad_value, int B, int Cq, int C, int H, int W, int P, int s, int G,
                                      int dtype, hipStream_t st) {
    if (!deform_bwd_region16_serves(B, Cq, C, H, W, P, s, G, dtype)) return hipErrorNotSupported;
    if (((uintptr_t)grad_out | (uintptr_t)q | (uintptr_t)offset | (uintptr_t)grad_q | (uintptr_t)grad_offset) % 4 != 0 ||
        ((uintptr_t)key_cl | (uintptr_t)value_cl) % 16 != 0)
        return hipErrorNotSupported;
    return dtype == 2 ? dreg::launch_bwd<f16_t>(grad_out, q, key_cl, value_cl, offset, grad_q, grad_offset, grad_key, grad_value, B, Cq, C, H, W, P, G, st)
                      : dreg::launch_bwd<bf16_t>(grad_out, q, key_cl, value_cl, offset, grad_q, grad_offset, grad_key, grad_value, B, Cq, C, H, W, P, G, st);
}

}  // namespace sapa
