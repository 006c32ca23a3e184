// Fused SAPA-D (deform_qk -> softmax -> deform_av) of contiguous fp32 tensors, up_factor 2 and at most 9
// sample points: every sample is gathered from a window in LDS, a pixel's points stay in registers.
//
// As in sapa_d_lds.hip a workgroup owns TPW x TPH low-res parents of one (image, group), a thread one
// output pixel, and the window -- the tile plus 4 cells on every side, one more behind for the +1 corners --
// passes through LDS in chunks of 16 channels as [cell][16 channels], zeros outside the image.  What differs
// is where the rest lives.  A sample's place and fractions and its logit (then weight) are registers, formed
// once: that kernel fetched the offsets again and formed floor, guard and window test again for each chunk of
// channels (6 times with 32 query and 64 value channels: a third of its vector instructions), and another
// third went into staging element by element.  Here a thread stages four channels of a cell at a time through
// four buffer loads whose offsets are fixed for the whole kernel, requested a chunk ahead, into the second of two
// buffers: one barrier per chunk.  A sample outside the image or the window points at cells that are always
// zero, so the channel loops have no selects; the rare one inside the image but outside the window comes from
// memory.  It is added at its point's place in the order: waves that have one aggregate in a loop over the points.
//
// Arithmetic and order of sums are those of sapa_d_lds.hip, bit for bit (reference:
// deformsapa/deformsapa/src/cuda/deform_qk_cuda_kernel.cu:180-193, deform_av_cuda_kernel.cu:178-192).
#include "deform_tap.hpp"
#include "kernels.hpp"

namespace sapa {

namespace dgather {

typedef unsigned u32;
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int S = 2, HR = 4, CH = 16;
constexpr int CST = CH + 4;                         // floats per cell: 16-byte reads spread over all bank groups
constexpr u32 OUTSIDE = 0x80000000u;                // a buffer offset beyond any extent
// a sample in the image, but not in the window: the rows and columns of its corners that are in the image, and the index
// (y + 1) W + x + 1 of its low corner (below 2^26 where a group's planes are within a descriptor's reach)
constexpr u32 FAR = 0x80000000u, FAR_Y0 = 1u << 30, FAR_Y1 = 1u << 29, FAR_X0 = 1u << 28, FAR_X1 = 1u << 27, FAR_INDEX = FAR_X1 - 1;

__device__ __forceinline__ __amdgpu_buffer_rsrc_t planes(const void *p, long bytes) {
    return __builtin_amdgcn_make_buffer_rsrc((void *)p, 0, (int)bytes, 0x00020000);
}

// PM: the most sample points
template <int PM, int TPW, int TPH>
__global__ void __launch_bounds__(TPW * TPH * S * S) __attribute__((amdgpu_waves_per_eu(4, 4)))
deform_gather_kernel(const float *__restrict__ q, const float *__restrict__ key, const float *__restrict__ value,
                     const float *__restrict__ offset, float *__restrict__ out, int Cq, int C, int H, int W, int P,
                     int G, int olayout, int tiles_x, int tiles_y, int nslices, int slice_chunks, int nblocks, int per_xcd) {
    constexpr int NT = TPW * TPH * S * S, TXP = TPW * S;
    constexpr int WW = TPW + 2 * HR + 1, WH = TPH + 2 * HR + 1, WIN = WW * WH;
    constexpr int RS = WW * CST;                    // floats between window rows
    constexpr int NOWHERE = WIN * CST;              // where samples that contribute nothing read zeros
    constexpr int BUF = NOWHERE + RS + CST + CH;
    constexpr int TASKS = WIN * (CH / 4), NST = (TASKS + NT - 1) / NT;

    __shared__ __attribute__((aligned(16))) float lds[2 * BUF];

    const int logical = (int)(blockIdx.x % 8) * per_xcd + (int)(blockIdx.x / 8);
    if (logical >= nblocks) return;
    // logical = tile * nslices + slice of the value chunks: a tile's slices meet in an XCD's L2
    const int slice = logical % nslices, tile = logical / nslices;
    const int tx = tile % tiles_x;
    const int ty = (tile / tiles_x) % tiles_y;
    const int g = (tile / (tiles_x * tiles_y)) % G;
    const int b = tile / (tiles_x * tiles_y * G);

    const int tid = threadIdx.x;
    const int hH = H * S, hW = W * S, GP = G * P, d = Cq / G, cg = C / G;
    const u32 lplane = (u32)(H * W) * 4u, hplane = (u32)(hH * hW) * 4u;         // bytes
    const int qw = tx * TXP + tid % TXP, qh = ty * TPH * S + tid / TXP;
    const bool active = qw < hW && qh < hH;
    // idle threads of a partial tile read through clamped coordinates
    const int cw = qw < hW ? qw : hW - 1, chh = qh < hH ? qh : hH - 1;
    const u32 pix = (u32)(chh * hW + cw) * 4u;
    const float ph = (float)(chh / S), pw = (float)(cw / S);
    const int wx0 = tx * TPW - HR, wy0 = ty * TPH - HR;
    const float *const qg = q + ((long)b * Cq + (long)g * d) * (hplane / 4);
    const float *const kg = key + ((long)b * Cq + (long)g * d) * (lplane / 4);
    const float *const vg = value + ((long)b * C + (long)g * cg) * (lplane / 4);
    const int nK = (d + CH - 1) / CH, firstV = slice * slice_chunks, leftV = (cg + CH - 1) / CH - firstV;
    const int ntot = nK + (leftV < slice_chunks ? leftV : slice_chunks);

    // ---- staging: task i of a thread is four channels of one cell ----
    u32 from[NST];
    int to[NST];
#pragma unroll
    for (int i = 0; i < NST; ++i) {
        const int task = tid + i * NT, four = task / WIN, cell = task % WIN;
        const int gy = wy0 + cell / WW, gx = wx0 + cell % WW;
        const bool ok = task < TASKS && gy >= 0 && gy < H && gx >= 0 && gx < W;
        from[i] = ok ? (u32)(4 * four) * lplane + (u32)(gy * W + gx) * 4u : OUTSIDE;
        to[i] = task < TASKS ? cell * CST + 4 * four : -1;
    }
    f32x4 st[NST];
    auto stage_load = [&](int j) __attribute__((always_inline)) {
        const bool is_key = j < nK;
        const int c0 = (is_key ? j : j - nK + firstV) * CH, nc = (is_key ? d : cg) - c0;
        const __amdgpu_buffer_rsrc_t r = planes((const char *)(is_key ? kg : vg) + (long)c0 * lplane, (long)(nc < CH ? nc : CH) * lplane);
#pragma unroll
        for (int i = 0; i < NST; ++i) {
            u32 at = from[i];                       // (opaque: or all four sums are kept)
            asm volatile("" : "+v"(at));
#pragma unroll
            for (int e = 0; e < 4; ++e)
                st[i][e] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, at + (u32)e * lplane, 0, 0));
        }
    };
    auto stage_store = [&](int j) __attribute__((always_inline)) {
        float *const dst = lds + (j & 1) * BUF;
#pragma unroll
        for (int i = 0; i < NST; ++i)
            if ((i + 1) * NT <= TASKS || to[i] >= 0) *(f32x4 *)(dst + to[i]) = st[i];
    };
    // channel c of the chunk's queries of this pixel; those behind the last are 0
    const __amdgpu_buffer_rsrc_t rq = planes(qg, (long)d * hplane);
    auto load_q = [&](int j, float (&v)[CH]) __attribute__((always_inline)) {
        u32 at = (u32)(j * CH) * hplane;
        const u32 end = (u32)d * hplane;
#pragma unroll
        for (int c = 0; c < CH; ++c) {
            v[c] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rq, pix, at, 0));
            at += at + hplane < end ? hplane : 0u;  // (no plane behind the last)
        }
    };
    auto clear_q = [&](int j, float (&v)[CH]) __attribute__((always_inline)) {
        const int nc = d - j * CH;
        if (nc < CH)
#pragma unroll
            for (int c = 0; c < CH; ++c) v[c] = c < nc ? v[c] : 0.f;
    };

    stage_load(0);
    // ---- the samples ----
    float lh[PM], lw[PM], lg[PM];
    int at[PM];                                     // place in the window (NOWHERE: none), or FAR and where in the image
    u32 far_wave = 0;                               // points with a sample in the image, but not in the window
    {
        const OffsetRef<float> op = offset_ref(offset, olayout, (long)b * GP + (long)g * P, chh, cw, S, H, W);
        float ow[PM], oh[PM];
#pragma unroll
        for (int p = 0; p < PM; ++p) {
            const int pp = p < P ? p : P - 1;
            ow[p] = op.base[(long)(2 * pp) * op.stride];
            oh[p] = op.base[(long)(2 * pp + 1) * op.stride];
        }
#pragma unroll
        for (int p = 0; p < PM; ++p) {
            const float kh = ph + oh[p], kw = pw + ow[p];
            const bool guard = active && p < P && kh > -1.f && kh < (float)H && kw > -1.f && kw < (float)W;
            const float fh = floor_(kh), fw = floor_(kw);
            const int hl = (int)fh - wy0, wl = (int)fw - wx0;
            const bool in = guard && hl >= 0 && hl <= WH - 2 && wl >= 0 && wl <= WW - 2;
            at[p] = in ? hl * RS + wl * CST : NOWHERE;
            lh[p] = guard ? kh - fh : 0.f;
            lw[p] = guard ? kw - fw : 0.f;
            lg[p] = 0.f;
            if (guard && !in) {
                const int y = (int)fh, x = (int)fw;             // -1 .. H - 1, -1 .. W - 1
                at[p] = (int)(FAR | (y >= 0 ? FAR_Y0 : 0u) | (y + 1 < H ? FAR_Y1 : 0u) | (x >= 0 ? FAR_X0 : 0u) |
                              (x + 1 < W ? FAR_X1 : 0u) | (u32)((y + 1) * W + x + 1));
            }
            far_wave |= __ballot(at[p] < 0) ? 1u << p : 0u;
        }
    }
    // the sample of code `code` (at[p] < 0) and fractions fy, fx in the channels c0 .. c0 + 15: add(c, value).  What bounds
    // it is the way to the cache and back: four channels at a time, 16 loads in flight, its place kept from the start (one
    // channel at a time behind the offsets fetched again, 8 images 64x64, C=256, 9 points, offsets of standard deviation
    // 2 / 3 / 4 / 6: 576 / 792 / 672 / 884 us, 235 / 306 / 449 / 803 so; sapa_d_lds.hip 520 / 601 / 619 / 857)
    auto far_sample = [&](int code, float fy, float fx, const float *src, int c0, int channels, auto &&add) __attribute__((always_inline)) {
        const __amdgpu_buffer_rsrc_t r = planes((const char *)src + (long)c0 * lplane, (long)(channels - c0 < CH ? channels - c0 : CH) * lplane);
        const u32 u = (u32)code, first = ((u & FAR_INDEX) - (u32)(W + 1)) * 4u;
        const bool y0 = u & FAR_Y0, y1 = u & FAR_Y1, x0 = u & FAR_X0, x1 = u & FAR_X1;
        u32 i1 = y0 && x0 ? first : OUTSIDE, i2 = y0 && x1 ? first + 4u : OUTSIDE;
        u32 i3 = y1 && x0 ? first + 4u * (u32)W : OUTSIDE, i4 = y1 && x1 ? first + 4u * (u32)W + 4u : OUTSIDE;
        const float hh = 1.f - fy, hw = 1.f - fx;
        const float w1 = hh * hw, w2 = hh * fx, w3 = fy * hw, w4 = fy * fx;
#pragma unroll
        for (int c4 = 0; c4 < CH; c4 += 4) {
            float v[4][4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                v[e][0] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, i1, 0, 0));
                v[e][1] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, i2, 0, 0));
                v[e][2] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, i3, 0, 0));
                v[e][3] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, i4, 0, 0));
                i1 += lplane, i2 += lplane, i3 += lplane, i4 += lplane;
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                float val = w1 * v[e][0];
                val = fma_(w2, v[e][1], val);
                val = fma_(w3, v[e][2], val);
                val = fma_(w4, v[e][3], val);
                add(c4 + e, val);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    // of at, lh, lw and lg those of point p
    auto point = [&](int p, int &code, float &fy, float &fx, float &l) __attribute__((always_inline)) {
        code = at[0], fy = lh[0], fx = lw[0], l = lg[0];
#pragma unroll
        for (int i = 1; i < PM; ++i) {
            const bool here = i == p;
            code = here ? at[i] : code, fy = here ? lh[i] : fy, fx = here ? lw[i] : fx, l = here ? lg[i] : l;
        }
    };

    for (int i = tid; i < 2 * (BUF - NOWHERE); i += NT)
        lds[i < BUF - NOWHERE ? NOWHERE + i : 2 * NOWHERE + i] = 0.f;
    float qv[CH];
    load_q(0, qv);
    stage_store(0);

    // ---- logits ----
    for (int j = 0; j < nK; ++j) {
        stage_load(j + 1);
        __syncthreads();
        clear_q(j, qv);
        const float *const win = lds + (j & 1) * BUF;
#pragma unroll
        for (int p = 0; p < PM; ++p) {
            if (p >= P) continue;
            const float *const wp = win + (at[p] < 0 ? NOWHERE : at[p]);
            float fy = lh[p], fx = lw[p];
            asm volatile("" : "+v"(fy), "+v"(fx));
            const float hh = 1.f - fy, hw = 1.f - fx;
            const float w1 = hh * hw, w2 = hh * fx, w3 = fy * hw, w4 = fy * fx;
            float acc = lg[p];
#pragma unroll
            for (int c4 = 0; c4 < CH; c4 += 4) {
                const f32x4 a1 = *(const f32x4 *)(wp + c4), a2 = *(const f32x4 *)(wp + CST + c4);
                const f32x4 a3 = *(const f32x4 *)(wp + RS + c4), a4 = *(const f32x4 *)(wp + RS + CST + c4);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    float val = w1 * a1[e];
                    val = fma_(w2, a2[e], val);
                    val = fma_(w3, a3[e], val);
                    val = fma_(w4, a4[e], val);
                    acc = fma_(val, qv[c4 + e], acc);
                }
            }
            // (a query that is not finite times the zeros of a sample that contributes nothing)
            lg[p] = (u32)at[p] < (u32)NOWHERE ? acc : lg[p];
            __builtin_amdgcn_sched_barrier(0);
        }
        for (u32 left = far_wave; left; left &= left - 1) {
            const int p = __builtin_ctz(left);
            int code;
            float fy, fx, acc;
            point(p, code, fy, fx, acc);
            if (code < 0) {
                far_sample(code, fy, fx, kg, j * CH, d, [&](int c, float val) __attribute__((always_inline)) { acc = fma_(val, qv[c], acc); });
#pragma unroll
                for (int i = 0; i < PM; ++i) lg[i] = i == p ? acc : lg[i];
            }
        }
        if (j + 1 < nK) load_q(j + 1, qv);
        stage_store(j + 1);
    }

    // ---- softmax over the points (one outside the image keeps logit 0 and takes part) ----
    {
        float m = lg[0];
#pragma unroll
        for (int p = 1; p < PM; ++p) m = p < P ? max_(m, lg[p]) : m;
        float sum = 0.f;
#pragma unroll
        for (int p = 0; p < PM; ++p) {
            lg[p] = exp_(lg[p] - m);
            sum = p < P ? sum + lg[p] : sum;
        }
        const float inv = 1.f / sum;
        // (a sample that contributes nothing: its weight times the zeros may not be NaN)
#pragma unroll
        for (int p = 0; p < PM; ++p) lg[p] = at[p] != NOWHERE ? lg[p] * inv : 0.f;
    }

    // ---- aggregation ----
    const __amdgpu_buffer_rsrc_t ro = planes(out + ((long)b * C + (long)g * cg) * (hplane / 4), (long)cg * hplane);
    const u32 opix = active ? pix : OUTSIDE;
    for (int j = nK; j < ntot; ++j) {
        if (j + 1 < ntot) stage_load(j + 1);
        __syncthreads();
        const float *const win = lds + (j & 1) * BUF;
        const int c0 = (j - nK + firstV) * CH, nc = cg - c0;
        float o[CH];
#pragma unroll
        for (int c = 0; c < CH; ++c) o[c] = 0.f;
        // sample of weight wa from the window, of place `cell` in it and fractions fy, fx
        auto window_sample = [&](int cell, float fy, float fx, float wa) __attribute__((always_inline)) {
            const float *const wp = win + cell;
            const float hh = 1.f - fy, hw = 1.f - fx;
            const float w1 = hh * hw, w2 = hh * fx, w3 = fy * hw, w4 = fy * fx;
#pragma unroll
            for (int c4 = 0; c4 < CH; c4 += 4) {
                const f32x4 a1 = *(const f32x4 *)(wp + c4), a2 = *(const f32x4 *)(wp + CST + c4);
                const f32x4 a3 = *(const f32x4 *)(wp + RS + c4), a4 = *(const f32x4 *)(wp + RS + CST + c4);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    float val = w1 * a1[e];
                    val = fma_(w2, a2[e], val);
                    val = fma_(w3, a3[e], val);
                    val = fma_(w4, a4[e], val);
                    o[c4 + e] = fma_(val, wa, o[c4 + e]);
                }
            }
        };
        if (far_wave == 0) {
#pragma unroll
            for (int p = 0; p < PM; ++p) {
                if (p >= P) continue;
                // (opaque: the weights of all samples kept over the loop do not fit the registers)
                float fy = lh[p], fx = lw[p];
                asm volatile("" : "+v"(fy), "+v"(fx));
                window_sample(at[p], fy, fx, lg[p]);
                __builtin_amdgcn_sched_barrier(0);
            }
        } else {
            // a sample beyond the window is added where its point stands: a loop with one body for all points, or
            // the code of such a sample would be there nine times
#pragma unroll 1
            for (int p = 0; p < P; ++p) {
                int code;
                float fy, fx, wa;
                point(p, code, fy, fx, wa);
                window_sample(code < 0 ? NOWHERE : code, fy, fx, code < 0 ? 0.f : wa);
                if (code < 0)
                    far_sample(code, fy, fx, vg, c0, cg, [&](int c, float val) __attribute__((always_inline)) { o[c] = fma_(val, wa, o[c]); });
            }
        }
        u32 plane = (u32)c0 * hplane;
        asm volatile("" : "+s"(plane));
#pragma unroll
        for (int c = 0; c < CH; ++c) {
            if (c < nc) __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(o[c]), ro, opix, plane, 0);
            plane += hplane;
        }
        if (j + 1 < ntot) stage_store(j + 1);
    }
}

template <int PM>
static hipError_t launch(const void *q, const void *key, const void *value, const void *offset, void *out, int B, int Cq, int C,
                         int H, int W, int P, int G, int olayout, hipStream_t st) {
    constexpr int TPW = 16, TPH = 8;
    const int tiles_x = (W + TPW - 1) / TPW, tiles_y = (H + TPH - 1) / TPH;
    const long tiles = (long)tiles_x * tiles_y * G * B;
    const int chunks = (C / G + CH - 1) / CH;
    // Fewer tiles than CUs: a workgroup's time is a chain of one step per 16 channels, so the value channels are split over
    // several workgroups per tile, each forming the weights again, up to one per CU (C=256, 9 points, one slice / two / four:
    // 1 image 16x16, 8 tiles, 37 / 27 / 22 us; 4 of 32x32, 128 tiles, 39 / 30 / 37; 2 of 64x64, 256 tiles, 43 / 47 / 66)
    long want = tiles > 0 ? 256 / tiles : 1;
    want = want < 1 ? 1 : want > chunks ? chunks : want;
    const int slice_chunks = (int)((chunks + want - 1) / want), nslices = (chunks + slice_chunks - 1) / slice_chunks;
    const long nb = tiles * nslices;
    if (nb > (1L << 30)) return hipErrorNotSupported;
    const int per_xcd = (int)((nb + 7) / 8);
    hipLaunchKernelGGL((deform_gather_kernel<PM, TPW, TPH>), dim3(per_xcd * 8), dim3(TPW * TPH * S * S), 0, st,
                       (const float *)q, (const float *)key, (const float *)value, (const float *)offset, (float *)out, Cq, C, H,
                       W, P, G, olayout, tiles_x, tiles_y, nslices, slice_chunks, (int)nb, per_xcd);
    return hipGetLastError();
}

}  // namespace dgather

// Up to 9 points: a point takes four registers, and with 12 they spill at the 16 waves per CU that two windows of 36 KB
// allow; from 13 the matrix form serves default calls.  Images at most 8 cells wide would leave half of each tile idle
// (8 x 8 tiles of sapa_d_lds.hip).  A group's planes lie within the reach of a buffer descriptor's 32-bit offsets.
hipError_t deform_gather_launch(const void *q, const void *key, const void *value, const void *offset, void *out, int B, int Cq,
                                int C, int H, int W, int P, int s, int G, int olayout, int dtype, hipStream_t st) {
    if (dtype != 0 || s != dgather::S || P < 1 || P > 9 || W <= 8) return hipErrorNotSupported;
    const long most = Cq > C ? Cq / G : C / G;
    if (most * H * W * (s * s) * 4L >= (1L << 31) || (most + 16) * (long)H * W * 4L >= (1L << 31)) return hipErrorNotSupported;
    if (P <= 5) return dgather::launch<5>(q, key, value, offset, out, B, Cq, C, H, W, P, G, olayout, st);
    return dgather::launch<9>(q, key, value, offset, out, B, Cq, C, H, W, P, G, olayout, st);
}

}  // namespace sapa
