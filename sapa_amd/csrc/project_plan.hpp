// How the tiles of a projection, or of two in one launch, are spread over waves and workgroups.  Host arithmetic
// alone (no HIP), so that it can be looked over for all sizes without a GPU.
#pragma once

namespace sapa {
namespace project {

// How a projection's tiles are spread: tiles per wave, waves per workgroup that have some, workgroups per image
struct Spread {
    long per, blocks[2];
    int waves;
};
// One workgroup is resident per CU (its weight planes fill most of the LDS) and the part has
// 256 CUs: two full rounds of workgroups where that leaves a wave 8 tiles or more (6 of 12 waves), else one
// (16 images: 200x336 pixels 301 us in two rounds against 315 in one; 100x168 pixels 71 us in
// one round against 98 in 272 workgroups; 256 -> 288, 8 images 128x128, 8 waves, 119 us in one against 130)
inline Spread plan32(const long (&tiles)[2], long sets, int nw) {
    const long ntiles = tiles[0] + tiles[1];
    const long slots = 256;
    long blocks = 2 * slots / sets > 1 ? 2 * slots / sets : 1;
    long per = (ntiles + nw * blocks - 1) / (nw * blocks);
    if (per < (nw == 8 ? 8 : 6)) {
        blocks = slots / sets > 1 ? slots / sets : 1;
        per = (ntiles + nw * blocks - 1) / (nw * blocks);
    }
    // ... and as few waves per workgroup as cover the image in that many tiles each, so that no workgroup of the
    // round is missing (240 workgroups of 12 waves else 256 of 11; 512 -> 72, 2 images 100x168, 8 waves in 198
    // workgroups 35.8 us, 7 in 228 31.3; fewer tiles than the chip has room for: a wave's matrix instructions are not
    // queued behind a second wave's; 4 images of 33x20 pixels, 256 -> 128 / 288: SAPA-D module 113 -> 104 us), but over
    // several tiles each not with less than 6 of 8 (128 -> 32, 16 images 50x84: 5 waves 12.4 us, 8 11.7)
    int waves = (int)((ntiles + blocks * per - 1) / (blocks * per));
    waves = waves < 1 ? 1 : waves > nw ? nw : waves;
    if (nw == 8 && per > 1 && waves < 6) waves = nw;
    // Two features end in a workgroup that is not full each: more waves, then tiles, per workgroup until an image has no
    // more workgroups than its share of the round (one each at least; fp32, 256 -> 64, modules' features with moments and
    // folds: 8 images 32x32 in 264 workgroups, two rounds, 42.4 us, in 224 32.5, a launch each 43.6; 16 of 14x14 in 272
    // 38.0, in 192 28.9; channels-last 15 of 18x30 in 270 51.5, in 225 40.7)
    Spread s{per, {0, 0}, waves};
    for (;;) {
        for (int i = 0; i < 2; ++i) s.blocks[i] = (tiles[i] + s.waves * s.per - 1) / (s.waves * s.per);
        if (s.blocks[0] + s.blocks[1] <= (blocks > 2 ? blocks : 2)) return s;
        if (s.waves < nw) ++s.waves;
        else ++s.per;
    }
}

// Workgroups of 4 waves: one round of 512 (and what rounding up per image and feature adds); a tile per wave only where
// all of them are resident, `resident` on each of 256 CUs (us with 2 tiles per wave at least and so, modules: 256
// channels, 1 image 50x84, planes 41 -> 36, 2 of 48x48 38 -> 34, 512 channels, 2 of 32x32 42 -> 36; in two rounds, SAPA-D
// channels-last, 512 channels, 2 of 32x32, 53 -> 56).
inline Spread plan16(const long (&tiles)[2], long sets, int resident) {
    const long all = (tiles[0] + tiles[1]) * sets;
    Spread s{(all + 4L * 512 - 1) / (4L * 512), {0, 0}, 4};
    for (;; ++s.per) {
        for (int i = 0; i < 2; ++i) s.blocks[i] = (tiles[i] + 4 * s.per - 1) / (4 * s.per);
        if (s.per > 1 || (s.blocks[0] + s.blocks[1]) * sets <= 256L * resident) return s;
    }
}

}  // namespace project
}  // namespace sapa
