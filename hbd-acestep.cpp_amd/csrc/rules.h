// rules.h -- dispatch rules as plain host functions of sizes, so that they can be
// checked without a GPU. Each says what was measured on both sides of its line.
#pragma once

#include <cstdint>

namespace mi {

// Q8_0 product of one row of x (nbk key blocks, ng groups of 64 weight rows): whether the
// prologue, the product and the key sum are one launch of a workgroup per row group. A
// wave takes an eighth of the keys (up to a block per split more), in sets of 4 blocks.
// us with the norm prologue, three launches / one, weights of 400 MB in turn:
//   1024 keys: 64 groups 8.0 / 5.6, 96 8.3 / 5.7, 256 7.4 / 6.5, 512 10.0 / 9.3, 2370 29.8 / 35.0
//   2048 keys: 96 groups 11.0 / 8.4, 192 13.4 / 9.5, 512 16.1 / 14.4; 6144 keys: 32 groups 12.0 / 14.2
// Past 256 row groups the product has no second sum to save, and a second round of
// workgroups stands against one: there it wins only with the sets near full (32 and 64
// blocks 0.93, 24 0.99, 48 0.99; 8 blocks 1.11, 16 1.03, 33 1.07, 40 1.07). Up to 128 row
// groups 33-80 blocks would win too (64 blocks 32 groups 7.8 / 7.2, 80 blocks 96 groups
// 11.5 / 9.2; 96 blocks 16 groups 8.9 / 9.3) but keep the three launches.
inline bool mmv_one_launch(uint32_t nbk, uint32_t ng) {
    if (ng > 512 || nbk > 64 || (nbk > 32 && ng < 128)) {
        return false;
    }
    const uint32_t share = (nbk + 7) / 8, sets = (share + 3) / 4;
    return ng <= 256 || share >= sets * 3;  // at most a quarter of the sets' slots empty
}

// Q8_0 product of more than 8 rows: whether the matrix kernel's 64 x 64 tiles (t64 of them,
// 512 threads each) take a product of nbk key blocks that 128 x 128 tiles would take with ks
// key splits; slots = resident workgroups. While they fit the slots they win everywhere
// measured (9 rows to 512 tiles; 592 weight rows x 498 blocks x 1625 rows 123 against 118 us
// is the one exception found). Past that, up to two and a half times over (us, 128 / 64):
//   64 key blocks: 1152 tiles 55 / 49, 1600 64 / 70; past 5 tiles per CU the times cross back
//     and forth (64-80 blocks: of the time, 1344-1536 tiles 0.88-0.97, 2016 0.91-0.94, 2432
//     1.08, 3344 0.93) and the 128 x 128 tiles stay
//   3 or 4 key splits stand against their second round: 640 tiles, 128 blocks 56 / 60
//   2 key splits: 0.85-0.95 of the time, at 800 tiles of 192 blocks or more 1.00-1.02 (304
//     blocks, 1217 rows 132 / 134; the 64 x 64 tiles all the same: they need no partials, and
//     the call without a workspace of its own takes sizes that partials would not leave room for)
//   short keys: the pipeline's start and the sum of the key groups weigh more the more tiles
//     a CU gets in turn: of the time, with 3 tiles per CU (768) 8 blocks 0.92, 6 1.0, 5 1.04,
//     1 1.11; with 4 (1024) 12 blocks 0.93, 10 1.0, 5 1.13; with 5 (1280) 16 blocks 0.97, 12 1.0,
//     5 1.22
inline bool mmq_small_tiles(uint64_t t64, uint64_t slots, uint64_t ks, uint32_t nbk) {
    if (t64 <= slots) {
        return true;
    }
    const uint64_t cu = (2 * t64 + slots - 1) / slots;  // tiles per CU
    return ks < 3 && cu <= 5 && nbk >= 4 * (cu - 1);
}

// APG: whether a workgroup takes a whole sample (its frames in rows of oc channels)
// instead of one or two channels of it (cg). The channel split fills the chip where
// there are few samples, but each of its workgroups takes a line request per frame for
// 16 bytes of it, so its time grows with n * oc; a workgroup per sample reads whole
// lines, and up to 256 samples take hardly longer than one. The line is where these
// two estimates cross (ns; 256 CUs, buffers of 500 MB in turn), us by sample / by channels:
//   64 channels:   1 x 6000 482 / 39, 8 x 750 59 / 11, 64 x 750 67 / 67, 128 x 750 77 / 131,
//                  256 x 1500 227 / 440, 16 x 100 8.2 / 8.1, 64 x 100 11.6 / 29.9, 1 x 12 3.3 / 4.2
//   1024 channels: 1 x 750 964 / 18, 16 x 750 1050 / 265, 8 x 12 12.8 / 50, 256 x 12 26 / 1553
inline bool apg_by_sample(uint32_t n, uint32_t t, uint32_t oc, uint32_t cg) {
    if (n > 65535) {
        return true;  // the channel split's grid has the samples in y
    }
    const uint32_t phases = 1024 / oc;  // frames that a sample's workgroup takes at a time
    const double   groups = (double) n * (oc / cg), rounds = (double) ((uint64_t) (groups + 255) / 256);
    const double   frames = (double) t / phases;  // of a thread
    const double   sample = 2000 + 30.0 * phases + (1100 + 6.0 * n) * frames;
    const double   over   = 0.03 * t * groups, chain = 4.5 * t;
    return sample < 1500 + 1400 * cg * rounds + (over > chain ? over : chain);
}

}  // namespace mi
