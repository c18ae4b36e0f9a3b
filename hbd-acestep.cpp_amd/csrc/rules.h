// rules.h -- dispatch rules as plain host functions of sizes, so that they can be
// checked without a GPU. Each says what was measured on both sides of its line.
#pragma once

#include <cstdint>

namespace mi {

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
