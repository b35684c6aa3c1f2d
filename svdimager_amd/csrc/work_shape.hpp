// Work shape of the MFMA window gridder: above how many records (coop_min) a half window is dense, and into pieces
// of how many (coop_cap) a dense half is cut.  The same source compiles for the device, the host and CPU probes.
#pragma once

#include <algorithm>
#include <cstddef>
#include <cstdint>

#include "svdi_math.hpp"

namespace svdi {

// A dense half's pieces: equal runs of `per` records (a multiple of 32), the last one shorter, as few as hold at most
// `cap` records each (rounded up to that multiple).  No records are no pieces: the callers ask for halves that are not dense too.
struct Pieces {
    uint32_t count, per;
};
SVDI_HD Pieces dense_pieces(uint32_t records, uint32_t cap) {
    if (records == 0) return {0u, 0u};
    const uint32_t n = (records - 1) / cap + 1;
    const uint32_t per = ((records - 1) / n + 32u) & ~31u;
    return {(records - 1) / per + 1, per};
}

constexpr uint32_t kCoopMinLeast = 256, kCoopMinMost = 1024;
constexpr uint32_t kCoopCapLeast = 2048, kCoopCapMost = 16384;

// The shape that a call asks for: the caller's numbers (0: none), else by the number of samples.  Fewer samples
// take smaller pieces, so that they still spread over the chip (a workgroup contracts a piece of
// 16384 records in about 100 us), and a lower threshold, so that no wavefront's item is a long
// chain.  Measured per call (coop_min / coop_cap): 8.4 M samples at 1024^2 869 us with
// 1024 / 16384, 882 with 1024 / 8192, 986 with 512 / 4096; 5.2 M at 512^2 700 with 1024 / 8192,
// 745 with 512 / 4096; 2.1 M at 1024^2 642 with 512 / 4096, 677 with 1024 / 8192; 1.4 M at 1000^2 635 with
// 512 / 4096, 661 with 256 / 2048, 672 with 1024 / 8192; 32 k at 128^2 210 with 256 / 2048, 232 with
// 1024 / 8192.
struct WorkShape {
    uint32_t coop_min, coop_cap;
};
inline WorkShape work_shape(size_t samples, uint32_t coop_min, uint32_t coop_cap) {
    auto clamped = [](size_t v, size_t lo, size_t hi) { return static_cast<uint32_t>(std::min(std::max(v, lo), hi)); };
    return {coop_min != 0 ? coop_min : clamped(samples / 4096, kCoopMinLeast, kCoopMinMost),
            coop_cap != 0 ? coop_cap : clamped(samples / 512, kCoopCapLeast, kCoopCapMost)};
}

// The most pieces that `records` records in `halves` halves can make: one for each half with more than coop_min,
// and one more for every coop_cap records.
inline size_t most_pieces(const WorkShape& s, size_t records, size_t halves) {
    return records / s.coop_cap + std::min(halves, records / (static_cast<size_t>(s.coop_min) + 1));
}

// Slots that snapshots of the usual arrays do with, from few samples on large grids to many on small ones: they make 1.4
// records a sample, and dense halves of several times coop_min on average (pieces made, and this: 29 and 46 for 32 k samples
// at 128^2, 951 and 1,536 for 1.4 M at 1000^2, 1,492 and 2,301 for 8.4 M at 1024^2, 915 and 1,056 for 2.1 M at 128^2, which with
// 518 slots took 388 us, so 353).
inline size_t usual_pieces(const WorkShape& s, size_t samples, size_t halves) {
    return samples * 3 / 2 / s.coop_cap + std::min(halves, samples * 3 / 16 / s.coop_min);
}

// Every piece takes a partial slot.  Where the slots are fewer than most_pieces (the worst case is several times what
// any snapshot makes: 17,361 for the SKA-Low one, which makes 1,492), the dense halves are counted by size first, and
// if their pieces do not fit, the shape is made coarser on the device: the pieces longer, until all dense records' take what the
// halves leave, at least half the slots, then the threshold higher by quarters of an octave, so that the smallest halves
// are left to wavefront items.
// words: [0] dense halves, [1] their records, [2 + 2 b], [3 + 2 b] those of size bucket b, which holds the halves of
// more than shape_threshold(coop_min, b) and at most shape_threshold(coop_min, b + 1) records.
constexpr int kShapeBuckets = 112;                 // 28 octaves: 32 records to 2^31
constexpr int kShapeWords = 2 + 2 * kShapeBuckets;
constexpr uint32_t kAllSlotsFit = 0xffffffffu;

SVDI_HD uint32_t shape_threshold(uint32_t coop_min, int b) {
    const uint64_t t = ((static_cast<uint64_t>(coop_min) * (4u + (b & 3))) << (b >> 2)) >> 2;
    return t < 0xffffffffu ? static_cast<uint32_t>(t) : 0xffffffffu;
}
SVDI_HD int shape_bucket(uint32_t coop_min, uint32_t records) {     // records > coop_min
    int b = 0;
    while (b + 4 < kShapeBuckets && shape_threshold(coop_min, b + 4) < records) b += 4;
    while (b + 1 < kShapeBuckets && shape_threshold(coop_min, b + 1) < records) ++b;
    return b;
}
SVDI_HD void fit_shape(const uint32_t* words, uint32_t slots, WorkShape& s) {
    if (slots == kAllSlotsFit || words[0] + words[1] / s.coop_cap <= slots) return;
    const uint32_t cuts = words[0] < slots / 2 ? slots - words[0] : slots / 2;
    const uint32_t cap = cuts != 0 ? words[1] / cuts + 1 : 0xffffffffu;
    if (cap > s.coop_cap) s.coop_cap = cap;
    uint32_t halves = 0, records = 0;
    int b = kShapeBuckets;
    for (; b > 0; --b) {
        halves += words[2 * b];
        records += words[2 * b + 1];
        if (halves + records / s.coop_cap > slots) break;
    }
    s.coop_min = b == kShapeBuckets ? 0xffffffffu : shape_threshold(s.coop_min, b);
}

}  // namespace svdi
