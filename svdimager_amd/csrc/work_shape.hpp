// Work shape of the MFMA window gridder: how a half window's records are cut into the pieces that workgroups
// contract.  The same source compiles for the device, the host and CPU probes.
#pragma once

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

}  // namespace svdi
