// Device-memory decisions of the schedule build (host only).
//
// Sizes in bytes; dn: cells x directions, dp: periodic cells x directions,
// rs: size of a stored rate.
#pragma once

#include <cstdint>

namespace ssw {

// What ssw_upload_state allocates: X, I and P, and per cell ten 8-byte arrays
// (state, source, timescales, rates, {source, attenuation} and the photon rate
// of a download) and the chemistry's queue.
inline int64_t state_bytes(int64_t cells, int64_t dn, int64_t dp, int64_t rs) {
    return (2 * dn + dp) * rs + cells * (10 * 8 + 2 * rs + 4);
}

// What the first rotation adds to the state: the rate offsets.
inline int64_t offset_bytes(int64_t dn, int64_t dp, int64_t rs) { return (dn + dp) * rs; }

// Whether the grouped replay's tiles are built: they and what the handle
// allocates after them have to fit into `free`, the memory that is free once
// all that was freed has come back. 1/16 and 1 MB for the rounding of the
// allocations; no part of it belongs to the device's size, since a small grid
// on a nearly full device has to be grouped as anywhere else.
inline bool cones_fit(int64_t tiles, int64_t later, int64_t free) {
    const int64_t need = tiles + later;
    return need + need / 16 + (1 << 20) <= free;
}

}  // namespace ssw
