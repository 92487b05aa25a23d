// Device-memory decisions of the schedule build (host only).
//
// Sizes in bytes; dn: cells x directions, dp: periodic cells x directions,
// rs: size of a stored rate.
#pragma once

#include <algorithm>
#include <cstdint>

namespace ssw {

// 16-byte planes of a tile of the compiled replays whose tasks have up to n
// upwind entries (two of them hold LDS words, the others the downwind area and
// the weights).
constexpr uint32_t tile_planes(bool fp32, uint32_t n) {
    if (fp32) return n <= 3 ? 2u : n <= 5 ? 3u : n <= 7 ? 4u : n <= 11 ? 5u : 6u;
    return n <= 1 ? 2u : n <= 3 ? 3u : n <= 5 ? 4u : n <= 7 ? 6u : n <= 9 ? 7u : n <= 11 ? 8u : 9u;
}

// Entries of the cone build's task list: a grid whose cones solve more is not grouped.
constexpr int64_t cone_list_cap(int64_t dn) { return dn + dn / 4 + (1 << 20); }

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
// all that was freed has come back. 1 MB and 1/16, at most 1 GB, for the
// rounding of the allocations and transient downloads; no part of it belongs to
// the device's size, since a small grid on a nearly full device has to be
// grouped as anywhere else.
inline bool cones_fit(int64_t tiles, int64_t later, int64_t free) {
    const int64_t need = tiles + later;
    return need + std::min<int64_t>(need / 16, 1 << 30) + (1 << 20) <= free;
}

// How a handle replays its sweeps: from the faces, from planes with one launch
// per level set, from tiles of cones, from tiles of directions.
enum class Replay { kGeometric, kPerLevel, kGrouped, kDirections };

struct Problem {
    int64_t cells, faces, periodic_cells, directions, levels;
    bool fp32;
};

// The most that a handle holds beside its grid arrays from the layering on:
// while the schedule is built, or with it, the active-set lists, the state and
// the photon rate of a download. Measured as a part of handle_bytes on jittered
// and clustered grids of 512 to 600000 cells, 1 to 84 directions, 1 and 4
// timestep levels, both precisions, from 100000 tasks on: 1.04 to 1.44 of a
// handle's peak from the faces (not every level's list was made), 1.03 to 1.17
// with planes, 1.08 to 1.44 with cones, 1.06 to 1.27 with directions' tiles; up
// to 2.5 for the tiles of cartesian grids, whose three upwind faces need fewer
// planes. Below that, minimum sizes count.
inline int64_t replay_bytes(const Problem& p, Replay r) {
    const int64_t n = p.cells, f = p.faces, d = p.directions, dn = d * n, more = p.levels - 1;
    const int64_t rs = p.fp32 ? 4 : 8, es = p.fp32 ? 8 : 16;
    const int64_t state = state_bytes(n, dn, p.periodic_cells * d, rs);
    int64_t root = 1;  // level sets: a third root of the cells times 28 to 43 on those grids
    while (root * root * root < n) root++;
    const int64_t kmax = std::min(n, 64 * root);
    // the widest tiles: half of the faces look upwind, some cells have more
    const int64_t planes = tile_planes(p.fp32, (uint32_t)std::min<int64_t>(13, (f + 2 * n - 1) / (2 * n) + 5));
    const int64_t layering = 18 * dn + 4 * n;  // counters, queues, depths; then the four sort arrays
    if (r == Replay::kGeometric) return std::max(std::max(layering, 20 * dn), 16 * dn + more * 4 * dn + state);
    if (r == Replay::kDirections) {
        const int64_t held = dn * (16 * planes + 4 + 8 + 2 * rs + (more ? 1 : 0));
        return std::max(layering, std::max(held + 6 * dn + 8 * d * kmax, held + state));
    }
    const int64_t compiled = dn * (16 + rs + 12 * es) + dn * es / 16;  // overflow entries: one for 16 tasks
    const int64_t level = std::max(layering, std::max(compiled + 12 * dn, compiled + 4 * dn + more * 4 * dn + state +
                                                                              40 * kmax));
    if (r == Replay::kPerLevel) return level;
    // cones: solved up to 1.57 times a task on those grids; indices, far and
    // extra entries of a task beside its planes; 16 wave slots of 16 bytes a cone
    const int64_t cap = cone_list_cap(dn), solved = std::min(cap, dn * 33 / 20), cones = dn / 64 + kmax;
    const int64_t tiles = solved * (16 * planes + 8 + 2 * f / n) + cones * 264;
    const int64_t build = std::max(23 * dn + 2 * f * d, tiles + 9 * dn + solved) + 4 * cap + 64 * cones;
    const int64_t run = tiles + 4 * dn + (more ? cones * (8 + 4 * more) : 0) + state;
    return std::max(level, std::max(build, run));  // `level` where they do not fit
}

// Device memory of a handle from the grid's upload through steps and
// downloads.
inline int64_t handle_bytes(const Problem& p, Replay r) {
    const int64_t n = p.cells, f = p.faces;
    const int64_t periodic = std::min(f, p.periodic_cells * ((f + n - 1) / n));  // faces
    const int64_t grid = (n + 1) * 4 + f * 36 + n * 29 + p.periodic_cells * 8 + periodic * 36;
    const int64_t upload = 37 * std::min(f, std::max<int64_t>(1 << 20, 16 * p.directions * n) / 37) + 20 * n;
    const int64_t b = grid + std::max(upload, replay_bytes(p, r));
    return b + b / 32 + (1 << 20);
}

}  // namespace ssw
