// libsubsweep_amd: MI355X (gfx950) sweep radiative transfer + hydrogen chemistry.
//
// Device layout (one handle = one resident problem):
//   faces      CSR over cells: off[N+1] (u32), geo[F] = {nx, ny, nz, area} (f64x4),
//              nk[F] = neighbour | kind << 30 (u32); for the Nper cells with a
//              periodic face also a compact list of those faces
//   cell state rho, x, T, source/D, attenuation, timestep, previous rate,
//              change timescale (f64[N]); timestep level (u8[N])
//   fluxes     X = outgoing rate / downwind effective area (FP64 or scaled FP32)
//              I = incoming rate at solve time (FP64 or scaled FP32)
//              direction-major [d * N + c]; in the compiled replays X in schedule
//              order (xpos), with direction sweeps I too
//              P[d * Nper + slot] periodic-source snapshot of the periodic cells
//   schedule   the (cell, direction) tasks of the full dependency graph in Kahn
//              order, level-major, within a level sorted by (direction, cell);
//              full_start[k] is where level set k begins. Four replay forms:
//              geometric  task records {cell | face_count << 25, first_face,
//                         direction, periodic slot} (16 B per task)
//              cones      the default: groups of level sets cut into cones,
//                         compiled into tiles whose entries name LDS words
//                         (k_sweep_cone)
//              directions one workgroup per direction, its tasks in tiles
//                         (k_sweep_dir)
//              per level  group levels 1, or where cones do not fit:
//                         per task a header {cell | direction << 25, periodic
//                         slot, overflow start, upwind count}, the effective area
//                         A, and its upwind local faces as (neighbour, weight)
//                         pairs in kPlanes planes: entry q of the task at
//                         position p of a level set starting at b with width W
//                         is planes[kPlanes * b + q * W + (p - b)] in FP64 and
//                         planes[kPlanes * b + ((q / 2) * W + (p - b)) * 2 + q % 2]
//                         in FP32, plane pairs of 16 bytes (coalesced across
//                         tasks, addressable without reading the header);
//                         entries q >= kPlanes (rare) sit in an overflow list,
//                         indexed per (direction, cell).
//              A sweep at timestep level l solves the cells with level >= l.
//              Restricted to those cells, the full graph's level sets are still
//              a valid order (an active task's active upwind neighbours are in
//              earlier level sets), so such a sweep replays the full schedule:
//              through a per-level list of the active positions (idx[l]),
//              made by a stream compaction when the active set changes, or the
//              cones that hold active tasks, or all tiles of the directions.
//
// The transport is the reference's upwind sweep (src/sweep/mod.rs:412-513)
// restated in pull form. A cell that is solved distributes the change of its
// outgoing rate over its downwind faces in proportion to area * (n . d)
// (:453-461), so the incoming rate of a cell equals, up to rounding,
//   I[c,d] = sum_{upwind local faces f} area_f (-n_f . d) * O[nb,d] / A[nb,d]
// with A[nb,d] = sum of area (n . d) over nb's downwind faces. Storing
// X = O / A lets every task gather its upwind neighbours' X instead of
// scattering with atomics. The upwind sum is evaluated in face order, one term
// after the other, and A by a fixed 16-way tree, in every kernel, so the
// geometric and the compiled replay give bitwise the same result, whatever
// order tasks run in. The level sets (Kahn layering of init_counts' counts,
// src/sweep/mod.rs:346-386) are built on the device once per grid, one workgroup
// per direction (k_layers); the level-set parity hook builds the layering of a
// restricted active set the same way.

#include <hip/hip_runtime.h>
#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <array>
#include <atomic>
#include <chrono>
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <exception>
#include <functional>
#include <limits>
#include <mutex>
#include <shared_mutex>
#include <thread>
#include <string>
#include <unordered_map>
#include <vector>

#include "../../include/subsweep_amd.h"
#include "chemistry.h"
#include "direction_bins.h"
#include "level_math.h"
#include "memory_plan.h"

namespace {

constexpr int kBlock = 256;
constexpr uint32_t kKindLocal = 0;
constexpr uint32_t kKindPeriodic = 1;
constexpr uint32_t kKindBoundary = 2;
constexpr uint32_t kNbrMask = 0x3FFFFFFFu;
constexpr uint32_t kNone = 0xFFFFFFFFu;
constexpr int kLanes = 16;                 // lanes per task in the geometric kernels
constexpr int kTasksPerBlock = kBlock / kLanes;
constexpr uint32_t kCellBits = 25;         // task record: cell index bits
constexpr uint32_t kCellMask = (1u << kCellBits) - 1u;
constexpr int kMaxFaces = 127;             // faces per cell
constexpr int kPlanes = 12;                // upwind entries per task held in planes
static_assert(kPlanes % 2 == 0, "FP32 plane entries are stored in pairs");
constexpr int kChunk = 4096;               // compaction chunk (tasks, within one level set)
constexpr int kRunBlock = 1024;            // workgroup of a run of narrow level sets (tasks per level set)
constexpr int kGroupT = 64;                // grouped replay: root tasks per workgroup (default; 32, 64 or 128)
constexpr int kGroupLevels = 4;            // grouped replay: level sets per group (default)
constexpr int kConeCap = 3072;             // grouped replay build: cone members / pending entries per workgroup
constexpr int kConeThreads = 256;
constexpr int kSortCap = 4096;             // grouped replay build: entries of one level set sorted in LDS
constexpr int kMaxGroup = 8;               // grouped replay: level sets per group
// grouped replay: level sets this narrow go kMaxGroup to a group. Their cones
// overlap more (1.18 -> 1.41 tasks solved per task on 20000 cells x 84
// directions), but a launch's first loads are paid half as often: that sweep
// 1.61 ms with 2048, 1.55 with 4096, 1.56 with 8192; on 117649 x 64 FP32 1.48,
// 1.47, 1.45; beyond, cones of wide level sets no longer fit.
constexpr uint32_t kNarrowGroup = 8192;
constexpr uint32_t kCus = 256;             // MI355X: compute units
constexpr uint32_t kXcds = 8;              // MI355X: accelerator dies, each with its own L2

// Staging of ssw_download_noalloc, which allocates nothing: a file-scope
// device array that every device the library runs on holds until the process
// ends. One output array of at most kNoAllocBytes / 8 cells passes through it
// at a time. Host code never uses the name `scratch` as an address (in host
// code it is a stand-in, not the device array): it uses the per-device address
// from hipGetSymbolAddress (noalloc_scratch below).
constexpr size_t kNoAllocBytes = size_t(64) << 20;
constexpr int kMaxDevices = 64;
static __device__ __align__(256) uint8_t scratch[kNoAllocBytes];

thread_local std::string g_err;
// Handles alive in the process.
std::atomic<int> g_live_handles{0};
// A stream capture is invalidated by the device-synchronising calls
// (allocation, free, blocking copies, stream creation and destruction) that
// other threads make while it runs. Those calls hold this lock shared; a
// capture holds it exclusively, so that handles driven from several threads
// (the request loop) capture their replays too.
std::shared_mutex g_capture_mu;
std::atomic<uint64_t> g_next_uid{0};

int fail(int code, const std::string& msg) {
    g_err = msg;
    return code;
}

#define HIP_TRY(expr)                                                                           \
    do {                                                                                        \
        hipError_t _e = (expr);                                                                 \
        if (_e != hipSuccess)                                                                   \
            return fail(_e == hipErrorOutOfMemory ? SSW_ERR_OOM : SSW_ERR_HIP,                  \
                        std::string(#expr) + ": " + hipGetErrorString(_e));                     \
    } while (0)

#define TRY(expr)                    \
    do {                             \
        int _r = (expr);             \
        if (_r != SSW_OK) return _r; \
    } while (0)

// ---------------------------------------------------------------------------
// device helpers

__device__ __forceinline__ double fdot(const double4& g, double dx, double dy, double dz) {
    // glam DVec3::dot: (x*x') + (y*y') + (z*z'), no contraction
    return (g.x * dx + g.y * dy) + g.z * dz;
}

// Upwind entry of the compiled schedule.
template <typename R>
struct Entry;
template <>
struct __align__(8) Entry<float> {
    uint32_t nb;
    float w;
};
template <>
struct __align__(16) Entry<double> {
    uint32_t nb;
    uint32_t pad;
    double w;
};

// The plane entries of a level set of width W, from the level set's first
// entry (kPlanes * W entries of storage; p is a task's offset in the level
// set). FP32 entries (8 bytes) are stored in plane pairs, entries 2h and
// 2h+1 of a task side by side, so that a task reads its kPlanes entries with
// kPlanes / 2 loads of 16 bytes (half the load instructions, and half the
// cache-line lookups where a workgroup's tasks sit at scattered positions).
// FP64 entries are split: the upwind positions four to 16 bytes (entry q of
// task p at uint32 index ((q / 4) * W + p) * 4 + q % 4), then the weights two
// to 16 bytes (at double index 6 * W + ((q / 2) * W + p) * 2 + q % 2), so that
// a task reads them with kPlanes / 4 + kPlanes / 2 loads of 16 bytes and no
// padding; the last quarter of the level set's storage is unused.
template <typename R>
__host__ __device__ __forceinline__ size_t plane_off(uint32_t q, uint32_t W, uint32_t p) {
    return ((size_t)(q >> 1) * W + p) * 2 + (q & 1u);  // FP32
}
__host__ __device__ __forceinline__ size_t plane_nb_off(uint32_t q, uint32_t W, uint32_t p) {
    return ((size_t)(q >> 2) * W + p) * 4 + (q & 3u);  // FP64 positions, uint32 index
}
__host__ __device__ __forceinline__ size_t plane_w_off(uint32_t q, uint32_t W, uint32_t p) {
    return (size_t)6 * W + ((size_t)(q >> 1) * W + p) * 2 + (q & 1u);  // FP64 weights, double index
}
static_assert(kPlanes % 4 == 0, "FP64 upwind positions are stored four to 16 bytes");

struct Geo {
    int64_t N;
    int D;
    int L;
    const uint32_t* off;
    const double4* geo;
    const uint32_t* nk;
    const double* dirs;      // D x 3
    const uint8_t* level;
    const uint32_t* pslot;   // N: periodic slot or kNone
    const uint32_t* pcells;  // Nper
    const uint32_t* pfoff;   // Nper + 1: periodic faces of each periodic cell
    const double4* pgeo;     // {normal, area} of each of them
    const uint32_t* pnb;     // and its neighbour
    int64_t Nper;
    uint32_t* cnt;           // D x N missing-upwind counters
    uint32_t* need;          // L: the active set of a sweep level changed
};

// Per-cell {transport source / D in the storage scale, attenuation} as the
// transport reads them: in its storage precision (the FP32 transport rounds
// both to float before use, so storing them rounded changes no result).
template <typename R>
struct SAOf {
    using T = double2;
};
template <>
struct SAOf<float> {
    using T = float2;
};
template <typename R>
using SA = typename SAOf<R>::T;

template <typename R>
struct Flux {
    R* X;                    // D x N, at xidx(d, c)
    const uint32_t* xpos;    // compiled replay: X of (c, d) at the task's schedule position xpos[d*N + c]
    R* I;                    // D x N, at iidx(d, c)
    const uint32_t* ipos;    // direction sweeps: I in X's order (= xpos); else NULL: d*N + c
    R* P;                    // D x Nper
    // After a rotation of the directions (ssw_rotate_directions), the rates
    // that the remap of the state left in place, as offsets to the pull sums:
    // the incoming rate of (c, d) is offI[d*N + c] + sum of the upwind X, the
    // periodic source offP[d*Nper + slot] + its periodic sum. NULL before any
    // rotation (offsets 0).
    R* offI;                 // D x N
    R* offP;                 // D x Nper
    const SA<R>* sa;         // N: {source / D in the storage scale, attenuation} (one load per task)
    R thr;                   // smallest R not below the threshold in the storage scale
    double inv_lref;         // storage scale of rates
    double inv_aref;         // storage scale of areas
};

// Where X of (cell c, direction d) is stored: direction-major d*N + c, or in
// the compiled replay the task's position in the schedule (level-major), so
// that a level set's gathers read what the previous level sets wrote densely.
template <typename R>
__device__ __forceinline__ size_t xidx(const Flux<R>& fl, int64_t N, uint32_t d, uint32_t c) {
    const size_t o = (size_t)d * N + c;
    return fl.xpos ? (size_t)fl.xpos[o] : o;
}

// Where I of (cell c, direction d) is stored.
template <typename R>
__device__ __forceinline__ size_t iidx(const Flux<R>& fl, int64_t N, uint32_t d, uint32_t c) {
    const size_t o = (size_t)d * N + c;
    return fl.ipos ? (size_t)fl.ipos[o] : o;
}

// Descriptor ranges of a grouped launch, one per build pass (the group's
// last level set's roots first): workgroups [off[r], off[r+1]) solve pass r's
// descriptors. n = 0: no ranges (the workgroup order is the descriptor order).
struct PassTab {
    uint32_t off[kMaxGroup + 1];
    int n;
};

// The descriptor of workgroup b: the hardware deals workgroups to the dies
// round-robin (b mod kXcds). Inside the pass range [o, o + c) that holds b,
// the workgroups of one die are those with the same x = (b - o) mod kXcds;
// they are given the contiguous run of the range's descriptors that starts
// at o + x*(c / kXcds) + min(x, c mod kXcds), in order. Neighbouring cones,
// which read the same schedule and X lines, then share one die's L2, and
// every die still gets an eighth of every pass.
__device__ __forceinline__ uint32_t pass_item(const PassTab& pt, uint32_t b) {
    if (pt.n == 0) return b;
    int r = 0;
    while (r + 1 < pt.n && b >= pt.off[r + 1]) r++;
    const uint32_t o = pt.off[r], c = pt.off[r + 1] - o, i = b - o;
    const uint32_t x = i % kXcds, q = c / kXcds, rem = c % kXcds;
    return o + x * q + min(x, rem) + i / kXcds;
}

// Block b of nb equal blocks in die order: the hardware deals workgroups to
// the dies round-robin (b mod kXcds); die x takes the contiguous run of
// blocks [x*q + min(x, r), ...) (q = nb / kXcds, r = nb mod kXcds), so that
// neighbouring blocks, whose gathers share cache lines, share its L2.
__device__ __forceinline__ uint32_t xcd_block(uint32_t b, uint32_t nb) {
    const uint32_t x = b % kXcds, q = nb / kXcds, r = nb % kXcds;
    return x * q + min(x, r) + b / kXcds;
}

__device__ __forceinline__ uint4 task_record(uint32_t c, uint32_t f0, uint32_t f1, uint32_t d, uint32_t ps) {
    return make_uint4(c | ((f1 - f0) << kCellBits), f0, d, ps);
}

__device__ __forceinline__ uint32_t wave_max(uint32_t v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = max(v, (uint32_t)__shfl_xor((int)v, o));
    return v;
}

// Per-cell inputs of a task's outgoing rate, loaded as soon as the task's cell
// is known so that they arrive with the upwind gathers.
template <typename R>
struct CellIn {
    double src;
    double att;
    R per;
    R off;  // incoming-rate offset after a rotation (0 before)
};

template <typename R>
__device__ __forceinline__ CellIn<R> cell_inputs(const Geo& g, const Flux<R>& fl, uint32_t c, uint32_t d,
                                                 uint32_t ps) {
    CellIn<R> ci;
    const SA<R> sa = fl.sa[c];
    ci.src = sa.x;
    ci.att = sa.y;
    // the periodic load uses slot 0 for cells without one (always a valid index)
    const R p = fl.P ? fl.P[(size_t)d * g.Nper + (ps != kNone ? ps : 0u)] : (R)0;
    ci.per = (ps != kNone) ? p : (R)0;
    ci.off = fl.offI ? fl.offI[(size_t)d * g.N + c] : (R)0;
    return ci;
}

// Outgoing rate of a solved task (Site::get_rate + HydrogenOnly::get_outgoing_rate,
// src/sweep/site.rs:49-56, src/chemistry/hydrogen_only/mod.rs:72-88) from its
// upwind sum `inc`, which is clamped on the way; oi: its place in I. Stored as
// X = O / A at ox, I at oi.
template <typename R, bool kOffsets>
__device__ __forceinline__ R outgoing_rate(const Flux<R>& fl, size_t oi, R& inc, const CellIn<R>& ci) {
    if (kOffsets && fl.offI) {
        // after a rotation the incoming rate is the remapped rate plus the
        // corrections since, offset + upwind sum; its persistent clamp
        // (Photons::make_positive) sets the offset to -sum, so that the rate
        // is 0 now and grows by the later corrections only
        R t = ci.off + inc;
        if (t < (R)0) {
            fl.offI[oi] = -inc;
            t = 0;
        }
        inc = t;
    } else if (inc < (R)0) {
        inc = 0;  // Photons::make_positive
    }
    R in = (inc + (R)ci.src) + ci.per;
    // a rate below the threshold; in FP32 the threshold is threshold / lref
    // (e.g. 1e-5 / 2^160), far below the float range: thr is rounded up, which
    // leaves the comparison with every float as it is
    return (in < fl.thr) ? (R)0 : in * (R)ci.att;
}

template <typename R>
__device__ __forceinline__ void finish_task(const Flux<R>& fl, size_t ox, size_t oi, R inc, const CellIn<R>& ci,
                                            R A) {
    const R out = outgoing_rate<R, true>(fl, oi, inc, ci);
    fl.X[ox] = (A > (R)0) ? out / A : (R)0;
    fl.I[oi] = inc;
}

// The face loop of one task of the geometric replay, kLanes lanes per task
// (one face each). Lane `sub` handles faces sub, sub + kLanes, ...; the loop
// runs to the longest face list of the wave so that every lane takes part in
// the shuffles. The upwind sum is accumulated in face order on every lane of
// the group; A is the xor-butterfly over the lanes' partial sums.
template <typename R>
__device__ __forceinline__ void task_faces(const Geo& g, const Flux<R>& fl, bool valid, uint4 r, uint32_t sub,
                                           uint32_t nfmax, double& A_out, R& inc_out) {
    const uint32_t nf = valid ? (r.x >> kCellBits) : 0u;
    const uint32_t d = r.z;
    const double dx = g.dirs[3 * d], dy = g.dirs[3 * d + 1], dz = g.dirs[3 * d + 2];
    const size_t dN = (size_t)d * g.N;
    const int lane = __lane_id();
    const int gbase = lane & ~(kLanes - 1);
    double A = 0.0;
    R inc = 0;
    for (uint32_t base = 0; base < nfmax; base += kLanes) {
        const uint32_t j = base + sub;
        const bool fa = j < nf;
        const uint32_t f = r.y + j;
        const double4 a = fa ? g.geo[f] : make_double4(0.0, 0.0, 0.0, 0.0);
        const uint32_t nk = fa ? g.nk[f] : (kKindBoundary << 30);
        const uint32_t nb = nk & kNbrMask;
        const bool local = (nk >> 30) == kKindLocal;
        const double dd = fdot(a, dx, dy, dz);
        const bool up = fa && local && dd < 0.0;
        const bool down = fa && dd > 0.0;
        // nb is a valid cell index on every lane (0 for lanes without a face
        // and for boundary faces), so the gathers and the neighbour loads are
        // unconditional and issue together; the products are selected after.
        const R w = up ? (R)(a.w * fl.inv_aref * -dd) : (R)0;
        const R xv = fl.X[dN + nb];
        const R v = up ? w * xv : (R)0;
        if (down) A += a.w * fl.inv_aref * dd;
#pragma unroll
        for (int l = 0; l < kLanes; l++) inc += __shfl(v, gbase + l);
    }
#pragma unroll
    for (int m = kLanes / 2; m > 0; m >>= 1) A += __shfl_xor(A, m, kLanes);
    A_out = A;
    inc_out = inc;
}

// ---------------------------------------------------------------------------
// grid checks and statistics (once per grid)

// Every local face c->nb needs a mirror face nb->c with exactly the negated
// normal, which makes the upwind/downwind classification of the pair agree.
// uneven: faces that one side repeats more often than the other. nb's upwind
// counter is then decremented more often than it counts: it may become ready
// before another of its upwind neighbours, so that only the replays that read
// upwind values from memory, one level set at a time, run on such grids.
__global__ void k_check_mirror(Geo g, unsigned long long* bad, unsigned long long* uneven) {
    int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= g.N) return;
    for (uint32_t f = g.off[c]; f < g.off[c + 1]; f++) {
        uint32_t nk = g.nk[f];
        if ((nk >> 30) != kKindLocal) continue;
        uint32_t nb = nk & kNbrMask;
        if ((int64_t)nb >= g.N || (int64_t)nb == c) {
            atomicAdd(bad, 1ull);
            continue;
        }
        double4 a = g.geo[f];
        uint32_t mirrors = 0, same = 0;
        for (uint32_t h = g.off[nb]; h < g.off[nb + 1]; h++) {
            uint32_t hk = g.nk[h];
            if ((hk >> 30) != kKindLocal || (int64_t)(hk & kNbrMask) != c) continue;
            double4 b = g.geo[h];
            if (b.x == -a.x && b.y == -a.y && b.z == -a.z) mirrors++;
        }
        if (mirrors == 0) atomicAdd(bad, 1ull);
        for (uint32_t h = g.off[c]; h < g.off[c + 1]; h++) {
            if (g.nk[h] != nk) continue;
            double4 b = g.geo[h];
            if (b.x == a.x && b.y == a.y && b.z == a.z) same++;
        }
        if (mirrors != same) atomicAdd(uneven, 1ull);
    }
}

// Thread t handles (cell t / D, direction t % D): the lanes of a wave share one
// or two cells, so the face loads are broadcasts.
__device__ __forceinline__ bool cell_dir(const Geo& g, uint32_t t, uint32_t& c, uint32_t& d) {
    c = t / (uint32_t)g.D;
    d = t - c * (uint32_t)g.D;
    return (int64_t)c < g.N;
}

constexpr int kFluxDirs = 8;    // directions per wave of the kernels that walk the faces of 64 cells
constexpr int kFluxCells = 64;

// Per (cell, direction): downwind faces by kind (the byte model), the number
// of upwind local faces beyond kPlanes (overflow entries) and, with `nups`,
// their number. A wave takes 64 cells and kFluxDirs directions; the counts
// leave a workgroup with one atomic each (one per wave made the four counters
// the bound: 4.9 ms on 262144 cells x 84 directions, 0.28 ms like this).
__global__ void __launch_bounds__(1024) k_face_stats(Geo g, unsigned long long* out4, uint32_t* ovf_count,
                                                     uint8_t* nups) {
    __shared__ unsigned long long sum[4];
    if (threadIdx.x < 4) sum[threadIdx.x] = 0;
    __syncthreads();
    const uint32_t lane = threadIdx.x % kFluxCells;
    const uint32_t w = __builtin_amdgcn_readfirstlane(threadIdx.x / kFluxCells);
    const int64_t c = (int64_t)blockIdx.x * kFluxCells + lane;
    uint32_t n[4] = {0, 0, 0, 0}, nup[kFluxDirs];
#pragma unroll
    for (int j = 0; j < kFluxDirs; j++) nup[j] = 0;
    const uint32_t f1 = c < g.N ? g.off[c + 1] : 0u;
    for (uint32_t f = c < g.N ? g.off[c] : 0u; f < f1; f++) {
        const uint32_t kind = g.nk[f] >> 30;
        const double4 a = g.geo[f];
#pragma unroll
        for (int j = 0; j < kFluxDirs; j++) {
            const int d = (int)w * kFluxDirs + j;
            if (d >= g.D) break;
            const double dd = fdot(a, g.dirs[3 * d], g.dirs[3 * d + 1], g.dirs[3 * d + 2]);
            n[0] += dd > 0.0 && kind == kKindLocal;
            n[1] += dd > 0.0 && kind == kKindPeriodic;
            n[2] += dd > 0.0 && kind == kKindBoundary;
            nup[j] += dd < 0.0 && kind == kKindLocal;
        }
    }
#pragma unroll
    for (int j = 0; j < kFluxDirs; j++) {
        const int d = (int)w * kFluxDirs + j;
        if (c >= g.N || d >= g.D) break;
        const uint32_t extra = nup[j] > (uint32_t)kPlanes ? nup[j] - kPlanes : 0u;
        n[3] += extra;
        if (ovf_count) ovf_count[(size_t)d * g.N + c] = extra;
        if (nups) nups[(size_t)d * g.N + c] = (uint8_t)nup[j];
    }
    for (int k = 0; k < 4; k++) {
        uint32_t v = n[k];
        for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o);
        if (lane == 0 && v) atomicAdd(&sum[k], (unsigned long long)v);
    }
    __syncthreads();
    if (threadIdx.x < 4 && sum[threadIdx.x]) atomicAdd(&out4[threadIdx.x], sum[threadIdx.x]);
}

// Start of the overflow entries (upwind entries q >= kPlanes, in face order)
// of every (cell, direction) in the overflow list, ovf_start[d*N + c]
// (assigned by an atomic cursor); the schedule writes the entries.
__global__ void k_overflow(Geo g, const uint32_t* ovf_count, uint32_t* ovf_start, uint32_t* cursor) {
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    uint32_t c, d;
    if (!cell_dir(g, t, c, d)) return;
    const size_t o = (size_t)d * g.N + c;
    const uint32_t extra = ovf_count[o];
    ovf_start[o] = extra ? atomicAdd(cursor, extra) : 0u;
}

// ---------------------------------------------------------------------------
// Kahn layering (once per grid for the full graph; on demand for a restricted
// active set, for the parity hook)

// init_counts (src/sweep/mod.rs:346-386) for the active set {level >= lvl}:
// the active local upwind neighbours of every active (cell, direction), kNone
// for inactive cells. Thread t handles (cell t / D, direction t % D).
__global__ void k_count(Geo g, int lvl) {
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    uint32_t c, d;
    if (!cell_dir(g, t, c, d)) return;
    uint32_t n = 0;
    const bool active = g.level[c] >= lvl;
    if (active) {
        const double dx = g.dirs[3 * d], dy = g.dirs[3 * d + 1], dz = g.dirs[3 * d + 2];
        for (uint32_t f = g.off[c]; f < g.off[c + 1]; f++) {
            const uint32_t nk = g.nk[f];
            if ((nk >> 30) != kKindLocal) continue;
            if (!(fdot(g.geo[f], dx, dy, dz) < 0.0)) continue;
            if (g.level[nk & kNbrMask] >= lvl) n++;
        }
    }
    g.cnt[(size_t)d * g.N + c] = active ? n : kNone;
}

// The level sets of every direction from its counters (handle_local_neighbour,
// src/sweep/mod.rs:487-503): one workgroup per direction, since no dependency
// crosses directions. The tasks of a level set decrement their local downwind
// neighbours' counters, 8 lanes a task, two faces each; a counter that reaches
// 0 queues its task for the next level set. Writes depth[d*N + c] of active
// tasks, adds each level set's tasks to hist[k], and their number and the
// direction's level sets to totals = {tasks, most level sets}.
// Bound: the chain of a level set (queue, face range, faces, counters, one
// barrier). With kLds the counters lie in LDS as bytes (at most 127 upwind
// faces; an inactive cell's byte starts at 255 and never reaches 0), up to
// kLayerCells cells; else they are decremented in memory, as on grids whose
// faces repeat unevenly: a byte decremented below 0 would borrow from the next
// cell's, a counter in memory only never becomes ready again. The queues are in
// LDS, longer ones go on in `spill` (2 N entries a direction). A launch for
// every level set of all directions took 5 to 30 us a level set: 32768 cells x
// 84 directions 4.5 -> 1.3 ms, 262144 cells 23 -> 9.8 ms, 2 M clustered 184 ->
// 113 ms, 12167 cells x 32 1.9 -> 0.73 ms.
constexpr uint32_t kLayerQueue = 2048;
constexpr uint32_t kLayerCells = 139264;  // 136 KiB of LDS beside the queues
template <bool kLds>
__global__ void __launch_bounds__(1024) k_layers(Geo g, uint32_t kcap, uint32_t* __restrict__ depth, uint32_t* spill,
                                                 uint32_t* hist, uint32_t* totals) {
    __shared__ uint32_t queue[2][kLayerQueue];
    __shared__ uint32_t len[2];
    __shared__ uint32_t bytes[kLds ? kLayerCells / 4 : 1];
    const uint32_t d = blockIdx.x, N = (uint32_t)g.N, tid = threadIdx.x;
    const size_t dN = (size_t)d * N;
    const double dx = g.dirs[3 * d], dy = g.dirs[3 * d + 1], dz = g.dirs[3 * d + 2];
    uint32_t* const cnt = g.cnt + dN;
    auto push = [&](uint32_t which, uint32_t c) {
        const uint32_t i = atomicAdd(&len[which], 1u);
        if (i < kLayerQueue) queue[which][i] = c;
        else spill[2 * dN + (size_t)which * N + i] = c;
    };
    if (tid < 2) len[tid] = 0;
    __syncthreads();
    for (uint32_t c0 = 4 * tid; c0 < N; c0 += 4096) {  // level set 0
        uint32_t word = 0;
        for (uint32_t u = 0; u < 4 && c0 + u < N; u++) {
            const uint32_t n = cnt[c0 + u];
            word |= min(n, 255u) << (8 * u);
            if (n == 0) push(0, c0 + u);
        }
        if (kLds) bytes[c0 / 4] = word;
    }
    __syncthreads();
    uint32_t total = 0, k = 0;
    for (;; k++) {
        const uint32_t cur = k & 1u, n = len[cur];
        if (n == 0 || k >= kcap) break;
        if (tid == 0) atomicAdd(&hist[k], n);
        total += n;
        for (uint32_t i = tid / 8; i < n; i += 128) {
            const uint32_t c = i < kLayerQueue ? queue[cur][i] : spill[2 * dN + (size_t)cur * N + i];
            const uint32_t sub = tid % 8, f1 = g.off[c + 1];
            if (sub == 0) depth[dN + c] = k;
            for (uint32_t f = g.off[c] + sub; f < f1; f += 16) {
                const uint32_t h = f + 8 < f1 ? f + 8 : f;
                const double4 a[2] = {g.geo[f], g.geo[h]};
                const uint32_t nk[2] = {g.nk[f], g.nk[h]};
#pragma unroll
                for (int u = 0; u < 2; u++) {
                    if ((u && h == f) || (nk[u] >> 30) != kKindLocal || !(fdot(a[u], dx, dy, dz) > 0.0)) continue;
                    const uint32_t nb = nk[u] & kNbrMask;
                    bool ready;
                    if (kLds) {
                        const uint32_t sh = 8 * (nb & 3u);
                        ready = ((atomicSub(&bytes[nb / 4], 1u << sh) >> sh) & 255u) == 1u;
                    } else {
                        ready = __hip_atomic_fetch_sub(&cnt[nb], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) ==
                                1u;
                    }
                    if (ready) push(cur ^ 1u, nb);
                }
            }
        }
        __syncthreads();
        if (tid == 0) len[cur] = 0;
        __syncthreads();
    }
    if (tid == 0) {
        atomicAdd(&totals[0], total);
        atomicMax(&totals[1], k);
    }
}

__global__ void k_iota(uint32_t* p, uint32_t n) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = i;
}

// Schedule position of every task: xpos[sorted[p]] = p.
__global__ void k_invert(const uint32_t* sorted, uint32_t* xpos, uint32_t n) {
    const uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p < n) xpos[sorted[p]] = p;
}

// The downwind area A of a task from its faces in order: lane l of the 16-lane
// kernels sums the faces l, l + 16, ..., then their xor butterfly as seen from
// lane 0.
struct AreaTree {
    double part[kLanes];
    __device__ __forceinline__ AreaTree() {
#pragma unroll
        for (int l = 0; l < kLanes; l++) part[l] = 0.0;
    }
    __device__ __forceinline__ void add(uint32_t face, double term) {
#pragma unroll
        for (int u = 0; u < kLanes; u++)
            if ((uint32_t)u == face % kLanes) part[u] += term;
    }
    __device__ __forceinline__ double total() {
#pragma unroll
        for (int m = kLanes / 2; m > 0; m >>= 1) {
            double nxt[kLanes];
#pragma unroll
            for (int l = 0; l < kLanes; l++) nxt[l] = part[l] + part[l ^ m];
#pragma unroll
            for (int l = 0; l < kLanes; l++) part[l] = nxt[l];
        }
        return part[0];
    }
};

// The full schedule from the tasks sorted by (depth, direction, cell): task t =
// d*N + c at position p of level set k (start b, width W). Compiled: header,
// A, plane entries and overflow entries, each entry naming the upwind task's
// schedule position (one thread per task, faces in order; A as the same
// 16-lane butterfly the geometric kernels form). Geometric: the task record.
template <typename R>
__global__ void k_schedule(Geo g, double inv_aref, const uint32_t* sorted, const uint32_t* fstart, int kmax,
                           int compiled, const uint32_t* xpos, const uint32_t* ovf_start, uint4* hdr, R* Av,
                           Entry<R>* planes, Entry<R>* ovf, uint4* recs) {
    const uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
    if ((int64_t)p >= (int64_t)g.D * g.N) return;
    int a = 0, bb = kmax - 1;  // level set of position p
    while (a < bb) {
        int m = (a + bb + 1) >> 1;
        if (fstart[m] <= p) a = m;
        else bb = m - 1;
    }
    const uint32_t b = fstart[a], W = fstart[a + 1] - b;
    const uint32_t t = sorted[p];
    const uint32_t d = t / (uint32_t)g.N, c = t - d * (uint32_t)g.N;
    const uint32_t f0 = g.off[c], f1 = g.off[c + 1], ps = g.pslot[c];
    if (!compiled) {
        recs[p] = task_record(c, f0, f1, d, ps);
        return;
    }
    const double dx = g.dirs[3 * d], dy = g.dirs[3 * d + 1], dz = g.dirs[3 * d + 2];
    AreaTree A;
    uint32_t q = 0;
    const uint32_t os = ovf_start[(size_t)d * g.N + c];
    for (uint32_t f = f0; f < f1; f++) {
        const double4 fa = g.geo[f];
        const uint32_t nk = g.nk[f];
        const double dd = fdot(fa, dx, dy, dz);
        if (dd > 0.0) {
            A.add(f - f0, fa.w * inv_aref * dd);
        } else if (dd < 0.0 && (nk >> 30) == kKindLocal) {
            Entry<R> e;
            e.nb = xpos[(size_t)d * g.N + (nk & kNbrMask)];
            if constexpr (sizeof(R) == 8) e.pad = 0;
            e.w = (R)(fa.w * inv_aref * -dd);
            if (q < (uint32_t)kPlanes) {
                Entry<R>* base = planes + (size_t)kPlanes * b;
                if constexpr (sizeof(R) == 4) {
                    base[plane_off<R>(q, W, p - b)] = e;
                } else {
                    reinterpret_cast<uint32_t*>(base)[plane_nb_off(q, W, p - b)] = e.nb;
                    reinterpret_cast<double*>(base)[plane_w_off(q, W, p - b)] = e.w;
                }
            } else {
                ovf[os + q - kPlanes] = e;
            }
            q++;
        }
    }
    hdr[p] = make_uint4(c | (d << kCellBits), ps, q > (uint32_t)kPlanes ? os : 0u, q);
    Av[p] = (R)A.total();
}

// ---------------------------------------------------------------------------
// compaction of the full schedule to an active set (per sweep level);
// chunks[j] = {level set, first position, end position, 0}, never across level sets

__device__ __forceinline__ uint32_t task_cell(const uint4* tasks, uint32_t p) { return tasks[p].x & kCellMask; }

__global__ void __launch_bounds__(kBlock) k_compact_count(Geo g, const uint4* tasks, const uint4* chunks,
                                                          uint32_t nchunks, int lvl, uint32_t* counts) {
    const uint32_t j = blockIdx.x;
    if (j >= nchunks) return;
    const uint4 ch = chunks[j];
    __shared__ uint32_t total;
    if (threadIdx.x == 0) total = 0;
    __syncthreads();
    uint32_t n = 0;
    for (uint32_t p = ch.y + threadIdx.x; p < ch.z; p += kBlock) n += g.level[task_cell(tasks, p)] >= lvl ? 1u : 0u;
    for (int o = 32; o > 0; o >>= 1) n += __shfl_down(n, o);
    if (__lane_id() == 0 && n) atomicAdd(&total, n);
    __syncthreads();
    if (threadIdx.x == 0) counts[j] = total;
}

// Writes the active positions of each chunk, in order, relative to the start
// of their level set: idx[offset[j] + rank] = p - fstart[level].
__global__ void __launch_bounds__(kBlock) k_compact_write(Geo g, const uint4* tasks, const uint4* chunks,
                                                          uint32_t nchunks, const uint32_t* fstart, int lvl,
                                                          const uint32_t* offset, uint32_t* idx) {
    const uint32_t j = blockIdx.x;
    if (j >= nchunks) return;
    const uint4 ch = chunks[j];
    const uint32_t b = fstart[ch.x];
    __shared__ uint32_t wave_tot[kBlock / 64];
    uint32_t base = offset[j];
    const int lane = __lane_id(), wv = threadIdx.x / 64;
    for (uint32_t p0 = ch.y; p0 < ch.z; p0 += kBlock) {
        const uint32_t p = p0 + threadIdx.x;
        const bool act = p < ch.z && g.level[task_cell(tasks, p)] >= lvl;
        const unsigned long long m = __ballot(act);
        if (lane == 0) wave_tot[wv] = (uint32_t)__popcll(m);
        __syncthreads();
        uint32_t before = 0, all = 0;
        for (int w = 0; w < kBlock / 64; w++) {
            if (w < wv) before += wave_tot[w];
            all += wave_tot[w];
        }
        if (act) idx[base + before + (uint32_t)__popcll(m & ((1ull << lane) - 1ull))] = p - b;
        base += all;
        __syncthreads();
    }
}

// Compacted level starts: cstart[k] = offset of the level set's first chunk.
__global__ void k_compact_starts(const uint32_t* first_chunk, const uint32_t* offset, int kmax, uint32_t total,
                                 uint32_t* cstart) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k < kmax) cstart[k] = offset[first_chunk[k]];
    if (k == kmax) cstart[k] = total;
}

// ---------------------------------------------------------------------------
// replay kernels

// Geometric replay of one level set: `count` tasks, kLanes lanes per task; with
// an index list, task i is record recs[idx[i]].
template <typename R>
__global__ void __launch_bounds__(kBlock) k_sweep_rec(Geo g, Flux<R> fl, const uint4* recs, const uint32_t* idx,
                                                      uint32_t count) {
    const uint32_t i = xcd_block(blockIdx.x, gridDim.x) * kTasksPerBlock + threadIdx.x / kLanes;
    const uint32_t sub = threadIdx.x % kLanes;
    const bool valid = i < count;
    const uint32_t p = valid ? (idx ? idx[i] : i) : 0u;
    const uint4 r = valid ? recs[p] : make_uint4(0, 0, 0, 0);
    const uint32_t ps = r.w;
    const uint32_t c = r.x & kCellMask, d = r.z;
    const CellIn<R> ci = cell_inputs<R>(g, fl, c, d, ps);
    const uint32_t nfmax = wave_max(valid ? (r.x >> kCellBits) : 0u);
    double A;
    R inc;
    task_faces<R>(g, fl, valid, r, sub, nfmax, A, inc);
    if (valid && sub == 0) finish_task<R>(fl, (size_t)d * g.N + c, (size_t)d * g.N + c, inc, ci, (R)A);
}

// One task of the compiled replay in three steps, so that the kernels that
// solve several level sets in one workgroup can load the next level set's
// schedule data while the current level set's gathers are in flight:
//   load_task   the schedule data of the task at position p of a level set
//               of width W whose header, A and plane entries start at hdr,
//               Av and planes (independent loads, no dependence on X);
//   issue_task  the upwind X gathers (at the upwind tasks' schedule
//               positions; entries past the upwind count gather the task's
//               own X, a valid index, and are not summed) and the cell inputs;
//   finish_task_c  the upwind sum in entry order, the overflow entries, and
//               the stores (X at the task's schedule position `self`).
template <typename R>
struct TaskS {
    Entry<R> e[kPlanes];
    uint4 h;
    R A;
};

// Overflow entries of a task read together with its upwind gathers (the
// rest, rarer, one after the other).
constexpr int kEarlyOvf = 2;

template <typename R>
struct TaskG {
    R x[kPlanes];
    Entry<R> o[kEarlyOvf];  // first overflow entries (tasks with more than kPlanes upwind faces)
    CellIn<R> ci;
};

template <typename R>
__device__ __forceinline__ void load_task(TaskS<R>& t, const uint4* hdr, const R* Av, const Entry<R>* planes,
                                          uint32_t W, uint32_t p) {
    if constexpr (sizeof(R) == 4) {  // plane pairs: one 16-byte load per two entries
        const uint4* pp = reinterpret_cast<const uint4*>(planes);
#pragma unroll
        for (int h = 0; h < kPlanes / 2; h++) {
            const uint4 v = pp[(size_t)h * W + p];
            t.e[2 * h].nb = v.x;
            t.e[2 * h].w = __uint_as_float(v.y);
            t.e[2 * h + 1].nb = v.z;
            t.e[2 * h + 1].w = __uint_as_float(v.w);
        }
    } else {  // positions four to a 16-byte load, weights two
        const uint4* pn = reinterpret_cast<const uint4*>(planes);
        const double2* pw = reinterpret_cast<const double2*>(reinterpret_cast<const double*>(planes) + 6 * (size_t)W);
#pragma unroll
        for (int h = 0; h < kPlanes / 4; h++) {
            const uint4 v = pn[(size_t)h * W + p];
            t.e[4 * h].nb = v.x;
            t.e[4 * h + 1].nb = v.y;
            t.e[4 * h + 2].nb = v.z;
            t.e[4 * h + 3].nb = v.w;
        }
#pragma unroll
        for (int h = 0; h < kPlanes / 2; h++) {
            const double2 v = pw[(size_t)h * W + p];
            t.e[2 * h].w = v.x;
            t.e[2 * h + 1].w = v.y;
        }
    }
    t.h = hdr[p];
    t.A = Av[p];
}

template <typename R>
__device__ __forceinline__ void issue_task(TaskG<R>& G, const Geo& g, const Flux<R>& fl, const TaskS<R>& t,
                                           const Entry<R>* ovf, uint32_t self) {
    const uint32_t c = t.h.x & kCellMask, d = t.h.x >> kCellBits, ps = t.h.y, nup = t.h.w;
    if (nup > (uint32_t)kPlanes) {  // indexes clamped to the task's own overflow entries
        const uint32_t last = nup - kPlanes - 1u;
#pragma unroll
        for (int k = 0; k < kEarlyOvf; k++) G.o[k] = ovf[t.h.z + min((uint32_t)k, last)];
    }
    G.ci = cell_inputs<R>(g, fl, c, d, ps);
#pragma unroll
    for (int q = 0; q < kPlanes; q++) G.x[q] = fl.X[(uint32_t)q < nup ? t.e[q].nb : self];
}

template <typename R>
__device__ __forceinline__ void finish_task_c(const Geo& g, const Flux<R>& fl, const TaskS<R>& t, const TaskG<R>& G,
                                              const Entry<R>* ovf, uint32_t self) {
    const uint32_t c = t.h.x & kCellMask, d = t.h.x >> kCellBits, nup = t.h.w;
    R inc = 0;
#pragma unroll
    for (int q = 0; q < kPlanes; q++) inc += ((uint32_t)q < nup) ? t.e[q].w * G.x[q] : (R)0;
    if (nup > (uint32_t)kPlanes) {  // the overflow entries, in entry order
        R xo[kEarlyOvf];
#pragma unroll
        for (int k = 0; k < kEarlyOvf; k++) xo[k] = fl.X[G.o[k].nb];
#pragma unroll
        for (int k = 0; k < kEarlyOvf; k++)
            if ((uint32_t)(kPlanes + k) < nup) inc += G.o[k].w * xo[k];
        for (uint32_t q = kPlanes + kEarlyOvf; q < nup; q++) {
            const Entry<R> o = ovf[t.h.z + q - kPlanes];
            inc += o.w * fl.X[o.nb];
        }
    }
    finish_task<R>(fl, self, (size_t)d * g.N + c, inc, G.ci, t.A);
}

// The three steps back to back: the task at position p of the level set that
// starts at schedule position b and has width W.
template <typename R>
__device__ __forceinline__ void comp_task(const Geo& g, const Flux<R>& fl, const uint4* hdr, const R* Av,
                                          const Entry<R>* planes, const Entry<R>* ovf, uint32_t b, uint32_t W,
                                          uint32_t p) {
    TaskS<R> t;
    TaskG<R> G;
    load_task<R>(t, hdr, Av, planes, W, p);
    issue_task<R>(G, g, fl, t, ovf, b + p);
    finish_task_c<R>(g, fl, t, G, ovf, b + p);
}

// Compiled replay of one level set of width W: one lane per task. With an
// index list, lane i solves the task at position idx[i] of the level set.
template <typename R, int kRecBlock>
__global__ void __launch_bounds__(kRecBlock) k_sweep_comp(Geo g, Flux<R> fl, const uint4* hdr, const R* Av,
                                                          const Entry<R>* planes, const Entry<R>* ovf, uint32_t b,
                                                          uint32_t W, const uint32_t* idx, uint32_t count) {
    const uint32_t i = xcd_block(blockIdx.x, gridDim.x) * kRecBlock + threadIdx.x;
    if (i >= count) return;
    comp_task<R>(g, fl, hdr, Av, planes, ovf, b, W, idx ? idx[i] : i);
}

// Lanes of the workgroup that solves a run of narrow level sets: at most this
// many active tasks per level set (FP64 tasks hold twice the registers).
template <typename R>
constexpr int run_block() {
    return sizeof(R) == 4 ? kRunBlock : kRunBlock / 2;
}

// Compiled replay of a run of consecutive narrow level sets (at most
// run_block<R>() active tasks each) by one workgroup, level set after level
// set, with a workgroup barrier in between: every wave of the workgroup runs
// on one CU, whose L1 is coherent within the workgroup, so the X stored for
// one level set is seen by the next after the barrier. run[j] = {first
// position b, width W, first index list entry, active count} of the run's
// j-th level set; without an index list entry i is position i.
// Software pipelined: while level set j's gathers are in flight, level set
// j+1's schedule data, level set j+2's index entries and run[j+3] are loaded,
// none of which level set j waits for. Every load is unconditional (lanes
// without a task, and level sets past the run's end, read a valid clamped
// entry) so that the waits stay exact; only the stores are predicated.
template <typename R>
__global__ void __launch_bounds__(run_block<R>()) k_sweep_comp_run(Geo g, Flux<R> fl, const uint4* __restrict__ hdr,
                                                                   const R* __restrict__ Av,
                                                                   const Entry<R>* __restrict__ planes,
                                                                   const Entry<R>* __restrict__ ovf,
                                                                   const uint32_t* __restrict__ idx,
                                                                   const uint4* __restrict__ run, int levels) {
    const uint32_t i = threadIdx.x;
    const int last = levels - 1;
    // position of lane i in level set r (a valid position for every lane)
    auto pos = [&](const uint4& r) -> uint32_t {
        const uint32_t k = min(i, r.w - 1u);
        return idx ? idx[r.z + k] : k;
    };
    uint4 r = run[0];
    uint32_t p = pos(r);
    TaskS<R> cur;
    load_task<R>(cur, hdr + r.x, Av + r.x, planes + (size_t)kPlanes * r.x, r.y, p);
    uint4 rn = run[min(1, last)];
    uint32_t pn = pos(rn);
    uint4 rnn = run[min(2, last)];
    for (int j = 0; j < levels; j++) {
        TaskG<R> G;
        issue_task<R>(G, g, fl, cur, ovf, r.x + p);
        TaskS<R> nxt;
        load_task<R>(nxt, hdr + rn.x, Av + rn.x, planes + (size_t)kPlanes * rn.x, rn.y, pn);
        const uint32_t pnn = pos(rnn);
        const uint4 rnnn = run[min(j + 3, last)];
        if (i < r.w) finish_task_c<R>(g, fl, cur, G, ovf, r.x + p);
        __syncthreads();
        r = rn;
        p = pn;
        cur = nxt;
        rn = rnn;
        pn = pnn;
        rnn = rnnn;
    }
}

// Direction sweeps (compiled replay): the tasks of one direction depend only
// on tasks of the same direction, so one workgroup per direction solves its
// direction's whole sweep, level set after level set with a workgroup barrier
// in between, and no dependency crosses workgroups or launches.
//
// X is stored in each direction's Kahn order (level set, then class of upwind
// counts, then cell): the q-th task of direction d has X index d*N + q. The
// last kRing values a workgroup solved sit in an LDS ring (slot q mod kRing).
// What a task reads of them was known when the schedule was built, so the
// schedule names LDS words, not tasks, and a level set costs one round of LDS
// reads between two barriers. Level sets are cut into tiles of up to 64 tasks,
// the work of one wave, dealt to the waves in turn. A tile's blob, planes of
// 16 bytes per task and then two lists:
//   slot planes    8 halfwords per task: {cell | upwind count << 25 (two
//                  halfwords), periodic source, entries 0-4}, {entries 5-12}
//   weight planes  {A, weight of entry 0, ...}: 4 (FP32) or 2 (FP64) values
//   far list       X indices of upwind values that the ring no longer holds
//                  (and, with kFarPeriodic, P indices of periodic sources)
//   extra list     weights, then words, of entries past the planes
// in the order S0 W0 W1 S1 W2 .. (FP64: S0 W0 W1 W2 S1 W3 ..), as many planes
// as the tile's largest upwind count needs (plane loads past them return 0:
// word 0, which holds 0, with weight 0). The wave loads the far values itself
// and puts them, as the extra entries, into a buffer of its own in LDS, whose
// words the entries name like the ring's. The tile's wave is fixed by its
// place in the direction, hence so are these words.
//
// Bound: a level set's chain (barrier, LDS reads, the sum in entry order, one
// division, LDS write) while the schedule streams past from HBM. A wave loads
// tile i+2's planes and tile i+1's cell inputs and far values before it waits
// for tile i's level set, in registers that no copy moves (the loop is
// unrolled over three sets), so no memory wait enters the chain. One wave per
// tile instead of one lane per task of a level set keeps 16 x 2 tiles in
// flight per CU where a level set holds 25 to 400 tasks. The wave that solved
// a tile passes the level set's end before it stores and loads anything, which
// else stands between the others and the next level set (0.62 -> 0.42 us per
// level set of 25 tasks). Per sweep, against one lane per task of a level set
// with its data two level sets ahead: 25.0 -> 7.1 ms on 2 M clustered cells x
// 84 directions (1.14 us per level set of 340 tasks, 2.3 TB/s), 2.41 -> 0.77
// ms on 262144 cells, FP64 2.95 -> 1.1 ms, 1.70 -> 0.39 ms on 23457 cells x 32.
//
// Far values: the load for tile i+1 goes out after this wave solved tile i-1;
// a wave's stores go out before it begins its next tile and are complete when
// it uses a load issued after them, at most two of its tiles later. So every
// value more than 5 * kWaves tiles and two level sets behind is in memory, and
// the ring holds more than that unless a level set is wider than kRing / 4:
// such directions (`wide`) complete their stores at every barrier and load
// their far values after it.
//
// Waits: every wave passes levels - 1 barriers, whatever tiles it has.
// A restricted sweep (lvl > 0; the host passes 0 when every cell is active)
// passes every task: a task whose cell is below level lvl is not solved and
// puts its stored X into the ring. Same arithmetic per task as the other
// replays.
template <typename R>
struct DirShape {
    static constexpr int kWaves = sizeof(R) == 4 ? 16 : 12;  // FP64: 168 VGPRs a wave
    static constexpr uint32_t kRing = sizeof(R) == 4 ? 32768u : 16384u;  // 128 KiB
    static constexpr int kPer = 16 / (int)sizeof(R);                     // values per weight plane
    static constexpr int kWPlanes = sizeof(R) == 4 ? 4 : 7;              // A and 13 weights
    static constexpr int kS1 = sizeof(R) == 4 ? 3 : 4;                   // place of the second slot plane
    static constexpr uint32_t kRingAt = 64;                              // words 0-63: 0
    static constexpr uint32_t kBufs = kRingAt + kRing;
    static constexpr uint32_t kBuf = 256 + 512 / (uint32_t)sizeof(R);    // 128 far, 128 weights, 128 words of 4 bytes
    static constexpr uint32_t kWords = kBufs + kWaves * kBuf;
    // planes that hold up to n entries
    __host__ __device__ static constexpr uint32_t planes(uint32_t n) { return ssw::tile_planes(sizeof(R) == 4, n); }
    // place of weight plane j
    __host__ __device__ static constexpr uint32_t wplane(uint32_t j) { return j + 1 < (uint32_t)kS1 ? j + 1 : j + 2; }
};
constexpr uint32_t kDirEntries = 13;           // entries in the planes; a task with more has 12 there and the rest
                                               // in the extra list from the position that entry 12's word gives
constexpr uint32_t kDirCap = 64;               // far and extra entries of a tile of more than one task
constexpr uint32_t kFarPeriodic = 0x80000000u;
constexpr int kStream = 2;                     // non-temporal: the schedule is read once per sweep and leaves the L2
                                               // to the cells' lines (13.8 -> 12.9 ms per sweep on 2 M cells)

// Classes of upwind counts by which a level set's tasks are sorted, so that a
// tile's tasks need about the same planes.
__host__ __device__ __forceinline__ uint32_t dir_class(uint32_t nup) {
    return (nup > 5) + (nup > 7) + (nup > 9) + (nup > 11);
}

typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// A tile, 32 bytes: blob offset in 16-byte units (two words), first q, end of
// the level set's q, level set, tasks | far << 8 | extra << 16 | planes << 24.
struct DirTile {
    uint64_t off;
    uint32_t q0, hi, k, cnt, nfar, nex, np;
};

template <typename R>
struct DirRegs {
    u32x4 s[2];
    uint32_t w[14 * sizeof(R) / 4];  // A and 13 weights (a register that nothing reads would be taken for another
                                     // use while its load is still on the way, and waited for)
    uint32_t far;     // far list entry of this lane
    R exw;            // extra entry of this lane
    uint32_t exs;
    SA<R> sa;         // one tile ahead: cell inputs, far value
    R fv;
    R off, xold;      // general variant only
    uint32_t lev;
    DirTile t;
};

template <typename R, bool kGeneral>
__global__ void __launch_bounds__(64 * DirShape<R>::kWaves) k_sweep_dir(Geo g, Flux<R> fl,
                                                                        const uint4* __restrict__ blob,
                                                                        const uint4* __restrict__ tiles,
                                                                        const uint4* __restrict__ dirs,
                                                                        const SA<R>* __restrict__ sas,
                                                                        const uint8_t* __restrict__ levs, int lvl) {
    using S = DirShape<R>;
    constexpr uint32_t kRing = S::kRing;
    __shared__ R lds[S::kWords];
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t d = blockIdx.x;
    const uint4 di = dirs[d];  // first tile, tiles, level sets, wide
    const uint32_t ntiles = di.y, levels = di.z;
    const bool wide = di.w != 0;
    const uint32_t dN = d * (uint32_t)g.N;
    R* const buf = lds + S::kBufs + w * S::kBuf;
    uint32_t* const bufs = reinterpret_cast<uint32_t*>(buf + 256);
    if (threadIdx.x < 64) lds[threadIdx.x] = (R)0;
    __syncthreads();

    // descriptor of the wave's i-th tile, as vector loads (scalar ones would
    // be waited for at the barriers); past the last tile it reads the last one
    uint4 da, db;
    auto fetch = [&](uint32_t i) {
        uint32_t at = 2u * (di.x + min(w + i * S::kWaves, ntiles - 1u));
        asm volatile("" : "+v"(at));
        da = tiles[at];
        db = tiles[at + 1u];
    };
    auto uni = [](uint32_t v) -> uint32_t { return __builtin_amdgcn_readfirstlane(v); };
    auto decode = [&](DirTile& t, uint32_t i) {
        const bool any = w + i * S::kWaves < ntiles;
        const uint32_t c = any ? uni(db.y) : 0u;
        t.off = (uint64_t)uni(da.x) | ((uint64_t)uni(da.y) << 32);
        t.q0 = uni(da.z);
        t.hi = uni(da.w);
        t.k = uni(db.x);
        t.cnt = c & 255u;
        t.nfar = (c >> 8) & 255u;
        t.nex = (c >> 16) & 255u;
        t.np = c >> 24;
    };
    auto rsrc = [&](const uint4* p, uint32_t bytes) {
        return __builtin_amdgcn_make_buffer_rsrc(const_cast<uint4*>(p), 0, (int)bytes, 0x00027000);
    };
    auto ex_units = [](uint32_t nex) { return (nex * (uint32_t)sizeof(R) + 15u) / 16u; };
    // the planes and lists of a tile (loads past them return 0)
    auto load = [&](DirRegs<R>& T) {
        const DirTile& t = T.t;
        const uint4* p = blob + t.off;
        const auto rp = rsrc(p, t.np * t.cnt * 16u);
        const uint32_t o = min(lane, max(t.cnt, 1u) - 1u) * 16u, st = t.cnt * 16u;
        T.s[0] = __builtin_amdgcn_raw_buffer_load_b128(rp, o, 0, kStream);
        p += t.np * t.cnt;
        T.far = __builtin_amdgcn_raw_buffer_load_b32(rsrc(p, t.nfar * 4u), lane * 4u, 0, kStream);
        __builtin_amdgcn_sched_barrier(0);  // loads return in order: what is needed first goes out first
#pragma unroll
        for (int j = 0; j < S::kWPlanes; j++) {
            if (j + 1 == S::kS1) T.s[1] = __builtin_amdgcn_raw_buffer_load_b128(rp, o + S::kS1 * st, 0, kStream);
            if (sizeof(R) == 4 && j == S::kWPlanes - 1) {
                const u32x2 v = __builtin_amdgcn_raw_buffer_load_b64(rp, o + S::wplane(j) * st, 0, kStream);
                T.w[4 * j] = v.x;
                T.w[4 * j + 1] = v.y;
            } else {
                const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(rp, o + S::wplane(j) * st, 0, kStream);
#pragma unroll
                for (int m = 0; m < 4; m++) T.w[4 * j + m] = v[m];
            }
        }
        p += (t.nfar + 3u) / 4u;
        if constexpr (sizeof(R) == 4) {
            T.exw = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rsrc(p, t.nex * 4u), lane * 4u, 0, kStream));
        } else {
            const u32x2 v = __builtin_amdgcn_raw_buffer_load_b64(rsrc(p, t.nex * 8u), lane * 8u, 0, kStream);
            T.exw = __hiloint2double((int)v.y, (int)v.x);
        }
        p += ex_units(t.nex);
        T.exs = __builtin_amdgcn_raw_buffer_load_b32(rsrc(p, t.nex * 4u), lane * 4u, 0, kStream);
    };
    auto far_value = [&](uint32_t at) -> R {
        const R* src = (at & kFarPeriodic) ? fl.P : fl.X;
        return src[at & ~kFarPeriodic];
    };
    auto pre = [&](DirRegs<R>& T) {
        const uint32_t p = dN + T.t.q0 + min(lane, max(T.t.cnt, 1u) - 1u);
        T.sa = sas[p];
        T.fv = far_value(T.far);
        if (kGeneral) {
            T.off = fl.offI ? fl.offI[(size_t)d * g.N + (T.s[0].x & kCellMask)] : (R)0;
            T.lev = lvl > 0 ? levs[p] : 0u;
            T.xold = lvl > 0 ? fl.X[p] : (R)0;
        }
    };
    uint32_t at_level = 0;
    auto pass_to = [&](uint32_t k) {
        while (at_level < k) {
            if (wide) __builtin_amdgcn_s_waitcnt(0);
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
            at_level++;
        }
    };
    auto slot = [&](const DirRegs<R>& T, int e) -> uint32_t {  // entry e's LDS word (-1: the periodic source's)
        const int h = e + 3;
        const uint32_t v = T.s[h / 8][(h % 8) / 2];
        return (h & 1) ? v >> 16 : v & 0xFFFFu;
    };
    auto weight = [&](const DirRegs<R>& T, int i) -> R {  // 0: A, 1 + e: entry e's
        if constexpr (sizeof(R) == 4) return __uint_as_float(T.w[i]);
        else return __hiloint2double((int)T.w[2 * i + 1], (int)T.w[2 * i]);
    };
    // next: level set of the wave's next tile (its own, if it has none)
    auto solve = [&](DirRegs<R>& T, uint32_t next) {
        const DirTile& t = T.t;
        if (t.cnt == 0) return;
        // the wave's buffer, before it waits for the level set (far values of a
        // wide direction after it); each load in a branch of its own, so that
        // no wait for it enters the others
        if (t.nex) {
            buf[128u + lane] = T.exw;
            bufs[lane] = T.exs;
            if (t.nex > 64u) {  // one task with more than 64 entries
                const uint4* p = blob + t.off + t.np * t.cnt + (t.nfar + 3u) / 4u;
                if (64u + lane < t.nex) {
                    buf[192u + lane] = reinterpret_cast<const R*>(p)[64u + lane];
                    bufs[64u + lane] = reinterpret_cast<const uint32_t*>(p + ex_units(t.nex))[64u + lane];
                }
            }
        }
        const uint32_t hdr = T.s[0].x, q = t.q0 + lane;
        const bool more = (hdr >> kCellBits) > kDirEntries;
        uint32_t at[kDirEntries + 1];  // LDS words of the periodic source and the entries
#pragma unroll
        for (int e = 0; e <= (int)kDirEntries; e++)
            at[e] = (e == (int)kDirEntries && more) ? 0u : slot(T, e - 1);
        if (sizeof(R) == 4) {  // formed before the barrier (FP64 has no registers for them)
#pragma unroll
            for (int e = 0; e <= (int)kDirEntries; e++) asm volatile("" : "+v"(at[e]));
        }
        if (wide) {
            pass_to(t.k);
            for (uint32_t j = 0; j < t.nfar; j += 64u) {
                const uint32_t* list = reinterpret_cast<const uint32_t*>(blob + t.off + t.np * t.cnt);
                if (j + lane < t.nfar) buf[j + lane] = far_value(list[j + lane]);
            }
        } else {
            buf[lane] = T.fv;
            if (t.nfar > 64u) {
                const uint32_t* list = reinterpret_cast<const uint32_t*>(blob + t.off + t.np * t.cnt);
                if (64u + lane < t.nfar) buf[64u + lane] = far_value(list[64u + lane]);
            }
            pass_to(t.k);
        }
        // all reads in one batch: those past the planes read word 0
        R x[kDirEntries + 1];
#pragma unroll
        for (int e = 0; e <= (int)kDirEntries; e++) x[e] = lds[at[e]];
        R inc = 0;
#pragma unroll
        for (int e = 0; e < (int)kDirEntries; e++) inc += weight(T, 1 + e) * x[1 + e];
        if (t.nex && more) {
            const uint32_t nup = hdr >> kCellBits;
            const uint32_t first = slot(T, (int)kDirEntries - 1) - (kDirEntries - 1u);
            for (uint32_t e0 = kDirEntries - 1u; e0 < nup; e0 += 4u) {  // four reads in flight
                R v[4], y[4];
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const uint32_t e = first + min(e0 + j, nup - 1u);
                    v[j] = buf[128u + e];
                    y[j] = lds[bufs[e]];
                }
#pragma unroll
                for (int j = 0; j < 4; j++) inc += e0 + j < nup ? v[j] * y[j] : (R)0;
            }
        }
        CellIn<R> ci;
        ci.src = T.sa.x;
        ci.att = T.sa.y;
        ci.per = x[0];
        ci.off = kGeneral ? T.off : (R)0;
        const R A = weight(T, 0);
        const size_t oi = (size_t)d * g.N + (hdr & kCellMask);
        bool act = lane < t.cnt;
        R xv;
        if (kGeneral) {
            const bool lev = T.lev >= (uint32_t)lvl;
            if (act && lev) {
                const R out = outgoing_rate<R, true>(fl, oi, inc, ci);
                xv = (A > (R)0) ? out / A : (R)0;
            } else {
                xv = T.xold;
            }
            if (act && q + kRing >= t.hi) lds[S::kRingAt + (q & (kRing - 1u))] = xv;
            act = act && lev;
        } else {
            const R out = outgoing_rate<R, false>(fl, oi, inc, ci);
            xv = (A > (R)0) ? out / A : (R)0;
            if (act && q + kRing >= t.hi) lds[S::kRingAt + (q & (kRing - 1u))] = xv;
        }
        // the level set's end before anything that does not belong to it: the
        // stores and the next tiles' loads run beside the next level set
        if (!wide && next > t.k) pass_to(t.k + 1u);
        if (act) {
            fl.X[dN + q] = xv;
            fl.I[dN + q] = inc;
        }
    };
    // iteration i: tile i+2's planes, tile i+1's inputs, tile i
    DirRegs<R> T0, T1, T2;
    fetch(0);
    decode(T0.t, 0);
    load(T0);
    fetch(1);
    decode(T1.t, 1);
    fetch(2);
    __builtin_amdgcn_sched_barrier(0);  // as in the loop: its waits count the loads after a fetch
    load(T1);
    __builtin_amdgcn_sched_barrier(0);
    pre(T0);
    __builtin_amdgcn_sched_barrier(0);
    auto step = [&](DirRegs<R>& a, DirRegs<R>& b, DirRegs<R>& c, uint32_t i) {
        decode(c.t, i + 2);
        fetch(i + 3);
        __builtin_amdgcn_sched_barrier(0);
        load(c);
        __builtin_amdgcn_sched_barrier(0);
        pre(b);
        __builtin_amdgcn_sched_barrier(0);
        solve(a, b.t.cnt ? b.t.k : a.t.k);
    };
    const uint32_t mine = ntiles > w ? (ntiles - w + S::kWaves - 1u) / S::kWaves : 0u;
    for (uint32_t i = 0; i < mine; i += 3) {
        step(T0, T1, T2, i);
        step(T1, T2, T0, i + 1);
        step(T2, T0, T1, i + 2);
    }
    pass_to(levels - 1u);
}

// The inputs of a direction sweep in X's order, before each sweep: every
// task's {source, attenuation} and, in a restricted sweep, its cell's level.
// Their gathers cost a CU one line at a time (44 ns per 64 tasks); here all
// CUs share them, in the sweep itself only the D that run it. With I stored in
// X's order likewise (chemistry gathers it), a sweep of 262144 cells x 84
// directions went from 1.24 to 0.90 ms, and one of 2 M clustered cells
// from 12.1 to 8.3 ms, these passes included (the gather in k_chemistry adds
// 1.4 ms there).
template <typename R>
__global__ void __launch_bounds__(kBlock) k_dir_inputs(const uint32_t* __restrict__ cell, const SA<R>* __restrict__ sa,
                                                       const uint8_t* __restrict__ level, SA<R>* __restrict__ sas,
                                                       uint8_t* __restrict__ levs, uint32_t n) {
    // a die takes consecutive positions: the level sets that cross the same
    // cells' lines share its L2
    const uint32_t p = xcd_block(blockIdx.x, gridDim.x) * kBlock + threadIdx.x;
    if (p >= n) return;
    const uint32_t c = cell[p];
    sas[p] = sa[c];
    if (levs) levs[p] = level[c];
}

// The lowest timestep level of the cells (direction sweeps: a restricted
// sweep whose active set is every cell runs as a full one).
__global__ void k_min_level(const uint8_t* __restrict__ level, int64_t n, uint32_t* out) {
    uint32_t m = 255u;
    for (int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; c < n; c += (int64_t)gridDim.x * blockDim.x)
        m = min(m, (uint32_t)level[c]);
    for (int o = 32; o > 0; o >>= 1) m = min(m, (uint32_t)__shfl_down((int)m, o));
    if (__lane_id() == 0) atomicMin(out, m);
}

// --- the direction sweeps' schedule, built once per grid ----------------------

// Sort key of every task t = d*N + c: direction, level set, class.
__global__ void k_dir_keys(const uint32_t* __restrict__ depth, const uint8_t* __restrict__ nup, uint32_t N,
                           uint32_t kmax, uint32_t n, uint32_t* __restrict__ key, uint32_t* __restrict__ val) {
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n) return;
    key[t] = ((t / N * kmax + depth[t]) << 3) | dir_class(nup[t]);
    val[t] = t;
}

// First position of every (direction, level set) in the sorted keys
// (start[d * kmax + k], which starts as kNone), the X index of every task, and
// the cell at every X index.
__global__ void k_dir_starts(const uint32_t* __restrict__ key, const uint32_t* __restrict__ sorted, uint32_t n,
                             uint32_t N, uint32_t* __restrict__ start, uint32_t* __restrict__ xpos,
                             uint32_t* __restrict__ cell) {
    const uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n) return;
    const uint32_t k = key[p] >> 3;
    if (p == 0 || (key[p - 1] >> 3) != k) start[k] = p;
    xpos[sorted[p]] = p;
    cell[p] = sorted[p] % N;
}

// End position of level set k of direction d in the sorted order (the level
// sets of a direction are its first ones, without gaps).
__device__ __forceinline__ uint32_t dir_level_end(const uint32_t* start, uint32_t d, uint32_t k, uint32_t kmax,
                                                  uint32_t N) {
    const uint32_t e = k + 1 < kmax ? start[d * kmax + k + 1] : kNone;
    return e != kNone ? e : (d + 1u) * N;
}

// Groups of up to 64 consecutive tasks of one level set: {first position,
// tasks, end of the level set, level set} at first[d * kmax + k] ...
__global__ void k_dir_groups(const uint32_t* __restrict__ start, const uint32_t* __restrict__ first, uint32_t N,
                             uint32_t D, uint32_t kmax, uint4* __restrict__ groups) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= D * kmax || start[i] == kNone) return;
    const uint32_t k = i % kmax, e = dir_level_end(start, i / kmax, k, kmax, N);
    uint32_t j = first[i];
    for (uint32_t p = start[i]; p < e; p += 64u) groups[j++] = make_uint4(p, min(64u, e - p), e, k);
}

// Entries of every task that its far list names: upwind values older than the
// ring at the end of the task's level set, and the periodic source. A wave
// takes 64 cells and kFluxDirs directions, as k_fluxes does.
template <typename R>
__global__ void __launch_bounds__(1024) k_dir_far(Geo g, const uint32_t* __restrict__ xpos,
                                                  const uint32_t* __restrict__ depth,
                                                  const uint32_t* __restrict__ start, uint32_t kmax,
                                                  uint8_t* __restrict__ nfar) {
    const uint32_t lane = threadIdx.x % kFluxCells;
    const uint32_t w = __builtin_amdgcn_readfirstlane(threadIdx.x / kFluxCells);
    const int64_t c0 = (int64_t)blockIdx.x * kFluxCells + lane;
    if (c0 >= g.N) return;
    const uint32_t c = (uint32_t)c0, N = (uint32_t)g.N;
    uint32_t hi[kFluxDirs], n[kFluxDirs];
#pragma unroll
    for (int j = 0; j < kFluxDirs; j++) {
        const uint32_t d = min(w * kFluxDirs + j, (uint32_t)g.D - 1u);
        hi[j] = dir_level_end(start, d, depth[(size_t)d * N + c], kmax, N);
        n[j] = (g.Nper && g.pslot[c] != kNone) ? 1u : 0u;
    }
    for (uint32_t f = g.off[c]; f < g.off[c + 1]; f++) {
        const double4 a = g.geo[f];
        const uint32_t nk = g.nk[f];
        if ((nk >> 30) != kKindLocal) continue;
#pragma unroll
        for (int j = 0; j < kFluxDirs; j++) {
            const uint32_t d = min(w * kFluxDirs + j, (uint32_t)g.D - 1u);
            if (fdot(a, g.dirs[3 * d], g.dirs[3 * d + 1], g.dirs[3 * d + 2]) < 0.0 &&
                xpos[(size_t)d * N + (nk & kNbrMask)] + DirShape<R>::kRing < hi[j])
                n[j]++;
        }
    }
#pragma unroll
    for (int j = 0; j < kFluxDirs; j++)
        if ((int)(w * kFluxDirs) + j < g.D) nfar[(size_t)(w * kFluxDirs + j) * N + c] = (uint8_t)n[j];
}

__device__ __forceinline__ uint32_t wave_scan(uint32_t v) {  // inclusive
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t u = (uint32_t)__shfl_up((int)v, o);
        if ((int)__lane_id() >= o) v += u;
    }
    return v;
}

// 16-byte units of n values of b bytes.
__host__ __device__ __forceinline__ uint32_t units16(uint32_t n, uint32_t b) { return (n * b + 15u) / 16u; }

// The tiles of one group, one wave: consecutive tasks while their far and
// extra entries stay within kDirCap (a task with more is a tile of its own).
// Calls tile(first lane, tasks, far, extra, planes, units) for each.
template <typename R, typename F>
__device__ __forceinline__ void dir_tiles(uint32_t cnt, uint32_t nup, uint32_t far, uint32_t pf, uint32_t pe, F tile) {
    const uint32_t lane = __lane_id();
    uint32_t a = 0;
    while (a < cnt) {
        const uint32_t bf = a ? (uint32_t)__shfl((int)pf, a - 1) : 0u, be = a ? (uint32_t)__shfl((int)pe, a - 1) : 0u;
        const unsigned long long over =
            __ballot(lane > a && lane < cnt && (pf - bf > kDirCap || pe - be > kDirCap));
        const uint32_t e = over ? (uint32_t)__ffsll((long long)over) - 1u : cnt;
        const uint32_t nf = (uint32_t)__shfl((int)pf, e - 1) - bf, ne = (uint32_t)__shfl((int)pe, e - 1) - be;
        const uint32_t np = DirShape<R>::planes(wave_max(lane >= a && lane < e ? nup : 0u));
        const uint32_t units = np * (e - a) + units16(nf, 4) + units16(ne, sizeof(R)) + units16(ne, 4);
        tile(a, e - a, bf, nf, be, ne, np, units);
        a = e;
    }
}

__device__ __forceinline__ uint32_t dir_extra(uint32_t nup) { return nup > kDirEntries ? nup - (kDirEntries - 1u) : 0u; }

// Tiles and blob units of every group, one wave per group.
template <typename R>
__global__ void __launch_bounds__(kBlock) k_dir_tile_count(const uint4* __restrict__ groups, uint32_t ng,
                                                           const uint32_t* __restrict__ sorted,
                                                           const uint8_t* __restrict__ nups,
                                                           const uint8_t* __restrict__ nfars, uint32_t* __restrict__ gt,
                                                           uint64_t* __restrict__ gu) {
    const uint32_t i = blockIdx.x * (kBlock / 64) + threadIdx.x / 64, lane = __lane_id();
    if (i >= ng) return;
    const uint4 G = groups[i];
    const uint32_t t = sorted[G.x + min(lane, G.y - 1u)];
    const uint32_t nup = nups[t], far = lane < G.y ? nfars[t] : 0u;
    uint32_t nt = 0;
    uint64_t nu = 0;
    dir_tiles<R>(G.y, nup, far, wave_scan(far), wave_scan(lane < G.y ? dir_extra(nup) : 0u),
                 [&](uint32_t, uint32_t, uint32_t, uint32_t, uint32_t, uint32_t, uint32_t, uint32_t units) {
                     nt++;
                     nu += units;
                 });
    if (lane == 0) {
        gt[i] = nt;
        gu[i] = nu;
    }
}

// Writes task li of a tile of cnt tasks and np planes at `base`: header,
// entries in face order, A as the 16-lane kernels form it. word(x) gives the
// LDS word that holds the upwind X of index x, or kNone: then x goes to the
// far list (at position fp on) and the entry names that place in the wave's
// buffer (word `buf` on). Entries past the planes go to the extra list (at
// position ep on).
template <typename R, typename W>
__device__ __forceinline__ void fill_task(const Geo& g, double inv_aref, uint32_t c, uint32_t d, uint32_t nup,
                                          const uint32_t* __restrict__ xpos, uint4* base, uint32_t np, uint32_t cnt,
                                          uint32_t li, uint32_t* flist, uint32_t fp, uint32_t buf, R* exw,
                                          uint32_t* exs, uint32_t ep, W word) {
    using S = DirShape<R>;
    const uint32_t inplane = nup > kDirEntries ? kDirEntries - 1u : kDirEntries;
    auto put_slot = [&](uint32_t h, uint32_t v) {  // halfword h of the slot planes
        reinterpret_cast<uint16_t*>(base + (h < 8 ? 0u : S::kS1 * cnt) + li)[h % 8] = (uint16_t)v;
    };
    auto put_weight = [&](uint32_t j, R v) {
        reinterpret_cast<R*>(base + S::wplane(j / S::kPer) * cnt + li)[j % S::kPer] = v;
    };
    const double dx = g.dirs[3 * d], dy = g.dirs[3 * d + 1], dz = g.dirs[3 * d + 2];
    const uint32_t hdr = c | (nup << kCellBits);
    put_slot(0, hdr & 0xFFFFu);
    put_slot(1, hdr >> 16);
    const uint32_t ps = g.pslot[c];
    if (g.Nper && ps != kNone) {
        flist[fp] = kFarPeriodic | (uint32_t)((size_t)d * g.Nper + ps);
        put_slot(2, buf + fp++);
    } else {
        put_slot(2, 0u);
    }
    AreaTree A;
    uint32_t q = 0;
    const uint32_t f0 = g.off[c], f1 = g.off[c + 1];
    for (uint32_t f = f0; f < f1; f++) {
        const double4 fa = g.geo[f];
        const uint32_t nk = g.nk[f];
        const double dd = fdot(fa, dx, dy, dz);
        if (dd > 0.0) {
            A.add(f - f0, fa.w * inv_aref * dd);
        } else if (dd < 0.0 && (nk >> 30) == kKindLocal) {
            const R wt = (R)(fa.w * inv_aref * -dd);
            const uint32_t x = xpos[(size_t)d * g.N + (nk & kNbrMask)];
            uint32_t at = word(x);
            if (at == kNone) {
                flist[fp] = x;
                at = buf + fp++;
            }
            if (q < inplane) {
                put_slot(3 + q, at);
                put_weight(1 + q, wt);
            } else {
                exw[ep + q - inplane] = wt;
                exs[ep + q - inplane] = at;
            }
            q++;
        }
    }
    put_weight(0, (R)A.total());
    // the rest of the tile's planes: word 0, weight 0
    const bool two = np > (uint32_t)S::kS1;
    const uint32_t nw = (np - (two ? 2u : 1u)) * S::kPer;
    for (uint32_t e = min(q, inplane); e < (two ? 13u : 5u); e++) put_slot(3 + e, 0u);
    for (uint32_t e = min(q, inplane); e + 1 < nw; e++) put_weight(1 + e, (R)0);
    if (nup > kDirEntries) put_slot(3 + kDirEntries - 1u, ep);
}

// The tiles and their blobs, one wave per group, one lane per task; the
// entries in face order, A as the 16-lane kernels form it. tfirst[d]: first
// tile of direction d (a tile's wave is its place in the direction mod
// kWaves).
template <typename R>
__global__ void __launch_bounds__(kBlock) k_dir_tile_fill(Geo g, double inv_aref, const uint4* __restrict__ groups,
                                                          uint32_t ng, const uint32_t* __restrict__ sorted,
                                                          const uint8_t* __restrict__ nups,
                                                          const uint8_t* __restrict__ nfars,
                                                          const uint32_t* __restrict__ xpos,
                                                          const uint32_t* __restrict__ ts, const uint64_t* __restrict__ us,
                                                          const uint32_t* __restrict__ tfirst, uint4* __restrict__ blob,
                                                          uint4* __restrict__ tiles) {
    using S = DirShape<R>;
    const uint32_t i = blockIdx.x * (kBlock / 64) + threadIdx.x / 64, lane = __lane_id();
    if (i >= ng) return;
    const uint4 G = groups[i];
    const uint32_t t = sorted[G.x + min(lane, G.y - 1u)];
    const uint32_t N = (uint32_t)g.N, d = t / N, c = t - d * N, dN = d * N;
    const uint32_t nup = nups[t], far = lane < G.y ? nfars[t] : 0u;
    const uint32_t pf = wave_scan(far), pe = wave_scan(lane < G.y ? dir_extra(nup) : 0u);
    uint32_t tile = ts[i];
    uint64_t off = us[i];
    dir_tiles<R>(G.y, nup, far, pf, pe, [&](uint32_t a, uint32_t cnt, uint32_t bf, uint32_t nf, uint32_t be, uint32_t ne,
                                            uint32_t np, uint32_t units) {
        uint4* const base = blob + off;
        if (lane == 0) {
            tiles[2 * (size_t)tile] = make_uint4((uint32_t)off, (uint32_t)(off >> 32), G.x + a - dN, G.z - dN);
            tiles[2 * (size_t)tile + 1] = make_uint4(G.w, cnt | (nf << 8) | (ne << 16) | (np << 24), 0u, 0u);
        }
        if (lane >= a && lane < a + cnt) {
            const uint32_t buf = S::kBufs + ((tile - tfirst[d]) % S::kWaves) * S::kBuf;
            uint4* const lists = base + np * cnt;
            uint4* const extra = lists + units16(nf, 4);
            fill_task<R>(g, inv_aref, c, d, nup, xpos, base, np, cnt, lane - a, reinterpret_cast<uint32_t*>(lists),
                         pf - far - bf, buf, reinterpret_cast<R*>(extra),
                         reinterpret_cast<uint32_t*>(extra + units16(ne, sizeof(R))), pe - dir_extra(nup) - be,
                         [&](uint32_t x) {
                             return x + S::kRing < G.z ? kNone : S::kRingAt + ((x - dN) & (S::kRing - 1u));
                         });
        }
        tile++;
        off += units;
    });
}

// ---------------------------------------------------------------------------
// grouped replay (full sweeps): m consecutive level sets per launch. Each
// workgroup owns a block of root tasks (kGroupT consecutive tasks of one level
// set of the group) and solves the roots' upwind cone inside the group, level
// set by level set with a workgroup barrier in between, so that every
// dependency inside the launch stays inside the workgroup (L1 coherent within
// the workgroup). Cones of different workgroups may overlap: such a task is
// solved by each of them from the same inputs with the same arithmetic and
// stores the same values. The roots of level set j are the tasks of j in no
// cone of a higher level set of the group.

// Sorts a[0, n2) ascending (n2 a power of two) in LDS, all lanes taking part.
__device__ void lds_sort(uint32_t* a, uint32_t n2) {
    for (uint32_t k = 2; k <= n2; k <<= 1)
        for (uint32_t jj = k >> 1; jj > 0; jj >>= 1) {
            for (uint32_t i = threadIdx.x; i < n2; i += blockDim.x) {
                const uint32_t ixj = i ^ jj;
                if (ixj > i) {
                    const uint32_t x = a[i], y = a[ixj];
                    if ((x > y) == ((i & k) == 0)) {
                        a[i] = y;
                        a[ixj] = x;
                    }
                }
            }
            __syncthreads();
        }
}

// Cone build: the upwind tasks of every task as schedule positions, task P's
// at up[uoff[P] ..] in face order (uoff the prefix sums of k_up_count). A wave
// per 64 cells and kFluxDirs directions reads each face once for all of them.
__global__ void k_up_count(const uint32_t* __restrict__ sorted, const uint8_t* __restrict__ nups, uint32_t n,
                           uint64_t* __restrict__ cnt) {
    const uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p <= n) cnt[p] = p < n ? nups[sorted[p]] : 0u;
}

__global__ void __launch_bounds__(1024) k_up_fill(Geo g, const uint32_t* __restrict__ xpos,
                                                  const uint64_t* __restrict__ uoff, uint32_t* __restrict__ up) {
    const uint32_t N = (uint32_t)g.N, lane = threadIdx.x % kFluxCells;
    const uint32_t w = __builtin_amdgcn_readfirstlane(threadIdx.x / kFluxCells);
    const uint32_t c = blockIdx.x * kFluxCells + lane;
    if (c >= N) return;
    uint64_t at[kFluxDirs];
#pragma unroll
    for (int j = 0; j < kFluxDirs; j++)
        at[j] = uoff[xpos[(size_t)min(w * kFluxDirs + j, (uint32_t)g.D - 1u) * N + c]];
    for (uint32_t f = g.off[c]; f < g.off[c + 1]; f++) {
        const double4 a = g.geo[f];
        const uint32_t nk = g.nk[f];
        if ((nk >> 30) != kKindLocal) continue;
#pragma unroll
        for (int j = 0; j < kFluxDirs; j++) {
            const uint32_t d = w * kFluxDirs + j;
            if (d < (uint32_t)g.D && fdot(a, g.dirs[3 * d], g.dirs[3 * d + 1], g.dirs[3 * d + 2]) < 0.0)
                up[at[j]++] = xpos[(size_t)d * N + (nk & kNbrMask)];
        }
    }
}

// Calls use(x) for the upwind positions x of the task at position P, eight
// loads in flight.
template <typename F>
__device__ __forceinline__ void each_upwind(const uint64_t* __restrict__ uoff, const uint32_t* __restrict__ up,
                                            uint32_t P, F use) {
    const uint64_t e0 = uoff[P], e1 = uoff[P + 1];
    for (uint64_t e = e0; e < e1; e += 8u) {
        uint32_t v[8];
#pragma unroll
        for (int j = 0; j < 8; j++) v[j] = up[min(e + j, e1 - 1u)];
#pragma unroll
        for (int j = 0; j < 8; j++)
            if (e + j < e1) use(v[j]);
    }
}

// Appends the upwind schedule positions in [lo, hi) of the task at position P
// to cand.
__device__ void push_upwind(const uint64_t* uoff, const uint32_t* up, uint32_t P, uint32_t lo, uint32_t hi,
                            uint32_t* cand, uint32_t* ncand, uint32_t* over) {
    each_upwind(uoff, up, P, [&](uint32_t v) {
        if (v < lo || v >= hi) return;
        const uint32_t k = atomicAdd(ncand, 1u);
        if (k < (uint32_t)kConeCap) cand[k] = v;
        else *over = 1u;
    });
}

// Workgroup descriptor of the grouped replay, two uint4: {list offset, level
// sets, counts of level sets 0|1, 2|3} and {counts 4|5, 6|7, 0, 0} (16 bits
// per count, level sets counted from the group's first).
__device__ __forceinline__ uint32_t desc_count(const uint4& d0, const uint4& d1, int ph) {
    const uint32_t w = ph < 2 ? d0.z : ph < 4 ? d0.w : ph < 6 ? d1.x : d1.y;
    return (ph & 1) ? (w >> 16) : (w & 0xFFFFu);
}

// One workgroup per block of at most 128 roots of one level set j of a group
// starting at level set k0, meta[block] = {k0, j, first root, roots}: its cone
// per level set (sorted, unique), written with the roots to the task list,
// level set k0 first, and its descriptor. Members and roots are marked done
// in todo. Roots are roots[first + r] or, without a root list, positions
// first + r. Pending upwind entries are kept per level set: those of level
// set i are taken out when i is processed.
__global__ void __launch_bounds__(kConeThreads) k_cone(const uint64_t* uoff, const uint32_t* up,
                                            const uint32_t* fstart, const uint4* meta, const uint32_t* roots,
                                            uint8_t* todo, uint32_t* list, uint32_t list_cap, uint32_t* cursor,
                                            uint4* desc, uint32_t* fail) {
    __shared__ uint32_t candA[kConeCap], candB[kConeCap], tmp[kSortCap], memb[kConeCap];
    __shared__ uint32_t ncand, nkeep, ntmp, nmemb, over, base;
    __shared__ uint32_t cnt[kMaxGroup], psum[kConeThreads / 64];
    uint32_t* cand = candA;
    uint32_t* keep = candB;
    const uint32_t tid = threadIdx.x;
    const uint4 mb = meta[blockIdx.x];
    const int k0 = (int)mb.x, j = (int)mb.y;
    const uint32_t n = mb.w;  // at most kConeThreads
    constexpr uint32_t T = kConeThreads;
    if (tid == 0) {
        ncand = 0;
        nmemb = 0;
        over = 0;
    }
    if (tid < (uint32_t)kMaxGroup) cnt[tid] = 0;
    __syncthreads();
    const uint32_t lo = fstart[k0];
    uint32_t root = 0;
    if (tid < n) {
        root = roots ? roots[mb.z + tid] : mb.z + tid;
        push_upwind(uoff, up, root, lo, fstart[j], cand, &ncand, &over);
    }
    __syncthreads();
    for (int i = j - 1; i >= k0; i--) {
        const uint32_t bi = fstart[i];
        if (tid == 0) {
            ntmp = 0;
            nkeep = 0;
        }
        __syncthreads();
        // pending entries of level set i to tmp, of lower level sets to keep
        const uint32_t nc = min(ncand, (uint32_t)kConeCap);
        for (uint32_t c = tid; c < nc; c += T) {
            const uint32_t v = cand[c];
            if (v >= bi) tmp[atomicAdd(&ntmp, 1u)] = v;  // entries are below the level sets done
            else keep[atomicAdd(&nkeep, 1u)] = v;
        }
        __syncthreads();
        {
            uint32_t* x = cand;
            cand = keep;
            keep = x;
        }
        if (tid == 0) ncand = nkeep;
        const uint32_t nt = ntmp;
        uint32_t n2 = 1;
        while (n2 < nt) n2 <<= 1;
        for (uint32_t c = nt + tid; c < n2; c += T) tmp[c] = kNone;
        __syncthreads();
        lds_sort(tmp, n2);
        // unique, in order: each lane compacts a contiguous chunk
        const uint32_t per = (nt + T - 1) / T;
        const uint32_t c0 = min(nt, tid * per), c1 = min(nt, c0 + per);
        uint32_t u = 0;
        for (uint32_t c = c0; c < c1; c++) u += (c == 0 || tmp[c] != tmp[c - 1]) ? 1u : 0u;
        const uint32_t incl = wave_scan(u);
        if (tid % 64u == 63u) psum[tid / 64u] = incl;
        __syncthreads();
        uint32_t before = incl - u, all = 0;
        for (uint32_t l = 0; l < T / 64u; l++) {
            if (l < tid / 64u) before += psum[l];
            all += psum[l];
        }
        if (tid == 0) {
            cnt[i - k0] = all;
            if (nmemb + all > (uint32_t)kConeCap) over = 1u;
        }
        __syncthreads();
        if (over) break;
        const uint32_t m0 = nmemb;
        uint32_t w = m0 + before;
        for (uint32_t c = c0; c < c1; c++)
            if (c == 0 || tmp[c] != tmp[c - 1]) memb[w++] = tmp[c];
        __syncthreads();
        if (tid == 0) nmemb = m0 + cnt[i - k0];
        __syncthreads();
        const uint32_t m1 = nmemb;
        if (i > k0)
            for (uint32_t c = m0 + tid; c < m1; c += T)
                push_upwind(uoff, up, memb[c], lo, bi, cand, &ncand, &over);
        __syncthreads();
    }
    if (over) {
        if (tid == 0) atomicOr(fail, 1u);
        return;
    }
    const uint32_t total = nmemb + n;
    if (tid == 0) {
        base = atomicAdd(cursor, total);
        if (base + total > list_cap) {
            atomicOr(fail, 2u);
            base = kNone;
        }
    }
    __syncthreads();
    if (base == kNone) return;
    // members were appended from level set j-1 down to k0; the list holds them
    // from k0 up, then the roots
    uint32_t src = nmemb, dst = 0;
    for (int i = k0; i < j; i++) {
        const uint32_t ci = cnt[i - k0];
        src -= ci;
        for (uint32_t c = tid; c < ci; c += T) {
            const uint32_t v = memb[src + c];
            list[base + dst + c] = v;
            todo[v] = 0;
        }
        dst += ci;
    }
    if (tid < n) {
        list[base + dst + tid] = root;
        todo[root] = 0;
    }
    if (tid == 0) {
        uint32_t c[kMaxGroup];
        for (int k = 0; k < kMaxGroup; k++) c[k] = 0;
        for (int i = k0; i < j; i++) c[i - k0] = cnt[i - k0];
        c[j - k0] = n;
        desc[2 * blockIdx.x] = make_uint4(base, (uint32_t)(j - k0 + 1), c[0] | (c[1] << 16), c[2] | (c[3] << 16));
        desc[2 * blockIdx.x + 1] = make_uint4(c[4] | (c[5] << 16), c[6] | (c[7] << 16), 0u, 0u);
    }
}

// Cone build: flags[p] = todo[p] for the positions of the level sets marked
// in lvlflag (binary search of p's level set in fstart), else 0.
__global__ void k_cone_flags(const uint32_t* fstart, int kmax, const uint8_t* lvlflag, const uint8_t* todo,
                             uint8_t* flags, uint32_t n) {
    const uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n) return;
    int a = 0, b = kmax - 1;
    while (a < b) {
        const int m = (a + b + 1) >> 1;
        if (fstart[m] <= p) a = m;
        else b = m - 1;
    }
    flags[p] = lvlflag[a] ? todo[p] : (uint8_t)0;
}

// Cone build: for level set lv[i], the range [lo, hi) of the sorted root list
// (nsel entries) holding its positions.
__global__ void k_cone_bounds(const uint32_t* roots, const uint32_t* nsel, const uint32_t* fstart, const int* lv,
                              int nlv, uint32_t* out) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nlv) return;
    const uint32_t n = *nsel;
    for (int e = 0; e < 2; e++) {
        const uint32_t key = fstart[lv[i] + e];
        uint32_t a = 0, z = n;
        while (a < z) {
            const uint32_t m = (a + z) >> 1;
            if (roots[m] < key) a = m + 1;
            else z = m;
        }
        out[2 * i + e] = a;
    }
}

// Descriptors into group order: out[i] = in[perm[i]] (two uint4 each).
__global__ void k_permute_desc(const uint4* in, const uint32_t* perm, uint4* out, uint32_t n) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    out[2 * i] = in[2 * perm[i]];
    out[2 * i + 1] = in[2 * perm[i] + 1];
}

// Grouped replay of a group of level sets: one workgroup per cone, compiled
// into tiles like a direction's (k_sweep_dir): up to 64 tasks of one level
// set, planes whose entries name LDS words, a far list. Here the LDS holds one
// word per task of the cone, so that X passes between the group's level sets
// through LDS, and everything older than the group is in memory when the
// launch starts: it is on the far list, whose loads go out with the tile's
// cell inputs. A wave takes a tile (tile i the wave i mod waves, which fixes
// the words of its buffer), loads all it needs, and waits for its level set
// only then: every wave passes level sets - 1 barriers, whatever tiles it has.
// Bound by the chain of a launch: descriptor, planes and far list, far values,
// then per level set a barrier, the LDS reads, the sum and a division. With
// planes in schedule order and upwind values gathered from memory, every level
// set ended with a store, a wait for it and a gather: a launch of 8 level sets
// took 14.6 us in the captured sweep of 32768 cells x 16 directions FP64 (6.1 us
// like this), one of 4 level sets 9.4 us on 117649 cells x 64 directions FP32
// (5.1 us).
//   tile  {blob offset (48 bits), LDS word of its first task (16 bits), tasks |
//         planes << 7 | extra << 11 | far << 19, level set in the cone | level
//         sets << 8 | tiles of the cone << 16}
//   blob  planes, {X index, I index} of the tasks, far list, extra weights,
//         extra words
// The first `waves` tiles of a group's b-th cone are at tiles[slot0 + b * waves]
// (those it does not have without tasks), the others from tiles[more[cone0 +
// b]] on: no load has to return before a wave's first descriptor is on its way.
// A group of more than 4 level sets has up to twice the tiles of one of 4;
// where each CU has one of its cones at most, its workgroups are of twice the
// waves (up to 16), so that no tile waits for another's end to load
// (32768 cells x 16 directions FP64, groups of 8: 9.1 -> 7.8 us a launch).
// A restricted sweep runs the cones with active tasks; a task whose cell is
// below level lvl is not solved and puts its stored X into its word.
template <typename R>
struct ConeShape {
    static constexpr uint32_t kAt = 64;                                         // words 0-63: 0
    static constexpr uint32_t kFar = 512;                                       // far entries of a tile
    static constexpr uint32_t kBuf = kFar + 128 + 512 / (uint32_t)sizeof(R);    // far, extra weights, extra words
    static constexpr int waves(int roots) { return roots == 32 ? 4 : roots == 64 ? 8 : 16; }
    static size_t bytes(int waves, uint32_t cone) { return sizeof(R) * (kAt + cone + (size_t)waves * kBuf); }
};

template <typename R, int kWaves, bool kGeneral>
__device__ __forceinline__ void cone_body(const Geo& g, const Flux<R>& fl, const uint4* __restrict__ blob,
                                          const uint4* __restrict__ tiles, const uint32_t* __restrict__ more,
                                          uint32_t b, uint32_t slot0, uint32_t cone0, uint32_t words, int lvl) {
    using S = DirShape<R>;
    using K = ConeShape<R>;
    extern __shared__ double cone_lds[];
    R* const lds = reinterpret_cast<R*>(cone_lds);
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    R* const buf = lds + K::kAt + words + w * K::kBuf;
    uint32_t* const bufs = reinterpret_cast<uint32_t*>(buf + K::kFar + 128);
    uint4 t = tiles[(size_t)slot0 + (size_t)b * kWaves + w];
    lds[lane] = (R)0;  // by every wave, before its own reads
    auto uni = [](uint32_t v) -> uint32_t { return __builtin_amdgcn_readfirstlane(v); };
    auto rsrc = [&](const uint4* p, uint32_t bytes) {
        return __builtin_amdgcn_make_buffer_rsrc(const_cast<uint4*>(p), 0, (int)bytes, 0x00027000);
    };
    uint32_t at_level = 0;
    auto pass_to = [&](uint32_t k) {  // every wave passes level sets - 1 barriers
        while (at_level < k) {
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
            at_level++;
        }
    };
    const uint32_t levels = (uni(t.w) >> 8) & 255u, n = uni(t.w) >> 16;
    for (uint32_t i = w; i < n; i += kWaves) {
        if (i >= kWaves) t = tiles[(size_t)more[cone0 + b] + i - kWaves];
        const uint64_t off = (uint64_t)uni(t.x) | ((uint64_t)(uni(t.y) & 0xFFFFu) << 32);
        const uint32_t word0 = uni(t.y) >> 16, k = uni(t.w) & 255u, pk = uni(t.z);
        const uint32_t cnt = pk & 127u, np = (pk >> 7) & 15u, nex = (pk >> 11) & 255u, nfar = pk >> 19;
        const uint32_t li = min(lane, cnt - 1u), st = cnt * 16u;
        const uint4* p = blob + off;
        const auto rp = rsrc(p, np * st);
        const u32x4 s0 = __builtin_amdgcn_raw_buffer_load_b128(rp, li * 16u, 0, 0);
        p += np * cnt;
        const uint2 at = reinterpret_cast<const uint2*>(p)[li];
        const uint32_t xi = at.x, oi = at.y;
        p += units16(cnt, 8);
        uint32_t far[K::kFar / 64];
        const auto rf = rsrc(p, nfar * 4u);
#pragma unroll
        for (int j = 0; j < (int)(K::kFar / 64); j++) {
            far[j] = 0;
            if (nfar > 64u * j) far[j] = __builtin_amdgcn_raw_buffer_load_b32(rf, (lane + 64u * j) * 4u, 0, 0);
        }
        const u32x4 s1 = __builtin_amdgcn_raw_buffer_load_b128(rp, li * 16u + S::kS1 * st, 0, 0);
        uint32_t wt[4 * S::kWPlanes];
#pragma unroll
        for (int j = 0; j < S::kWPlanes; j++) {
            const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(rp, li * 16u + S::wplane(j) * st, 0, 0);
#pragma unroll
            for (int m = 0; m < 4; m++) wt[4 * j + m] = v[m];
        }
        p += units16(nfar, 4);
        const uint32_t hdr = s0.x, c = hdr & kCellMask, nup = hdr >> kCellBits;
        const SA<R> sa = fl.sa[c];
        R off_i = 0, xold = 0;
        uint32_t lev = 0;
        if (kGeneral) {
            if (fl.offI) off_i = fl.offI[oi];
            if (lvl > 0) {
                lev = g.level[c];
                xold = fl.X[xi];
            }
        }
        R fv[K::kFar / 64];
#pragma unroll
        for (int j = 0; j < (int)(K::kFar / 64); j++) {
            fv[j] = (R)0;
            if (nfar > 64u * j) {
                const R* src = (far[j] & kFarPeriodic) ? fl.P : fl.X;
                fv[j] = src[far[j] & ~kFarPeriodic];
            }
        }
        for (uint32_t e = lane; e < nex; e += 64u) {
            buf[K::kFar + e] = reinterpret_cast<const R*>(p)[e];
            bufs[e] = reinterpret_cast<const uint32_t*>(p + units16(nex, sizeof(R)))[e];
        }
#pragma unroll
        for (int j = 0; j < (int)(K::kFar / 64); j++)
            if (nfar > 64u * j) buf[64u * j + lane] = fv[j];
        const bool more = nup > kDirEntries;
        auto half = [&](int h) -> uint32_t {
            const uint32_t v = h < 8 ? s0[(h % 8) / 2] : s1[(h % 8) / 2];
            return (h & 1) ? v >> 16 : v & 0xFFFFu;
        };
        auto weight = [&](int m) -> R {
            if constexpr (sizeof(R) == 4) return __uint_as_float(wt[m]);
            else return __hiloint2double((int)wt[2 * m + 1], (int)wt[2 * m]);
        };
        pass_to(k);
        R x[kDirEntries + 1];
#pragma unroll
        for (int e = 0; e <= (int)kDirEntries; e++) x[e] = lds[(e == (int)kDirEntries && more) ? 0u : half(e + 2)];
        R inc = 0;
#pragma unroll
        for (int e = 0; e < (int)kDirEntries; e++) inc += weight(1 + e) * x[1 + e];
        if (nex && more) {
            const uint32_t first = half((int)kDirEntries + 2) - (kDirEntries - 1u);
            for (uint32_t e0 = kDirEntries - 1u; e0 < nup; e0 += 4u) {
                R v[4], y[4];
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const uint32_t e = first + min(e0 + j, nup - 1u);
                    v[j] = buf[K::kFar + e];
                    y[j] = lds[bufs[e]];
                }
#pragma unroll
                for (int j = 0; j < 4; j++) inc += e0 + j < nup ? v[j] * y[j] : (R)0;
            }
        }
        const CellIn<R> ci{sa.x, sa.y, x[0], off_i};
        const R A = weight(0);
        bool act = lane < cnt && (!kGeneral || lev >= (uint32_t)lvl);
        R xv = xold;
        if (act) {
            const R out = outgoing_rate<R, kGeneral>(fl, oi, inc, ci);
            xv = (A > (R)0) ? out / A : (R)0;
        }
        if (lane < cnt) lds[word0 + lane] = xv;
        // a wave's last tile: its level set's end before its stores
        if (i + kWaves >= n) pass_to(min(k + 1u, levels - 1u));
        if (act) {
            fl.X[xi] = xv;
            fl.I[oi] = inc;
        }
    }
    pass_to(levels - 1u);
}

template <typename R, int kWaves, bool kGeneral>
__global__ void __launch_bounds__(64 * kWaves) k_sweep_cone(Geo g, Flux<R> fl, const uint4* __restrict__ blob,
                                                            const uint4* __restrict__ tiles,
                                                            const uint32_t* __restrict__ more,
                                                            const uint32_t* __restrict__ sel, uint32_t slot0,
                                                            uint32_t cone0, uint32_t words, int lvl,
                                                            PassTab pt) {
    const uint32_t b = pass_item(pt, blockIdx.x);
    cone_body<R, kWaves, kGeneral>(g, fl, blob, tiles, more, sel ? sel[b] : b, slot0, cone0, words, lvl);
}

// One problem's grouped launch inside a packed launch: everything the grouped
// kernel reads of its handle, and its workgroups [start, start + blocks) of
// the packed grid (start a multiple of kXcds, so that the die-aware order of
// its cones holds as in a launch of its own).
template <typename R>
struct GroupJob {
    int64_t N;
    R* X;
    R* I;
    R* P;
    R* offI;
    const SA<R>* sa;
    R thr;
    const uint8_t* level;
    const uint4* blob;
    const uint4* tiles;
    const uint32_t* more;
    const uint32_t* sel;
    uint32_t slot0, cone0, words;
    int lvl;
    uint32_t start, blocks;
    PassTab pt;
};

constexpr int kMaxPack = 8;  // problems per packed launch (kernel arguments of ~1.5 KB)

template <typename R>
struct PackArgs {
    GroupJob<R> job[kMaxPack];
    int n;
};

// Grouped launches of up to kMaxPack problems in one launch: workgroup b runs
// the job whose range holds it, as k_sweep_cone would run it alone.
template <typename R, int kWaves, bool kGeneral>
__global__ void __launch_bounds__(64 * kWaves) k_sweep_cone_pack(const PackArgs<R> a) {
    int j = 0;
    for (int k = 1; k < a.n; k++)
        if (blockIdx.x >= a.job[k].start) j = k;
    const GroupJob<R>& J = a.job[j];
    const uint32_t i = blockIdx.x - J.start;
    if (i >= J.blocks) return;  // padding up to the next job's die-aligned start
    Geo g{};
    g.N = J.N;
    g.level = J.level;
    Flux<R> fl{};
    fl.X = J.X;
    fl.I = J.I;
    fl.P = J.P;
    fl.offI = J.offI;
    fl.sa = J.sa;
    fl.thr = J.thr;
    const uint32_t b = pass_item(J.pt, i);
    cone_body<R, kWaves, kGeneral>(g, fl, J.blob, J.tiles, J.more, J.sel ? J.sel[b] : b, J.slot0, J.cone0, J.words, J.lvl);
}

// Tiles of every cone: counted (kFill = false, one wave each: the tiles past
// the first `waves` and blob units of each cone, the far entries of each task
// of the list, and the largest cone of each group into words) or written (four
// waves each, a tile the wave). ginfo[gmap[cone]]: the cone's group.
template <typename R, bool kFill>
__global__ void __launch_bounds__(kFill ? 256 : 64) k_cone_tiles(
    Geo g, double inv_aref, const uint32_t* __restrict__ sorted, const uint32_t* __restrict__ xpos,
    const uint64_t* __restrict__ uoff, const uint32_t* __restrict__ up, const uint32_t* __restrict__ fstart,
    const uint8_t* __restrict__ nups, uint8_t* __restrict__ fars, const uint4* __restrict__ desc,
    const uint32_t* __restrict__ list, const uint32_t* __restrict__ gmap, const uint4* __restrict__ ginfo,
    uint32_t* __restrict__ ct, uint64_t* __restrict__ cu, uint32_t* __restrict__ words,
    const uint32_t* __restrict__ ts, const uint64_t* __restrict__ us, uint32_t slots, uint4* __restrict__ blob,
    uint4* __restrict__ tiles, uint32_t* __restrict__ more) {
    using K = ConeShape<R>;
    extern __shared__ uint32_t memb[];  // kFill: the cone's tasks
    __shared__ uint32_t fs[kMaxGroup + 1], zs[kMaxGroup + 1];
    const uint32_t w = blockIdx.x, lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    const uint4 d0 = desc[2 * (size_t)w], d1 = desc[2 * (size_t)w + 1];
    const uint4 G = ginfo[gmap[w]];
    const uint32_t k0 = G.x, waves = G.y, slot = G.z + (w - G.w) * waves, levels = d0.y, N = (uint32_t)g.N;
    uint32_t total = 0;
    for (uint32_t ph = 0; ph < levels; ph++) total += desc_count(d0, d1, (int)ph);
    if (kFill) {
        if (threadIdx.x == 0)
            for (uint32_t ph = 0, z = 0; ph <= levels; ph++) {
                fs[ph] = fstart[k0 + ph];
                zs[ph] = z;
                z += ph < levels ? desc_count(d0, d1, (int)ph) : 0u;
            }
        for (uint32_t i = threadIdx.x; i < total; i += blockDim.x) memb[i] = list[d0.x + i];
        __syncthreads();
    }
    const uint32_t lo = fstart[k0], cone = d0.x;
    uint32_t seg = 0, nt = 0, all = 0;
    uint64_t off = kFill ? us[w] : 0;
    const uint32_t more0 = kFill ? slots + ts[w] : 0u;
    if (kFill) all = waves + ts[w + 1] - ts[w];  // the tiles, if more than `waves`
    for (uint32_t ph = 0; ph < levels; ph++) {
        const uint32_t m = desc_count(d0, d1, (int)ph);
        for (uint32_t b = 0; b < m; b += 64u) {
            const uint32_t n = min(64u, m - b), at = cone + seg + b + min(lane, n - 1u), P = list[at];
            const uint32_t t = sorted[P], nup = nups[t];
            uint32_t far = 0;
            if (lane < n) {
                if (kFill) {
                    far = fars[at];
                } else {
                    far = (g.Nper && g.pslot[t % N] != kNone) ? 1u : 0u;
                    each_upwind(uoff, up, P, [&](uint32_t x) { far += x < lo ? 1u : 0u; });
                    fars[at] = (uint8_t)far;
                }
            }
            const uint32_t ex = lane < n ? dir_extra(nup) : 0u, pf = wave_scan(far), pe = wave_scan(ex);
            for (uint32_t a = 0; a < n;) {
                const uint32_t bf = a ? (uint32_t)__shfl((int)pf, a - 1) : 0u;
                const uint32_t be = a ? (uint32_t)__shfl((int)pe, a - 1) : 0u;
                const unsigned long long over =
                    __ballot(lane > a && lane < n && (pf - bf > K::kFar || pe - be > kDirCap));
                const uint32_t e = over ? (uint32_t)__ffsll((long long)over) - 1u : n, cnt = e - a;
                const uint32_t nf = (uint32_t)__shfl((int)pf, e - 1) - bf, ne = (uint32_t)__shfl((int)pe, e - 1) - be;
                const uint32_t np = DirShape<R>::planes(wave_max(lane >= a && lane < e ? nup : 0u));
                if (kFill && nt % (blockDim.x / 64u) == wave) {
                    uint4* const base = blob + off;
                    uint2* const at2 = reinterpret_cast<uint2*>(base + np * cnt);
                    uint4* const lists = base + np * cnt + units16(cnt, 8);
                    uint4* const extra = lists + units16(nf, 4);
                    if (lane == 0)
                        tiles[nt < waves ? slot + nt : (size_t)more0 + nt - waves] = make_uint4(
                            (uint32_t)off, (uint32_t)(off >> 32) | ((K::kAt + seg + b + a) << 16),
                            cnt | (np << 7) | (ne << 11) | (nf << 19), ph | (levels << 8) | (all << 16));
                    if (lane >= a && lane < e) {
                        at2[lane - a] = make_uint2(P, t);
                        fill_task<R>(g, inv_aref, t % N, t / N, nup, xpos, base, np, cnt, lane - a,
                                     reinterpret_cast<uint32_t*>(lists), pf - far - bf,
                                     K::kAt + words[gmap[w]] + (nt % waves) * K::kBuf, reinterpret_cast<R*>(extra),
                                     reinterpret_cast<uint32_t*>(extra + units16(ne, sizeof(R))), pe - ex - be,
                                     [&](uint32_t x) {
                                         if (x < lo) return kNone;
                                         uint32_t q = 0;  // its level set, then its place there
                                         while (fs[q + 1] <= x) q++;
                                         uint32_t z0 = zs[q], z1 = zs[q + 1];
                                         while (z1 - z0 > 1) {
                                             const uint32_t z = (z0 + z1) / 2;
                                             if (memb[z] <= x) z0 = z;
                                             else z1 = z;
                                         }
                                         return K::kAt + z0;
                                     });
                    }
                }
                off += np * cnt + units16(cnt, 8) + units16(nf, 4) + units16(ne, sizeof(R)) + units16(ne, 4);
                nt++;
                a = e;
            }
        }
        seg += m;
    }
    if (!kFill) {
        if (lane == 0) {
            ct[w] = nt > waves ? nt - waves : 0u;
            cu[w] = off;
            atomicMax(&words[gmap[w]], total);
        }
        return;
    }
    // the number of tiles, now known, in the descriptors of a cone that has no
    // more than `waves`; the places it does not use
    if (all > waves) {
        if (threadIdx.x == 0) more[w] = more0;
        return;
    }
    __syncthreads();
    if (threadIdx.x < waves) {
        uint4* const t = tiles + slot + threadIdx.x;
        if (threadIdx.x < nt) t->w = (t->w & 0xFFFFu) | (nt << 16);
        else *t = make_uint4(0u, 0u, 0u, (levels << 8) | (nt << 16));
    }
}

// The grouped replay of a restricted sweep (active set {level >= lvl}): a wave
// per cone counts its active tasks; cones that have some are kept (k_place_cone
// then packs each group's in order), and the active tasks and kept cones of
// each group are summed into gcount and gblocks (gmap: group of each cone).
__global__ void __launch_bounds__(64) k_cone_active(Geo g, int lvl, const uint4* __restrict__ blob,
                                                    const uint4* __restrict__ tiles,
                                                    const uint32_t* __restrict__ more,
                                                    const uint4* __restrict__ ginfo,
                                                    const uint32_t* __restrict__ gmap, uint32_t* kept,
                                                    uint32_t* gcount, uint32_t* gblocks) {
    const uint4 G = ginfo[gmap[blockIdx.x]];
    const uint32_t waves = G.y, slot = G.z + (blockIdx.x - G.w) * waves, tn = tiles[slot].w >> 16;
    uint32_t n = 0;
    for (uint32_t i = 0; i < tn; i++) {
        const uint4 t = tiles[i < waves ? slot + i : (size_t)more[blockIdx.x] + i - waves];
        const uint32_t cnt = t.z & 127u;
        const uint32_t hdr = blob[((uint64_t)t.x | ((uint64_t)(t.y & 0xFFFFu) << 32)) + min(threadIdx.x, cnt - 1u)].x;
        n += (uint32_t)__popcll(__ballot(threadIdx.x < cnt && g.level[hdr & kCellMask] >= lvl));
    }
    if (threadIdx.x == 0) {
        kept[blockIdx.x] = n ? 1u : 0u;
        if (n) {
            atomicAdd(&gcount[gmap[blockIdx.x]], n);
            atomicAdd(&gblocks[gmap[blockIdx.x]], 1u);
        }
    }
}

// Packs the kept cones: cone w of group g (whose cones start at gbase[g]) goes
// to place pos[w] - pos[gbase[g]] of the group (pos the exclusive prefix sum
// of kept), so each group's kept cones keep their order (and with it the pass
// ranges of the die-aware launch order). sel holds cones counted from the
// group's first.
__global__ void k_place_cone(const uint32_t* __restrict__ kept, const uint32_t* __restrict__ pos,
                             const uint32_t* __restrict__ gmap, const uint32_t* __restrict__ gbase, uint32_t* sel,
                             uint32_t n) {
    const uint32_t w = blockIdx.x * blockDim.x + threadIdx.x;
    if (w >= n || !kept[w]) return;
    const uint32_t b = gbase[gmap[w]];
    sel[b + (pos[w] - pos[b])] = w - b;
}

__global__ void k_gather_u32(const uint32_t* __restrict__ src, const uint32_t* __restrict__ idx, uint32_t* out,
                             uint32_t n) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = src[idx[i]];
}

// ---------------------------------------------------------------------------
// per-sweep kernels

struct ChemArgs {
    double* rho;
    double* x;
    double* T;
    double* src;             // source per direction bin (SI)
    void* sa;                // SA<R>[N], .y: attenuation of the next sweep
    double* species_ts;
    double* prev_rate;
    double* change_ts;
    double* photon;          // sum of the incoming rates (SI); -1: not solved by the last sweep
    const double* vol;
    const double* size;
    double max_ts;
    double thr;
    double safety;
    double scale_factor;
    int prevent_cooling;
    double lref;             // storage scale of I (rate = I * lref)
    unsigned long long* failures;
    unsigned long long* active;
    unsigned long long* limiting;  // [3] TimescaleCounter: temperature, ionisation fraction, photon rate
    uint32_t* queue;         // {cells queued, cells taken beyond the first ones}, then the queued cells
};

// The arguments of the kernels after a sweep, for one handle, or for the
// handles of a packed step (one per blockIdx.y).
template <typename R>
struct ChemJob {
    Geo g;
    Flux<R> fl;
    ChemArgs ca;
    int lvl;
};
constexpr int kChemJobs = 4;
template <typename R, int kJobs>
struct ChemJobs {
    ChemJob<R> job[kJobs];
    __device__ __forceinline__ const ChemJob<R>& mine() const { return job[kJobs > 1 ? blockIdx.y : 0]; }
};

// Periodic source of every periodic cell from the current X, after each
// sweep: the chemistry of the sweep reads it (the reference's periodic
// corrections have all arrived when update_chemistry runs), and the next
// sweep's transport reads it as the value at its start (X does not change in
// between). A wave takes 64 periodic cells and kPerDirs directions, two faces
// at a time, from a list of the periodic faces alone: all its gathers of X
// (two dependent loads each, the bound) are in flight together, and P is
// stored in runs. With a thread per cell and direction, lanes across
// directions, and the faces read through the grid's list: 153 us on 262144
// cells x 84 directions, 88 on 157464 x 64, 32 on 20000 x 84 FP64; like this
// 108, 47 and 29. The first
// thread empties the queue of the chemistry that follows.
constexpr int kPerDirs = 2;
template <typename R, int kJobs>
__global__ void __launch_bounds__(kBlock) k_periodic(const ChemJobs<R, kJobs> jobs) {
    const ChemJob<R>& J = jobs.mine();
    const Geo& g = J.g;
    const Flux<R>& fl = J.fl;
    if (blockIdx.x == 0 && threadIdx.x == 0) J.ca.queue[0] = J.ca.queue[1] = 0u;
    if (fl.P == nullptr) return;
    const uint32_t dblocks = ((uint32_t)g.D + kPerDirs - 1u) / kPerDirs;
    const uint32_t w = __builtin_amdgcn_readfirstlane((blockIdx.x * kBlock + threadIdx.x) / 64u);
    const uint32_t s = (w / dblocks) * 64u + (threadIdx.x & 63u), d0 = (w % dblocks) * kPerDirs;
    if ((int64_t)s >= g.Nper) return;
    R acc[kPerDirs];
#pragma unroll
    for (int j = 0; j < kPerDirs; j++)
        acc[j] = fl.offP ? fl.offP[(size_t)min(d0 + j, (uint32_t)g.D - 1u) * g.Nper + s] : (R)0;
    const uint32_t e1 = g.pfoff[s + 1];
    for (uint32_t e = g.pfoff[s]; e < e1; e += 2) {
        R wt[2][kPerDirs], x[2][kPerDirs];
        bool up[2][kPerDirs];
#pragma unroll
        for (int u = 0; u < 2; u++) {
            const uint32_t f = min(e + u, e1 - 1u);
            const double4 a = g.pgeo[f];
            const uint32_t nb = g.pnb[f];
#pragma unroll
            for (int j = 0; j < kPerDirs; j++) {
                const uint32_t d = min(d0 + j, (uint32_t)g.D - 1u);  // past the last direction: not stored
                const double dd = fdot(a, g.dirs[3 * d], g.dirs[3 * d + 1], g.dirs[3 * d + 2]);
                up[u][j] = dd < 0.0 && e + u < e1;
                wt[u][j] = (R)(a.w * fl.inv_aref * -dd);
                x[u][j] = up[u][j] ? fl.X[xidx(fl, g.N, d, nb)] : (R)0;
            }
        }
#pragma unroll
        for (int u = 0; u < 2; u++)
#pragma unroll
            for (int j = 0; j < kPerDirs; j++)
                if (up[u][j]) acc[j] += wt[u][j] * x[u][j];
    }
#pragma unroll
    for (int j = 0; j < kPerDirs; j++)
        if (d0 + j < (uint32_t)g.D) fl.P[(size_t)(d0 + j) * g.Nper + s] = acc[j];
}

// Adds the number of lanes with `pred` to *counter with one atomic per wave
// (lanes outside the current control flow take no part).
__device__ __forceinline__ void wave_count(bool pred, unsigned long long* counter) {
    const unsigned long long m = __ballot(pred);
    if (m && __lane_id() == __ffsll((long long)__ballot(1)) - 1) atomicAdd(counter, (unsigned long long)__popcll(m));
}

// The cell of c for the solver, at summed rate `rate`.
__device__ __forceinline__ ssw::Cell solver_cell(const ChemArgs& ca, int64_t c, double rate) {
    ssw::Cell cell;
    cell.x = ca.x[c];
    cell.T = ca.T[c];
    cell.rho = ca.rho[c];
    cell.vol = ca.vol[c];
    cell.len = ca.size[c];
    cell.rate = rate;
    cell.a = ca.scale_factor;
    return cell;
}

// The end of a cell's update: state, timescales, process counts (lanes with
// `own` only) and the attenuation for the next sweep.
template <typename R>
__device__ __forceinline__ void finish_chemistry(const ChemArgs& ca, int64_t c, const ssw::Cell& cell, double rate_ts,
                                                 const ssw::Walk& w, bool own) {
    // Timescale::min (src/chemistry/timescale.rs:32-38): a tie goes to the chemistry
    const bool rate_limits = rate_ts < w.ts;
    const double change = rate_limits ? rate_ts : w.ts;
    // TimescaleCounter::count (src/chemistry/timescale.rs:80-87)
    const int process = rate_limits ? 2 : w.proc;
    const bool counted = own && change < ca.max_ts;
    wave_count(counted && process == 0, &ca.limiting[0]);
    wave_count(counted && process == 1, &ca.limiting[1]);
    wave_count(counted && process == 2, &ca.limiting[2]);
    wave_count(own && w.failed, ca.failures);
    const R att = (R)ssw::non_absorbed_fraction(cell.rho, cell.x, cell.len);
    if (!own) return;
    ca.x[c] = cell.x;
    ca.T[c] = cell.T;
    ca.species_ts[c] = w.ts;
    ca.change_ts[c] = change;
    ((SA<R>*)ca.sa)[c].y = att;
}

// update_chemistry (src/sweep/mod.rs:549-574) for the active cells, then the
// attenuation of the updated cell for the next sweep. One lane per cell for
// the rate and the first attempt of the solver; cells whose full step is
// rejected go to the queue of k_chemistry_tail, else a wave would last as long
// as its slowest cell's sub-steps, one after the other.
// The rates of kChemDirs directions are loaded together, the last ones clamped
// to the last direction: with the loop unrolled six times, and its remainder
// one dependent gather after the other, a frame of 2 M clustered cells x 84
// directions took 89.4 ms, with 8, 12 and 16 at once 87.0, 87.4 and 87.5.
constexpr int kChemDirs = 8;
template <typename R, int kJobs>
__global__ void __launch_bounds__(kBlock) k_chemistry(const ChemJobs<R, kJobs> jobs) {
    const ChemJob<R>& J = jobs.mine();
    const Geo& g = J.g;
    const Flux<R>& fl = J.fl;
    const ChemArgs& ca = J.ca;
    const int lvl = J.lvl;
    const uint32_t nb = (uint32_t)((g.N + kBlock - 1) / kBlock);
    if (blockIdx.x >= nb) return;  // another handle's cells are more
    // a die takes consecutive cells: where I is gathered (direction sweeps),
    // they share its lines in the die's L2
    int64_t c = (int64_t)xcd_block(blockIdx.x, nb) * kBlock + threadIdx.x;
    if (c == 0) g.need[lvl] = 0;  // the active-set list of this sweep level is current
    if (c >= g.N) return;
    int lev = g.level[c];
    {
        unsigned long long m = __ballot(lev >= lvl);
        if (__lane_id() == __ffsll((long long)__ballot(1)) - 1 && m)
            atomicAdd(ca.active, (unsigned long long)__popcll(m));
    }
    if (lev < lvl) {
        ca.photon[c] = -1.0;
        return;
    }
    const double dt = ca.max_ts * ssw::powi(0.5, lev);
    const uint32_t ps = g.pslot[c];
    const bool has_p = ps != kNone && fl.P;
    const double src = ca.src[c];
    double rate = 0.0, incoming = 0.0;
    for (int d0 = 0; d0 < g.D; d0 += kChemDirs) {
        R inc[kChemDirs], per[kChemDirs];
#pragma unroll
        for (int j = 0; j < kChemDirs; j++)
            inc[j] = fl.I[iidx(fl, g.N, (uint32_t)min(d0 + j, g.D - 1), (uint32_t)c)];
        // current periodic source (k_periodic ran after the sweep)
#pragma unroll
        for (int j = 0; j < kChemDirs; j++) per[j] = (R)0;
        if (has_p) {
#pragma unroll
            for (int j = 0; j < kChemDirs; j++) per[j] = fl.P[(size_t)min(d0 + j, g.D - 1) * g.Nper + ps];
        }
#pragma unroll
        for (int j = 0; j < kChemDirs; j++) {
            if (d0 + j >= g.D) break;
            const double i = (double)inc[j] * ca.lref;
            rate += (i + src) + (double)per[j] * ca.lref;  // sum over d of Site::get_rate, in direction order
            incoming += i;                                 // the photon rate, as k_fluxes sums it
        }
    }
    ca.photon[c] = incoming;
    double rel;
    if (fabs(rate) < fabs(ca.thr)) {
        rel = 0.0;
    } else {  // PhotonRate::relative_change_to(..).abs() (src/chemistry/mod.rs:73-77)
        rel = fabs(fmin(fabs(fabs(rate - ca.prev_rate[c]) / rate), ssw::kInvEps));
    }
    ca.prev_rate[c] = rate;
    const double rate_ts = dt / rel;
    ssw::Cell cell = solver_cell(ca, c, rate);
    const ssw::Floor floor{ca.prevent_cooling != 0, cell.T, cell.x};
    ssw::Walk w;
    w.dt = dt;
    const bool done = ssw::walk_step(cell, floor, dt, ca.safety, w, ssw::Serial());
    const unsigned long long m = __ballot(!done);
    if (m) {  // queued, with the photon rate's timescale in change_ts
        uint32_t at = 0;
        const int leader = __ffsll((long long)__ballot(1)) - 1;
        if ((int)__lane_id() == leader) at = atomicAdd(&ca.queue[0], (uint32_t)__popcll(m));
        at = (uint32_t)__shfl((int)at, leader);
        if (!done) {
            ca.queue[2 + at + (uint32_t)__popcll(m & ((1ull << __lane_id()) - 1ull))] = (uint32_t)c;
            ca.change_ts[c] = rate_ts;
        }
    }
    if (done) finish_chemistry<R>(ca, c, cell, rate_ts, w, true);
}

// The queued cells' sub-steps, from the first rejection on. Bound: the chain
// of one cell's sub-steps (up to a few hundred near a source), each mostly its
// powers (0.4 us each). So a quad of lanes takes a cell and shares them, two
// rounds of them before the temperature's step and two before the ionised
// fraction's instead of eleven powers, and a quad that has finished its cell
// takes the next one while the others of its wave go on. About half of the
// attempts are rejected and made again with half the step; so where there are
// lanes for it (few cells queued, or the queue empty and the quads of a row of
// 16 lanes idle), `team` = 2 or 4 quads take one cell, quad q its step halved
// q times, and the first of them that is accepted counts: what they would come
// to one after the other. First step of 262144 cells with 64 sources: 3.03 ms
// with a quad a cell, 1.66 like this; of 32768 cells 1.37 and 0.86; both some
// 0.02 once the gas has settled.
template <typename R, int kJobs>
__global__ void __launch_bounds__(64) k_chemistry_tail(const ChemJobs<R, kJobs> jobs) {
    const Geo& g = jobs.mine().g;
    const ChemArgs& ca = jobs.mine().ca;
    const uint32_t n = ca.queue[0], lane = threadIdx.x;
    uint32_t team = n <= gridDim.x * 4u ? 4u : n <= gridDim.x * 8u ? 2u : 1u;
    const uint32_t per = 16u / team, first = gridDim.x * per;
    uint32_t i = blockIdx.x * per + lane / (4u * team);
    int64_t c = 0;
    double dt = 0.0;
    ssw::Cell cell{};
    ssw::Floor floor{};
    ssw::Walk w;
    ssw::HeatRates h{};
    bool have = false, hot = false;  // hot: h belongs to the cell's state
    for (;;) {
        if (!have && i < n) {
            c = ca.queue[2 + i];
            dt = ca.max_ts * ssw::powi(0.5, g.level[c]);
            cell = solver_cell(ca, c, ca.prev_rate[c]);
            floor = ssw::Floor{ca.prevent_cooling != 0, cell.T, cell.x};
            w = ssw::Walk();
            w.depth = 1;  // the full step was rejected: its two halves are pending
            w.lo = 2;
            w.dt = dt / 2.0;
            have = true;
            hot = false;
        }
        const unsigned long long busy = __ballot(have);
        if (busy == 0ull) break;
        // a row with idle quads (the queue is empty): fewer, larger teams
        const uint32_t row = (uint32_t)(busy >> (lane & 48u)) & 0xFFFFu, cells = (uint32_t)__popc(row) / (4u * team);
        const uint32_t want = cells == 1u ? 4u : cells == 2u ? 2u : team;
        if (__ballot(want > team)) {
            uint32_t from = lane;
            bool moved = want > team;
            if (moved) {  // the (lane / team's lanes)-th of the row's cells
                uint32_t left = row;
                const uint32_t lanes = (1u << (4u * team)) - 1u;
                if (cells == 2u && (lane & 15u) >= 8u) left &= ~(lanes << (uint32_t)(__ffs((int)left) - 1));
                from = (lane & 48u) + (uint32_t)(__ffs((int)left) - 1);
            }
            auto take = [&](auto v) { return __shfl(v, (int)from); };
            c = (int64_t)take((long long)c);
            dt = take(dt);
            cell.x = take(cell.x);
            cell.T = take(cell.T);
            cell.rho = take(cell.rho);
            cell.vol = take(cell.vol);
            cell.len = take(cell.len);
            cell.rate = take(cell.rate);
            cell.a = ca.scale_factor;
            floor.on = ca.prevent_cooling != 0;
            floor.T = take(floor.T);
            floor.x = take(floor.x);
            w.lo = (uint64_t)take((unsigned long long)w.lo);
            w.hi = (uint64_t)take((unsigned long long)w.hi);
            w.depth = take(w.depth);
            w.dt = take(w.dt);
            w.ts = take(w.ts);
            w.proc = take(w.proc);
            if (moved) {
                team = want;
                have = true;
                hot = false;
            }
        }
        if (!have) continue;
        const uint32_t base = lane & ~(4u * team - 1u), q = (lane - base) / 4u;
        bool ended = false;
        ssw::clamp_state(cell, floor);
        if (w.depth > ssw::kMaxDepth) {
            w.overflow(dt);
            ended = true;
        } else {
            if (!hot) h = ssw::heat_rates(cell, ssw::Quad());
            ssw::Cell t = cell;
            double dtq = w.dt, ts = 0.0;
            for (uint32_t k = 0; k < q; k++) dtq = dtq / 2.0;
            int proc = 0;
            const bool ok = w.depth + (int)q <= ssw::kMaxDepth &&
                            ssw::try_step(t, floor, dtq, ca.safety, ts, proc, h, ssw::Quad());
            const uint32_t m = (uint32_t)(__ballot(ok) >> base) & ((1u << (4u * team)) - 1u);
            const uint32_t at = m ? (uint32_t)(__ffs((int)m) - 1) : 0u;
            const uint32_t rejected = m ? at / 4u : min(team, (uint32_t)(ssw::kMaxDepth + 1 - w.depth));
            for (uint32_t k = 0; k < rejected; k++) w.halve();
            hot = m == 0u;
            if (m) {
                cell.T = __shfl(t.T, (int)(base + at));
                cell.x = __shfl(t.x, (int)(base + at));
                w.ts = __shfl(ts, (int)(base + at));
                w.proc = __shfl(proc, (int)(base + at));
                ended = w.next(dt);
            }
        }
        if (ended) {
            finish_chemistry<R>(ca, c, cell, ca.change_ts[c], w, lane == base);
            have = false;
            uint32_t next = 0;
            if (lane == base) next = atomicAdd(&ca.queue[1], 1u);
            i = first + (uint32_t)__shfl((int)next, (int)base);
        }
    }
}

// The optional chemistry outputs (src/sweep/chemistry_output.rs:25-67) of
// every cell: Sweep::get_solver (src/sweep/mod.rs:612-632) with the rate
// summed over directions in direction order as in update_chemistry, the
// current x and T, and no floor (an output that is NULL is left out).
template <typename R>
__global__ void __launch_bounds__(64) k_chem_outputs(Geo g, Flux<R> fl, ChemArgs ca, double* out0, double* out1,
                                                     double* out2, double* out3) {
    int64_t c = (int64_t)xcd_block(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
    if (c >= g.N) return;
    const uint32_t ps = g.pslot[c];
    const bool has_p = ps != kNone && fl.P;
    const double src = ca.src[c];
    double rate = 0.0;
#pragma unroll 6
    for (int d = 0; d < g.D; d++) {
        const double inc = (double)fl.I[iidx(fl, g.N, (uint32_t)d, (uint32_t)c)] * ca.lref;
        const double per = has_p ? (double)fl.P[(size_t)d * g.Nper + ps] * ca.lref : 0.0;
        rate += (inc + src) + per;  // Site::get_rate (src/sweep/site.rs:53-56)
    }
    ssw::Cell cell;
    cell.x = ca.x[c];
    cell.T = ca.T[c];
    cell.rho = ca.rho[c];
    cell.vol = ca.vol[c];
    cell.len = ca.size[c];
    cell.rate = rate;
    cell.a = ca.scale_factor;
    double out[4];
    ssw::chemistry_outputs(cell, out);
    if (out0) out0[c] = out[0];
    if (out1) out1[c] = out[1];
    if (out2) out2[c] = out[2];
    if (out3) out3[c] = out[3];
}

// update_timestep_levels (src/sweep/mod.rs:576-589) for all cells. Marks the
// sweep levels whose active set changed.
__global__ void k_levels(Geo g, const double* change_ts, uint8_t* level, double max_ts, double safety,
                         int lowest) {
    int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= g.N) return;
    double desired = safety * change_ts[c];
    int lev = ssw::level_from_ratio(max_ts / desired, g.L);
    if (lev < lowest) lev = lowest;
    int old = level[c];
    level[c] = (uint8_t)lev;
    for (int l = 0; l < g.L; l++)
        if ((old >= l) != (lev >= l)) g.need[l] = 1;
}

// Pull evaluation of the current incoming / outgoing / periodic rates of every
// (cell, direction) in SI units (parity hooks, rotations, and the photon-rate
// output after a restricted sweep). A wave takes 64 consecutive cells and
// kFluxDirs consecutive directions, a workgroup all directions of its cells:
// each face is read once per wave and tested against the wave's directions, so
// that their gathers of X (the bound: two dependent loads each, through xpos)
// are independent of one another and in flight together. The sums run over
// the faces in face order, the photon rate over the directions in direction
// order (wave after wave through LDS). Photon rate of 262144 cells x 84
// directions: 9.2 ms with one thread per cell and its directions one after the
// other, 2.46 ms like this.
template <typename R, bool kAll>
__global__ void __launch_bounds__(1024) k_fluxes(Geo g, Flux<R> fl, double lref, double* I_out, double* O_out,
                                                 double* P_out, double* photon_rate, const uint32_t* rate_idx,
                                                 const double* missing) {
    __shared__ double sum[kFluxCells];
    const uint32_t lane = threadIdx.x % kFluxCells;
    const uint32_t w = __builtin_amdgcn_readfirstlane(threadIdx.x / kFluxCells);  // uniform: scalar direction loads
    const int64_t c0 = (int64_t)blockIdx.x * kFluxCells + lane;
    const bool valid = c0 < g.N;
    // only cells without a rate: where none of the workgroup's is
    if (missing && !__ballot(valid && missing[c0] < 0.0)) return;
    const uint32_t c = valid ? (uint32_t)c0 : 0u;
    const int d0 = (int)w * kFluxDirs;
    double A[kFluxDirs];
    R inc[kFluxDirs], per[kFluxDirs];
#pragma unroll
    for (int j = 0; j < kFluxDirs; j++) {
        A[j] = 0.0;
        inc[j] = per[j] = (R)0;
    }
    const uint32_t f1 = valid ? g.off[c + 1] : 0u;
    for (uint32_t f = valid ? g.off[c] : 0u; f < f1; f++) {
        const double4 a = g.geo[f];
        const uint32_t nk = g.nk[f];
        const uint32_t nb = nk & kNbrMask, kind = nk >> 30;
#pragma unroll
        for (int j = 0; j < kFluxDirs; j++) {
            const int d = min(d0 + j, g.D - 1);  // past the last direction: repeated, not used
            const double dd = fdot(a, g.dirs[3 * d], g.dirs[3 * d + 1], g.dirs[3 * d + 2]);
            if (kAll && dd > 0.0) A[j] += a.w * dd;
            const bool up = dd < 0.0 && (kAll ? kind != kKindBoundary : kind == kKindLocal);
            if (up) {
                const R v = (R)(a.w * fl.inv_aref * -dd) * fl.X[xidx(fl, g.N, (uint32_t)d, nb)];
                if (!kAll || kind == kKindLocal) inc[j] += v;
                else per[j] += v;
            }
        }
    }
    double in_si[kFluxDirs];
#pragma unroll
    for (int j = 0; j < kFluxDirs; j++) {
        in_si[j] = 0.0;
        const int d = d0 + j;
        if (!valid || d >= g.D) continue;
        const size_t o = (size_t)d * g.N + c;
        if (fl.offI) inc[j] = fl.offI[o] + inc[j];
        in_si[j] = (double)inc[j] * lref;
        if (kAll) {
            if (fl.offP && g.pslot[c] != kNone) per[j] = fl.offP[(size_t)d * g.Nper + g.pslot[c]] + per[j];
            if (I_out) I_out[o] = in_si[j];
            if (P_out) P_out[o] = (double)per[j] * lref;
            if (O_out) O_out[o] = (double)fl.X[xidx(fl, g.N, (uint32_t)d, c)] * (A[j] * fl.inv_aref) * lref;
        }
    }
    if (kAll) return;
    const uint32_t nw = blockDim.x / kFluxCells;
    for (uint32_t k = 0; k < nw; k++) {
        if (k == w) {
            double t = k ? sum[lane] : 0.0;
#pragma unroll
            for (int j = 0; j < kFluxDirs; j++)
                if (d0 + j < g.D) t += in_si[j];
            sum[lane] = t;
        }
        __syncthreads();
    }
    // rate_idx: the caller's index of each internal cell (NULL: internal order)
    if (w == 0 && valid) photon_rate[rate_idx ? rate_idx[c] : c] = sum[lane];
}

// rotate_directions_system (src/sweep/direction/mod.rs:158-175), state part,
// one thread per (cell c, direction d) after the schedule of the rotated
// directions is built: remap (:190-205) leaves every rate of direction d equal
// to the old rate of the last direction times kept[d] (1 or 0), for incoming,
// outgoing and periodic rates alike. Old rates (FP64, SI, [d*N + c]) come
// from k_fluxes before the rotation. Writes X = O / A with the rotated
// downwind area, I, the periodic source, and the remapped I and periodic
// source into the offsets (k_rotate_offsets subtracts the pull sums).
template <typename R>
__global__ void k_rotate_state(Geo g, Flux<R> fl, const double* __restrict__ kept, const double* __restrict__ Iold,
                               const double* __restrict__ Oold, const double* __restrict__ Pold) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (int64_t)g.D * g.N) return;
    const uint32_t d = (uint32_t)(t / g.N);
    const uint32_t c = (uint32_t)(t - (int64_t)d * g.N);
    const size_t last = (size_t)(g.D - 1) * g.N + c;
    const double k = kept[d];
    const double inc = Iold[last] * k, out = Oold[last] * k, per = Pold[last] * k;
    const double dx = g.dirs[3 * d], dy = g.dirs[3 * d + 1], dz = g.dirs[3 * d + 2];
    double A = 0.0;
    for (uint32_t f = g.off[c]; f < g.off[c + 1]; f++) {
        const double4 a = g.geo[f];
        const double dd = fdot(a, dx, dy, dz);
        if (dd > 0.0) A += a.w * fl.inv_aref * dd;
    }
    const R Ar = (R)A;
    const R o = (R)(out * fl.inv_lref);
    fl.X[xidx(fl, g.N, d, c)] = (Ar > (R)0) ? o / Ar : (R)0;
    const size_t oi = (size_t)d * g.N + c;
    fl.I[iidx(fl, g.N, d, c)] = (R)(inc * fl.inv_lref);
    fl.offI[oi] = (R)(inc * fl.inv_lref);
    const uint32_t ps = g.pslot[c];
    if (ps != kNone && fl.P) {
        fl.P[(size_t)d * g.Nper + ps] = (R)(per * fl.inv_lref);
        fl.offP[(size_t)d * g.Nper + ps] = (R)(per * fl.inv_lref);
    }
}

// The offsets of the rotated state: remapped rate minus the pull sum of the
// rotated X over the upwind faces (local for I, periodic for the periodic
// source), so that offset + sum gives the remapped rate back and grows by the
// corrections of later solves, as the reference's accumulated rates do.
template <typename R>
__global__ void k_rotate_offsets(Geo g, Flux<R> fl) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (int64_t)g.D * g.N) return;
    const uint32_t d = (uint32_t)(t / g.N);
    const uint32_t c = (uint32_t)(t - (int64_t)d * g.N);
    const double dx = g.dirs[3 * d], dy = g.dirs[3 * d + 1], dz = g.dirs[3 * d + 2];
    R inc = 0, per = 0;
    for (uint32_t f = g.off[c]; f < g.off[c + 1]; f++) {
        const double4 a = g.geo[f];
        const uint32_t nk = g.nk[f];
        const double dd = fdot(a, dx, dy, dz);
        if (dd < 0.0 && (nk >> 30) != kKindBoundary) {
            const R v = (R)(a.w * fl.inv_aref * -dd) * fl.X[xidx(fl, g.N, d, nk & kNbrMask)];
            if ((nk >> 30) == kKindLocal) inc += v;
            else per += v;
        }
    }
    const size_t oi = (size_t)d * g.N + c;
    fl.offI[oi] = fl.offI[oi] - inc;
    const uint32_t ps = g.pslot[c];
    if (ps != kNone && fl.P) fl.offP[(size_t)d * g.Nper + ps] = fl.offP[(size_t)d * g.Nper + ps] - per;
}

// dst[idx[i]] = src[i]: a per-cell array from the internal into the caller's order.
template <typename T>
__global__ void k_to_caller(const T* __restrict__ src, const uint32_t* __restrict__ idx, T* __restrict__ dst,
                            int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) dst[idx[i]] = src[i];
}

// Outputs of up to 6 per-cell arrays for the caller's cells [j0, j0 + n) into
// pinned host memory, in the caller's order (perm: internal cell of each
// caller's cell; NULL: the same): consecutive lanes write consecutive values
// over the bus, and the scattered side of the permutation stays in HBM.
struct OutputArrays {
    const double* a[6];
    const uint8_t* level;
    int n;
};
__global__ void __launch_bounds__(kBlock) k_stage_outputs(OutputArrays src, const uint32_t* __restrict__ perm,
                                                          uint32_t j0, uint32_t n, uint32_t stride,
                                                          double* __restrict__ out) {
    const uint32_t j = blockIdx.x * kBlock + threadIdx.x;
    if (j >= n) return;
    const uint32_t i = perm ? perm[j0 + j] : j0 + j;
    for (int k = 0; k < src.n; k++) out[(size_t)k * stride + j] = src.a[k][i];
    if (src.level) reinterpret_cast<uint8_t*>(out + (size_t)src.n * stride)[j] = src.level[i];
}

// Direction-major copy of X from the schedule-position order.
template <typename R>
__global__ void k_gather_x(const R* X, const uint32_t* xpos, R* out, int64_t n) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = X[xpos[i]];
}

// X from the direction-major order into the schedule-position order.
template <typename R>
__global__ void k_scatter_x(R* X, const uint32_t* xpos, const R* in, int64_t n) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) X[xpos[i]] = in[i];
}

__global__ void k_fill_u32(uint32_t* p, uint32_t v, int64_t n) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

template <typename R>
__global__ void k_attenuation(const double* src, double lref, const double* rho, const double* x, const double* size,
                              SA<R>* sa, int64_t n) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    sa[i].x = (R)(src[i] / lref);
    sa[i].y = (R)ssw::non_absorbed_fraction(rho[i], x[i], size[i]);
}

// ---------------------------------------------------------------------------
// grid upload: the caller's arrays are copied as they are, and ordered and
// packed here. On the host (a sort of the Morton codes, and faces gathered
// cell by cell into new arrays) it took 4.2 ms for 32768 cells with 15.5 faces
// each, and as long again where the arrays' pages were new to the process.

// Morton (Z-order) code of a position quantised to 21 bits per axis.
__global__ void k_morton(const double* __restrict__ pos, double3 lo, double3 inv_ext, uint64_t* __restrict__ key,
                         uint32_t* __restrict__ idx, uint32_t n) {
    const uint32_t c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= n) return;
    const double l[3] = {lo.x, lo.y, lo.z}, e[3] = {inv_ext.x, inv_ext.y, inv_ext.z};
    uint64_t code = 0;
    for (int k = 0; k < 3; k++) {
        double u = (pos[3 * (size_t)c + k] - l[k]) * e[k];
        u = u < 0.0 ? 0.0 : u;
        u = 1.0 < u ? 1.0 : u;
        const uint64_t q = (uint64_t)(u * 2097151.0);
        for (int b = 0; b < 21; b++) code |= ((q >> b) & 1ull) << (3 * b + k);
    }
    key[c] = code;
    idx[c] = c;
}

// Per-cell array in the caller's order -> internal order.
template <typename T>
__global__ void k_to_internal(const T* __restrict__ in, const uint32_t* __restrict__ inv, T* __restrict__ out,
                              uint32_t n) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = in[inv[i]];
}

// Faces of the caller's cells c0 .. c1-1 (f0: the first of them, at index 0 of
// the four face arrays) to their places in the internal order, each cell's
// faces in the caller's order, 16 lanes to a cell. A non-periodic sweep treats
// periodic faces as boundaries. pcount: a cell's periodic faces, with 2^32 if
// it has any. bad: the first invalid face, 2 * its place + 1 if it is its
// neighbour that is out of range.
__global__ void __launch_bounds__(kBlock) k_pack_faces(
    const uint32_t* __restrict__ coff, uint32_t c0, uint32_t c1, uint32_t f0, const double* __restrict__ normal,
    const double* __restrict__ area, const int32_t* __restrict__ nbr, const uint8_t* __restrict__ kind,
    const uint32_t* __restrict__ perm, const uint32_t* __restrict__ off, int periodic, uint32_t n,
    double4* __restrict__ geo, uint32_t* __restrict__ nk, uint64_t* __restrict__ pcount, unsigned long long* bad) {
    const uint32_t c = c0 + blockIdx.x * (kBlock / 16) + threadIdx.x / 16, sub = threadIdx.x & 15u;
    if (c >= c1) return;
    const uint32_t i = perm ? perm[c] : c, a = coff[c], m = coff[c + 1] - a, o = off[i];
    uint32_t np = 0;
    for (uint32_t r = 0; r < m; r += 16u) {
        const uint32_t j = r + sub;
        bool per = false;
        if (j < m) {
            const uint32_t f = a - f0 + j, fi = o + j;
            uint32_t k = kind[f];
            if (k > 2u) {
                atomicMin(bad, 2ull * fi);
                k = kKindBoundary;
            }
            if (k == kKindPeriodic && !periodic) k = kKindBoundary;
            uint32_t nb = 0;
            if (k != kKindBoundary) {
                const int32_t v = nbr[f];
                if (v < 0 || (uint32_t)v >= n) atomicMin(bad, 2ull * fi + 1ull);
                else nb = perm ? perm[v] : (uint32_t)v;
            }
            per = k == kKindPeriodic;
            geo[fi] = make_double4(normal[3 * (size_t)f], normal[3 * (size_t)f + 1], normal[3 * (size_t)f + 2], area[f]);
            nk[fi] = nb | (k << 30);
        }
        np += (uint32_t)__popc((uint32_t)(__ballot(per) >> (threadIdx.x & 48u)) & 0xFFFFu);
    }
    if (sub == 0) pcount[i] = np ? (1ull << 32) | np : 0ull;
}

// The periodic cells' slots and the list of their periodic faces, from the
// prefix sums of pcount.
__global__ void k_pack_periodic(const uint64_t* __restrict__ pcount, const uint64_t* __restrict__ psum,
                                const uint32_t* __restrict__ off, const double4* __restrict__ geo,
                                const uint32_t* __restrict__ nk, uint32_t n, uint32_t* __restrict__ pslot,
                                uint32_t* __restrict__ pcells, uint32_t* __restrict__ pfoff,
                                double4* __restrict__ pgeo, uint32_t* __restrict__ pnb) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i > n) return;
    const uint32_t slot = (uint32_t)(psum[i] >> 32);
    uint32_t at = (uint32_t)psum[i];
    if (i == n || pcount[i]) pfoff[slot] = at;
    if (i == n) return;
    pslot[i] = pcount[i] ? slot : kNone;
    if (!pcount[i]) return;
    pcells[slot] = i;
    for (uint32_t f = off[i]; f < off[i + 1]; f++)
        if ((nk[f] >> 30) == kKindPeriodic) {
            pgeo[at] = geo[f];
            pnb[at++] = nk[f] & kNbrMask;
        }
}

// ---------------------------------------------------------------------------
// host side

// TimestepState (src/sweep/timestep_state.rs:4-80)
struct TimestepState {
    double max_ts = 0;
    int L = 1;
    int lowest = 0;
    bool first_done = false;
    void init(double m, int n) {
        max_ts = m;
        L = n;
        lowest = n - 1;
        first_done = false;
    }
    std::vector<int> sweep_order() const {  // :22-27, 70-75
        int num = L - lowest;
        std::vector<int> out;
        for (uint32_t i = 0; i < (1u << (num - 1)); i++) {
            int fb = i ? __builtin_ctz(i) : num - 1;
            out.push_back(lowest + (num - 1 - fb));
        }
        return out;
    }
    void advance() {  // :37-48
        if (first_done && lowest > 0) lowest -= 1;
        if (!first_done) first_done = true;
    }
    double current_max_timestep() const { return max_ts * ssw::powi(0.5, lowest); }
};

unsigned grid_for(int64_t n) { return (unsigned)std::max<int64_t>(1, (n + kBlock - 1) / kBlock); }

}  // namespace

// Shared with the library's other translation units (placement.hip): the
// thread's error message and the lock that device allocations hold shared
// while a stream capture holds it exclusively.
namespace ssw_detail {
void set_error(const std::string& msg) { g_err = msg; }
std::shared_mutex& capture_mutex() { return g_capture_mu; }
}  // namespace ssw_detail

struct ssw_sweep {
    ssw_sweep_parameters p{};
    int D = 0;
    std::vector<double> dirs;
    int device = 0;
    hipStream_t stream = nullptr;
    bool fp32 = false;
    int mode_request = SSW_TRANSPORT_MODE_AUTO;
    int rec_block = 64;                             // compiled replay block size
    bool graphs_on = true;                          // capture replays as graphs
    bool narrow_runs = true;                        // runs of narrow level sets in one workgroup
    bool dir_sweeps = false;                        // full sweeps: one workgroup per direction
    // direction sweeps' schedule: tiles, their blobs, and per direction {first
    // tile, tiles, level sets, wide}; the cell of every task in X's order, and
    // in that order the cell inputs of the running sweep (k_dir_inputs); the
    // upwind counts the build starts from
    uint4 *d_dirblob = nullptr, *d_dirtiles = nullptr, *d_dirinfo = nullptr;
    uint32_t* d_dircell = nullptr;
    void* d_dirsa = nullptr;
    uint8_t* d_dirlev = nullptr;
    uint8_t* d_nup = nullptr;
    int group_request = kGroupLevels;               // level sets per grouped launch (1: off)
    int group_block = kGroupT;                      // grouped replay: root tasks per workgroup
    // grouped replay of full sweeps (compiled): per group of level sets its
    // first level set, level-set count and cones
    struct Group {
        int k0, levels;
        uint32_t desc0, ndesc;
        PassTab passes;  // cone ranges of the build passes, relative to desc0
        uint32_t words;  // tasks of its largest cone
        int waves;       // of its workgroups
        uint32_t slot0;  // its first tile descriptor
    };
    std::vector<Group> groups;
    uint4 *d_coneblob = nullptr, *d_conetiles = nullptr;
    uint32_t* d_conemore = nullptr;
    uint32_t* d_gmap = nullptr;                     // group of each cone
    uint4* d_ginfo = nullptr;                       // per group: first level set, waves, first tile, first cone
    uint32_t ndesc = 0;
    // restricted sweeps (level >= 1): kept cones, active tasks per group
    std::vector<uint32_t*> d_gsel_l;
    uint32_t* d_gcount = nullptr;
    uint32_t* d_gbase = nullptr;                    // first cone of each group
    uint32_t* d_gblocks = nullptr;                  // restricted sweep: workgroups with active tasks per group
    // global cone index of every pass boundary of every group (group
    // gi's npass + 1 boundaries from pbound_start[gi]); per restricted sweep
    // level the pass ranges of each group's kept cones
    uint32_t* d_pbound = nullptr;
    std::vector<uint32_t> pbound_start;
    // restricted sweeps' filter scratch, held from the cone build on: kept
    // flags, their prefix sum, the pass bounds' packed positions and the scan's
    // temporary storage
    uint32_t *d_gf_kept = nullptr, *d_gf_pos = nullptr, *d_gf_pbval = nullptr;
    uint8_t* d_gf_scan = nullptr;
    size_t gf_scan_bytes = 0;
    std::vector<std::vector<PassTab>> gpass_l;
    std::vector<std::vector<uint32_t>> gcount, gblocks;
    int64_t group_tasks = 0;                        // tasks solved per full sweep by the grouped replay
    bool group_fallback = false;                    // groups requested but a cone did not fit
    bool compiled = false;
    // grid
    int64_t N = 0, F = 0, Nper = 0;
    bool have_grid = false, have_state = false;
    bool have_schedule = false;                     // the schedule is whole (a failed rotation may leave none)
    // internal cell order: internal index perm[c] for caller's cell c (Morton
    // order of the positions given with ssw_set_cell_positions), inv = perm^-1
    std::vector<double> pos;
    std::vector<uint32_t> perm, inv;
    bool permuted = false;
    uint32_t *d_inv = nullptr, *d_perm = nullptr;   // inv and perm on the device (permuted grids only)
    bool downloaded = false;                        // later downloads go through the pinned staging
    uint32_t *d_off = nullptr, *d_nk = nullptr, *d_pslot = nullptr, *d_pcells = nullptr;
    std::vector<uint32_t> h_pcells;                 // internal cell of each periodic slot
    uint32_t *d_pfoff = nullptr, *d_pnb = nullptr;
    double4* d_pgeo = nullptr;
    double4* d_geo = nullptr;
    double *d_dirs = nullptr, *d_vol = nullptr, *d_size = nullptr;
    double aref = 1.0;
    double dw[3] = {0, 0, 0};
    int64_t ovf_total = 0;
    bool uneven_faces = false;                      // k_check_mirror's `uneven`
    // upwind counters, held only while a layering or a count runs
    uint32_t *d_cnt = nullptr, *d_need = nullptr;
    // full schedule
    int kmax = 0;
    std::vector<uint32_t> full_start;               // kmax + 1 level starts
    uint32_t* d_fstart = nullptr;
    uint4* d_recs = nullptr;                        // geometric
    uint4* d_hdr = nullptr;                         // compiled
    void* d_A = nullptr;
    void* d_planes = nullptr;
    uint32_t* d_ovf_start = nullptr;
    void* d_ovf = nullptr;
    uint32_t* d_xpos = nullptr;                     // compiled: schedule position of each (d, c)
    // compaction to active sets
    uint32_t nchunks = 0;
    uint4* d_chunks = nullptr;
    uint32_t* d_first_chunk = nullptr;              // kmax: first chunk of each level set
    uint32_t *d_ccount = nullptr, *d_coff = nullptr, *d_cstart = nullptr;
    void* d_scan_tmp = nullptr;
    size_t scan_tmp_bytes = 0;
    std::vector<uint32_t*> d_idx;                   // per sweep level >= 1: active positions
    std::vector<std::vector<uint32_t>> cstart;      // per sweep level: level starts in idx
    std::vector<int> list_ok;                       // per sweep level: idx / cstart current
    // per sweep level: the grouped replay's filter kept every task (the
    // active set is all cells), so the level replays the full sweep's launches
    std::vector<int> list_full;
    std::vector<int> replays;                       // per sweep level: replays since the list was made
    std::vector<hipGraphExec_t> graphs;             // per sweep level: captured replay
    // replay plan per sweep level: one launch per level set, or one launch per
    // run of consecutive narrow level sets (compiled replay)
    struct ReplayItem {
        int k;          // level set (single launch) or first level set of the run / group
        int levels;     // 0: single launch; else the run's non-empty level sets (or the group's level sets)
        uint32_t tab;   // the run's first entry in the run table (the group's index)
        int group;      // 1: a group of the grouped replay
    };
    std::vector<std::vector<ReplayItem>> plan;
    std::vector<std::vector<uint4>> runtab;         // host copies of the run tables
    std::vector<uint4*> d_runtab;
    // state
    double *d_rho = nullptr, *d_x = nullptr, *d_T = nullptr, *d_src = nullptr;
    void* d_sa = nullptr;                           // SA<R>: {transport source / D, attenuation}
    double *d_sts = nullptr, *d_prev = nullptr, *d_change = nullptr;
    // of the last step: chemistry updates, then the 3 limiting processes' counts
    unsigned long long* d_active = nullptr;
    double* d_photon = nullptr;                     // photon rates of a download (internal order)
    double* d_rate = nullptr;                       // photon rates from the last sweep's chemistry
    uint32_t* d_chemq = nullptr;                    // k_chemistry's queue (ChemArgs::queue)
    uint8_t* d_level = nullptr;
    void *d_X = nullptr, *d_I = nullptr, *d_P = nullptr;
    void *d_offI = nullptr, *d_offP = nullptr;      // rate offsets after a rotation (Flux::offI / offP)
    bool rotated = false;                           // directions rotated since ssw_create
    // every source and periodic source is >= 0, every face's area, and every X
    // (not known after a checkpoint was loaded, until a full sweep has solved
    // them all): no incoming rate is negative, so none is clamped when it is stored
    bool nonneg = false, areas_nonneg = false, x_nonneg = false;
    // the incoming rates that the last sweep's cells read are the pull sums
    // over the current X: nothing was clamped, no rotation has left offsets,
    // and no cell was solved before an upwind neighbour (uneven_faces)
    // (other cells may have been solved before their upwind neighbours were
    // solved again: their d_rate is -1)
    bool rates_current = false;
    bool rates_partial = false;                     // the last sweep did not solve every cell
    unsigned long long* d_fail = nullptr;
    double lref = 1.0;
    TimestepState ts;
    int64_t bytes = 0, peak_bytes = 0;
    int64_t capacity = 0;                           // expected_free
    std::unordered_map<void*, size_t> alloc;
    int64_t sweeps_last = 0;
    int64_t builds_last = 0;
    int64_t capture_failures = 0;
    // timing
    bool timing = false;
    std::vector<hipEvent_t> ev;
    hipEvent_t sync_ev = nullptr;                   // orders the handle's stream against a packed step
    uint64_t uid = 0;                               // process-unique handle id (packed-step graphs)
    uint64_t epoch = 0;                             // bumped whenever a replay plan or its graph changes
    double t_transport_total = 0, t_chem_total = 0, t_build_total = 0;
    int64_t n_transport = 0;
};

namespace {

std::array<std::atomic<int64_t>, kMaxDevices> g_held{};  // device bytes of all handles, per device

std::atomic<int64_t>& held(const ssw_sweep* s) { return g_held[(size_t)s->device % kMaxDevices]; }

// Device memory that is free once all that the process's handles have freed is
// back. Freed memory is reported, and can be allocated again, only some time
// after the free (16.8 M cells: 57 GB were still missing when the tiles were to
// be allocated), so it is counted from the most that was free and held together
// since the call began (expect_frees).
int64_t expected_free(ssw_sweep* s) {
    size_t free_b = 0, total_b = 0;
    if (hipMemGetInfo(&free_b, &total_b) != hipSuccess) {
        (void)hipGetLastError();
        return 0;
    }
    s->capacity = std::max(s->capacity, (int64_t)free_b + held(s));
    return s->capacity - held(s);
}

void expect_frees(ssw_sweep* s) {
    s->capacity = 0;
    (void)expected_free(s);
}

template <typename T>
void dfree(ssw_sweep* s, T*& p) {
    if (p) {
        std::shared_lock<std::shared_mutex> lock(g_capture_mu);
        auto it = s->alloc.find((void*)p);
        if (it != s->alloc.end()) {
            s->bytes -= (int64_t)it->second;
            held(s) -= (int64_t)it->second;
            s->alloc.erase(it);
        }
        (void)hipFree((void*)p);
    }
    p = nullptr;
}

template <typename T>
int dalloc(ssw_sweep* s, T** p, size_t count) {
    dfree(s, *p);
    if (count == 0) count = 1;
    hipError_t e;
    for (int tries = 0;; tries++) {
        {
            std::shared_lock<std::shared_mutex> lock(g_capture_mu);
            e = hipMalloc((void**)p, count * sizeof(T));
        }
        // memory that was freed and is not back yet: at most 2 s
        if (e != hipErrorOutOfMemory || tries == 100 || expected_free(s) < (int64_t)(count * sizeof(T))) break;
        (void)hipGetLastError();
        std::this_thread::sleep_for(std::chrono::milliseconds(20));
    }
    if (e != hipSuccess) {
        *p = nullptr;
        (void)hipGetLastError();
        return fail(SSW_ERR_OOM, std::string("hipMalloc of ") + std::to_string(count * sizeof(T)) +
                                     " bytes failed: " + hipGetErrorString(e));
    }
    s->bytes += (int64_t)(count * sizeof(T));
    held(s) += (int64_t)(count * sizeof(T));
    s->peak_bytes = std::max(s->peak_bytes, s->bytes);
    s->alloc[(void*)*p] = count * sizeof(T);
    return SSW_OK;
}

// Runs its function when the scope ends, also on an early error return: the
// transient device buffers of a call are freed on every path.
struct Defer {
    std::function<void()> f;
    ~Defer() { f(); }
};

size_t real_size(const ssw_sweep* s) { return s->fp32 ? 4 : 8; }
size_t entry_size(const ssw_sweep* s) { return s->fp32 ? sizeof(Entry<float>) : sizeof(Entry<double>); }
size_t sa_size(const ssw_sweep* s) { return s->fp32 ? sizeof(float2) : sizeof(double2); }

Geo make_geo(ssw_sweep* s) {
    Geo g;
    g.N = s->N;
    g.D = s->D;
    g.L = s->p.num_timestep_levels;
    g.off = s->d_off;
    g.geo = s->d_geo;
    g.nk = s->d_nk;
    g.dirs = s->d_dirs;
    g.level = s->d_level;
    g.pslot = s->d_pslot;
    g.pcells = s->d_pcells;
    g.pfoff = s->d_pfoff;
    g.pgeo = s->d_pgeo;
    g.pnb = s->d_pnb;
    g.Nper = s->Nper;
    g.cnt = s->d_cnt;
    g.need = s->d_need;
    return g;
}

template <typename R>
Flux<R> make_flux(ssw_sweep* s) {
    Flux<R> f;
    f.X = (R*)s->d_X;
    f.xpos = s->compiled ? s->d_xpos : nullptr;
    f.I = (R*)s->d_I;
    f.ipos = s->d_dirinfo ? s->d_xpos : nullptr;
    f.P = (R*)s->d_P;
    f.offI = (R*)s->d_offI;
    f.offP = (R*)s->d_offP;
    f.sa = (const SA<R>*)s->d_sa;
    f.inv_lref = 1.0 / s->lref;
    f.inv_aref = 1.0 / s->aref;
    const double thr = s->p.significant_rate_threshold * f.inv_lref;
    f.thr = (R)thr;
    if ((double)f.thr < thr) f.thr = std::nextafter(f.thr, std::numeric_limits<R>::infinity());
    return f;
}

// The internal cell order for the current grid: Morton order of the given
// positions (equal codes in the caller's order), or the caller's order.
int make_order(ssw_sweep* s, int64_t n) {
    s->permuted = (int64_t)s->pos.size() == 3 * n;
    s->perm.resize(n);
    s->inv.resize(n);
    if (!s->permuted) {
        for (int64_t c = 0; c < n; c++) s->perm[c] = s->inv[c] = (uint32_t)c;
        return SSW_OK;
    }
    double lo[3] = {HUGE_VAL, HUGE_VAL, HUGE_VAL}, hi[3] = {-HUGE_VAL, -HUGE_VAL, -HUGE_VAL}, ie[3];
    for (int64_t c = 0; c < n; c++)
        for (int k = 0; k < 3; k++) {
            lo[k] = std::min(lo[k], s->pos[3 * c + k]);
            hi[k] = std::max(hi[k], s->pos[3 * c + k]);
        }
    for (int k = 0; k < 3; k++) ie[k] = hi[k] > lo[k] ? 1.0 / (hi[k] - lo[k]) : 0.0;
    double* pos = nullptr;
    uint64_t *key = nullptr, *key2 = nullptr;
    uint32_t* idx = nullptr;
    uint8_t* tmp = nullptr;
    Defer cleanup{[&] {
        dfree(s, pos);
        dfree(s, key);
        dfree(s, key2);
        dfree(s, idx);
        dfree(s, tmp);
    }};
    TRY(dalloc(s, &pos, 3 * n));
    TRY(dalloc(s, &key, n));
    TRY(dalloc(s, &key2, n));
    TRY(dalloc(s, &idx, n));
    TRY(dalloc(s, &s->d_inv, n));
    TRY(dalloc(s, &s->d_perm, n));
    size_t tb = 0;
    HIP_TRY(hipcub::DeviceRadixSort::SortPairs(nullptr, tb, key, key2, idx, s->d_inv, (int)n, 0, 63, s->stream));
    TRY(dalloc(s, &tmp, tb));
    HIP_TRY(hipMemcpyAsync(pos, s->pos.data(), 3 * n * sizeof(double), hipMemcpyHostToDevice, s->stream));
    k_morton<<<grid_for(n), kBlock, 0, s->stream>>>(pos, make_double3(lo[0], lo[1], lo[2]),
                                                    make_double3(ie[0], ie[1], ie[2]), key, idx, (uint32_t)n);
    HIP_TRY(hipcub::DeviceRadixSort::SortPairs(tmp, tb, key, key2, idx, s->d_inv, (int)n, 0, 63, s->stream));
    k_invert<<<grid_for(n), kBlock, 0, s->stream>>>(s->d_inv, s->d_perm, (uint32_t)n);
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipMemcpyAsync(s->inv.data(), s->d_inv, n * 4, hipMemcpyDeviceToHost, s->stream));
    HIP_TRY(hipMemcpyAsync(s->perm.data(), s->d_perm, n * 4, hipMemcpyDeviceToHost, s->stream));
    HIP_TRY(hipStreamSynchronize(s->stream));
    return SSW_OK;
}

// Per-cell host array in the caller's order -> device array in internal order,
// over `stage` (n values; not read before on the stream) where they differ.
int upload_cells(ssw_sweep* s, const double* in, double* stage, double* out) {
    HIP_TRY(hipMemcpyAsync(s->permuted ? stage : out, in, s->N * sizeof(double), hipMemcpyHostToDevice, s->stream));
    if (s->permuted)
        k_to_internal<double><<<grid_for(s->N), kBlock, 0, s->stream>>>(stage, s->d_inv, out, (uint32_t)s->N);
    HIP_TRY(hipGetLastError());
    return SSW_OK;
}

// Per-cell host array in the caller's order -> internal order.
template <typename T>
const T* to_internal(const ssw_sweep* s, const T* in, std::vector<T>& tmp) {
    if (!s->permuted) return in;
    tmp.resize(s->N);
    for (int64_t i = 0; i < s->N; i++) tmp[i] = in[s->inv[i]];
    return tmp.data();
}

// `blocks` consecutive per-cell arrays (e.g. one per direction) in internal
// order -> the caller's order, in place.
template <typename T>
void to_caller(const ssw_sweep* s, T* a, int64_t blocks) {
    if (!s->permuted) return;
    std::vector<T> tmp(s->N);
    for (int64_t b = 0; b < blocks; b++) {
        T* x = a + b * s->N;
        for (int64_t i = 0; i < s->N; i++) tmp[s->inv[i]] = x[i];
        std::copy(tmp.begin(), tmp.end(), x);
    }
}

// k_fluxes for the incoming, outgoing and periodic rates of every (cell,
// direction).
void launch_fluxes(ssw_sweep* s, const Geo& g, double* dI, double* dO, double* dP) {
    const unsigned nb = (unsigned)((s->N + kFluxCells - 1) / kFluxCells);
    const unsigned lanes = (unsigned)(kFluxCells * ((s->D + kFluxDirs - 1) / kFluxDirs));
    if (s->fp32)
        k_fluxes<float, true><<<nb, lanes, 0, s->stream>>>(g, make_flux<float>(s), s->lref, dI, dO, dP, nullptr,
                                                           nullptr, nullptr);
    else
        k_fluxes<double, true><<<nb, lanes, 0, s->stream>>>(g, make_flux<double>(s), s->lref, dI, dO, dP, nullptr,
                                                            nullptr, nullptr);
}

// The photon rates in d_rate: as the last sweep's chemistry summed them from
// the incoming rates it read (ssw_sweep::rates_current; 262144 cells x 84
// directions: a sum of its own from the stored rates took 0.10 ms, a pull of
// all 2.46), pulled for the cells that sweep did not solve. Without current
// rates all are pulled, into `out` (at their caller indices with ridx).
int photon_rates(ssw_sweep* s, const Geo& g, double* out, const uint32_t* ridx) {
    const unsigned nb = (unsigned)((s->N + kFluxCells - 1) / kFluxCells);
    const unsigned lanes = (unsigned)(kFluxCells * ((s->D + kFluxDirs - 1) / kFluxDirs));
    const double* missing = nullptr;
    if (s->rates_current) {
        if (!s->rates_partial) return SSW_OK;
        missing = out = s->d_rate;
        ridx = nullptr;
    }
    if (s->fp32)
        k_fluxes<float, false><<<nb, lanes, 0, s->stream>>>(g, make_flux<float>(s), s->lref, nullptr, nullptr, nullptr,
                                                            out, ridx, missing);
    else
        k_fluxes<double, false><<<nb, lanes, 0, s->stream>>>(g, make_flux<double>(s), s->lref, nullptr, nullptr,
                                                             nullptr, out, ridx, missing);
    HIP_TRY(hipGetLastError());
    return SSW_OK;
}

int set_need_all(ssw_sweep* s, uint32_t v) {
    k_fill_u32<<<1, kBlock, 0, s->stream>>>(s->d_need, v, s->p.num_timestep_levels);
    HIP_TRY(hipGetLastError());
    return SSW_OK;
}

// The per-cell {source / D, attenuation} pairs to and from the device, in
// the transport's storage precision there (synchronous).
int upload_sa(ssw_sweep* s, const std::vector<double2>& sa) {
    const size_t n = sa.size();
    if (s->fp32) {
        std::vector<float2> f(n);
        for (size_t c = 0; c < n; c++) f[c] = make_float2((float)sa[c].x, (float)sa[c].y);
        HIP_TRY(hipMemcpyAsync(s->d_sa, f.data(), n * sizeof(float2), hipMemcpyHostToDevice, s->stream));
        HIP_TRY(hipStreamSynchronize(s->stream));
    } else {
        HIP_TRY(hipMemcpyAsync(s->d_sa, sa.data(), n * sizeof(double2), hipMemcpyHostToDevice, s->stream));
        HIP_TRY(hipStreamSynchronize(s->stream));
    }
    return SSW_OK;
}

int download_sa(ssw_sweep* s, std::vector<double2>& sa) {
    const size_t n = sa.size();
    if (s->fp32) {
        std::vector<float2> f(n);
        HIP_TRY(hipMemcpyAsync(f.data(), s->d_sa, n * sizeof(float2), hipMemcpyDeviceToHost, s->stream));
        HIP_TRY(hipStreamSynchronize(s->stream));
        for (size_t c = 0; c < n; c++) sa[c] = make_double2((double)f[c].x, (double)f[c].y);
    } else {
        HIP_TRY(hipMemcpyAsync(sa.data(), s->d_sa, n * sizeof(double2), hipMemcpyDeviceToHost, s->stream));
        HIP_TRY(hipStreamSynchronize(s->stream));
    }
    return SSW_OK;
}

void drop_list(ssw_sweep* s, int lvl) {
    s->epoch++;
    if (lvl >= (int)s->list_ok.size()) return;
    s->list_ok[lvl] = 0;
    s->list_full[lvl] = 0;
    s->replays[lvl] = 0;
    if (s->graphs[lvl]) {
        (void)hipGraphExecDestroy(s->graphs[lvl]);
        s->graphs[lvl] = nullptr;
    }
}

void drop_all_lists(ssw_sweep* s) {
    for (int l = 0; l < (int)s->list_ok.size(); l++) drop_list(s, l);
}

// Kahn layering of the active set {level >= lvl}: every active task's depth
// into d_depth, the number of level sets and, with `starts`, where each of
// them starts in level order. The upwind counters are freed again.
// `expected` active tasks must all be placed, else the graph has a cycle.
int kahn_layering(ssw_sweep* s, int lvl, int64_t expected, uint32_t* d_depth, int* depth_out,
                  std::vector<uint32_t>* starts) {
    const size_t DN = (size_t)s->D * s->N;
    const uint32_t kcap = (uint32_t)std::min<int64_t>(s->N + 1, 1 << 22);
    uint32_t *spill = nullptr, *hist = nullptr;  // hist: totals, then the level sets' tasks
    Defer cleanup{[&] {
        dfree(s, spill);
        dfree(s, hist);
        dfree(s, s->d_cnt);
    }};
    if (!s->d_cnt) TRY(dalloc(s, &s->d_cnt, DN));
    TRY(dalloc(s, &spill, 2 * DN));
    TRY(dalloc(s, &hist, (size_t)kcap + 2));
    const Geo g = make_geo(s);
    k_fill_u32<<<grid_for((int64_t)kcap + 2), kBlock, 0, s->stream>>>(hist, 0u, (int64_t)kcap + 2);
    k_count<<<grid_for((int64_t)DN), kBlock, 0, s->stream>>>(g, lvl);
    if (s->N <= (int64_t)kLayerCells && !s->uneven_faces)
        k_layers<true><<<s->D, 1024, 0, s->stream>>>(g, kcap, d_depth, spill, hist + 2, hist);
    else
        k_layers<false><<<s->D, 1024, 0, s->stream>>>(g, kcap, d_depth, spill, hist + 2, hist);
    HIP_TRY(hipGetLastError());
    uint32_t totals[2] = {0, 0};
    HIP_TRY(hipMemcpyAsync(totals, hist, sizeof(totals), hipMemcpyDeviceToHost, s->stream));
    HIP_TRY(hipStreamSynchronize(s->stream));
    if ((int64_t)totals[0] != expected) {
        if (totals[1] >= kcap) return fail(SSW_ERR_CYCLE, "level-set depth exceeds its bound");
        return fail(SSW_ERR_CYCLE, "dependency cycle: " + std::to_string(expected - (int64_t)totals[0]) +
                                       " cell-direction pairs never become ready");
    }
    *depth_out = (int)std::max(1u, totals[1]);  // no active task: one empty level set
    if (starts) {
        std::vector<uint32_t> h((size_t)*depth_out);
        HIP_TRY(hipMemcpyAsync(h.data(), hist + 2, h.size() * 4, hipMemcpyDeviceToHost, s->stream));
        HIP_TRY(hipStreamSynchronize(s->stream));
        starts->assign(1, 0u);
        for (uint32_t v : h) starts->push_back(starts->back() + v);
    }
    return SSW_OK;
}

// The replay plan of sweep level lvl from its level starts (the full
// schedule's for level 0, the active-set list's otherwise): in the compiled
// replay, each maximal run of at least two consecutive non-empty level sets of
// at most run_block<R>() active tasks (empty level sets inside a run are skipped)
// becomes one single-workgroup launch over a run table entry per level set;
// every other non-empty level set is one launch.
int plan_replay(ssw_sweep* s, int lvl) {
    s->epoch++;  // graphs of packed sweeps captured from the old plan no longer match
    const std::vector<uint32_t>& fs = s->full_start;
    const std::vector<uint32_t>& cs = lvl == 0 ? fs : s->cstart[lvl];
    std::vector<ssw_sweep::ReplayItem>& plan = s->plan[lvl];
    std::vector<uint4>& tab = s->runtab[lvl];
    plan.clear();
    tab.clear();
    if (s->d_dirinfo) {  // direction sweeps: one launch, restricted sweeps included
        plan.push_back({0, s->kmax, 0u, 2});
        dfree(s, s->d_runtab[lvl]);
        return SSW_OK;
    }
    if (!s->groups.empty()) {  // the grouped replay (restricted sweeps: groups with active tasks)
        for (size_t i = 0; i < s->groups.size(); i++)
            if (s->groups[i].ndesc && (lvl == 0 || s->gcount[lvl][i] > 0))
                plan.push_back({s->groups[i].k0, s->groups[i].levels, (uint32_t)i, 1});
        dfree(s, s->d_runtab[lvl]);
        return SSW_OK;
    }
    const bool runs = s->compiled && s->narrow_runs;
    const uint32_t rb = s->fp32 ? (uint32_t)run_block<float>() : (uint32_t)run_block<double>();
    int k = 0;
    while (k < s->kmax) {
        const uint32_t count = cs[k + 1] - cs[k];
        if (count == 0) {
            k++;
            continue;
        }
        if (!runs || count > rb) {
            plan.push_back({k, 0, 0u, 0});
            k++;
            continue;
        }
        const uint32_t t0 = (uint32_t)tab.size();
        int k1 = k;
        for (; k1 < s->kmax && cs[k1 + 1] - cs[k1] <= rb; k1++) {
            const uint32_t c = cs[k1 + 1] - cs[k1];
            if (c) tab.push_back(make_uint4(fs[k1], fs[k1 + 1] - fs[k1], cs[k1], c));
        }
        const int n = (int)(tab.size() - t0);
        if (n >= 2) {
            plan.push_back({k, n, t0, 0});
        } else {
            tab.resize(t0);
            plan.push_back({k, 0, 0u, 0});
        }
        k = k1;
    }
    if (!tab.empty()) {
        TRY(dalloc(s, &s->d_runtab[lvl], tab.size()));
        HIP_TRY(hipMemcpyAsync(s->d_runtab[lvl], tab.data(), tab.size() * sizeof(uint4), hipMemcpyHostToDevice,
                               s->stream));
    } else {
        dfree(s, s->d_runtab[lvl]);
    }
    return SSW_OK;
}

// A kernel of the grouped replay by waves per workgroup and whether it is a
// restricted sweep or has offsets.
#define SSW_CONE_KERNEL(name, R, waves, general)                                       \
    ((waves) == 4 ? ((general) ? name<R, 4, true> : name<R, 4, false>)                 \
     : (waves) == 8 ? ((general) ? name<R, 8, true> : name<R, 8, false>)               \
                    : ((general) ? name<R, 16, true> : name<R, 16, false>))

void free_groups(ssw_sweep* s);

// The grouped replay of full sweeps (compiled replay, group_request >= 2):
// groups of m consecutive level sets; in each group, from its last level set
// down to its first, the level set's tasks in no cone yet become roots, in
// blocks of kGroupT, whose cones are built (k_cone) and compiled into tiles
// (k_cone_tiles). If a cone exceeds the LDS capacity, the task list its bound
// or the tiles the free memory, there are no groups.
template <typename R>
int build_groups_t(ssw_sweep* s, const uint32_t* sorted, uint32_t narrow_group, bool* retry) {
    const int m = s->group_request;
    const size_t DN = (size_t)s->D * s->N;
    const std::vector<uint32_t>& fs = s->full_start;
    const int T = s->group_block;
    const size_t desc_cap = DN / T + (size_t)s->kmax + 1;  // at most ceil(width / T) per level set
    const size_t list_cap = (size_t)ssw::cone_list_cap((int64_t)DN);
    // groups of m level sets, of kMaxGroup where that many consecutive level
    // sets hold at most narrow_group tasks each (the narrow ends of the
    // graph, whose cones stay small); per pass r the level set
    // k0 + levels - 1 - r of each group that has it (pass 0: the last level
    // sets, all tasks roots)
    s->groups.clear();
    int mmax = 0;
    for (int k0 = 0; k0 < s->kmax;) {
        int mk = m;
        if (m < kMaxGroup && k0 + kMaxGroup <= s->kmax) {
            bool narrow = true;
            for (int k = k0; narrow && k < k0 + kMaxGroup; k++) narrow = fs[k + 1] - fs[k] <= narrow_group;
            if (narrow) mk = kMaxGroup;
        }
        const int lv = std::min(s->kmax, k0 + mk) - k0;
        uint32_t widest = 0;
        for (int k = k0; k < k0 + lv; k++) widest = std::max(widest, fs[k + 1] - fs[k]);
        const int waves = ConeShape<R>::waves(T) * (lv > kGroupLevels && widest <= (uint32_t)T * kCus ? 2 : 1);
        s->groups.push_back({k0, lv, 0u, 0u, PassTab{}, 0u, std::min(waves, 16), 0u});
        mmax = std::max(mmax, lv);
        k0 += mk;
    }
    const size_t ng = s->groups.size();
    size_t pass_roots = 1;
    for (int r = 1; r < mmax; r++) {
        size_t w = 0;
        for (const ssw_sweep::Group& gr : s->groups)
            if (gr.levels > r) w += fs[gr.k0 + gr.levels - r] - fs[gr.k0 + gr.levels - 1 - r];
        pass_roots = std::max(pass_roots, w);
    }
    uint8_t *todo = nullptr, *flags = nullptr, *lvlflag = nullptr, *tmp = nullptr;
    uint32_t *roots = nullptr, *ctl = nullptr, *bounds = nullptr, *perm = nullptr;  // ctl: cursor, fail, selected
    uint32_t *list = nullptr, *words = nullptr, *ct = nullptr, *ts = nullptr;
    uint64_t *cu = nullptr, *us = nullptr, *ucnt = nullptr, *uoff = nullptr;
    uint32_t* up = nullptr;
    uint8_t* fars = nullptr;
    int* lv = nullptr;
    uint4 *meta = nullptr, *desc_rm = nullptr, *desc = nullptr;
    Defer cleanup{[&] {
        for (uint8_t** p : {&todo, &flags, &lvlflag, &tmp}) dfree(s, *p);
        for (uint32_t** p : {&roots, &ctl, &bounds, &perm, &list, &words, &ct, &ts}) dfree(s, *p);
        for (uint64_t** p : {&cu, &us, &ucnt, &uoff}) dfree(s, *p);
        dfree(s, up);
        dfree(s, fars);
        dfree(s, lv);
        for (uint4** p : {&meta, &desc_rm, &desc}) dfree(s, *p);
    }};
    const Geo g = make_geo(s);
    // every task's upwind positions
    TRY(dalloc(s, &ucnt, DN + 1));
    TRY(dalloc(s, &uoff, DN + 1));
    k_up_count<<<grid_for((int64_t)DN + 1), kBlock, 0, s->stream>>>(sorted, s->d_nup, (uint32_t)DN, ucnt);
    size_t ub = 0;
    HIP_TRY(hipcub::DeviceScan::ExclusiveSum(nullptr, ub, ucnt, uoff, (int)(DN + 1), s->stream));
    TRY(dalloc(s, &tmp, ub));
    HIP_TRY(hipcub::DeviceScan::ExclusiveSum(tmp, ub, ucnt, uoff, (int)(DN + 1), s->stream));
    uint64_t nup_all = 0;
    HIP_TRY(hipMemcpyAsync(&nup_all, uoff + DN, 8, hipMemcpyDeviceToHost, s->stream));
    HIP_TRY(hipStreamSynchronize(s->stream));
    dfree(s, tmp);
    dfree(s, ucnt);
    TRY(dalloc(s, &up, std::max<size_t>(1, (size_t)nup_all)));
    k_up_fill<<<(unsigned)((s->N + kFluxCells - 1) / kFluxCells),
                kFluxCells * ((s->D + kFluxDirs - 1) / kFluxDirs), 0, s->stream>>>(g, s->d_xpos, uoff, up);
    HIP_TRY(hipGetLastError());
    TRY(dalloc(s, &todo, DN));
    TRY(dalloc(s, &ctl, 3));
    TRY(dalloc(s, &list, list_cap));
    TRY(dalloc(s, &desc_rm, 2 * desc_cap));
    HIP_TRY(hipMemsetAsync(todo, 1, DN, s->stream));
    HIP_TRY(hipMemsetAsync(ctl, 0, 12, s->stream));
    size_t tb = 0;
    if (mmax > 1) {
        TRY(dalloc(s, &flags, DN));
        TRY(dalloc(s, &lvlflag, (size_t)s->kmax));
        TRY(dalloc(s, &roots, pass_roots));
        TRY(dalloc(s, &lv, ng));
        TRY(dalloc(s, &bounds, 2 * ng));
        HIP_TRY(hipcub::DeviceSelect::Flagged(nullptr, tb, hipcub::CountingInputIterator<uint32_t>(0u), flags, roots,
                                              ctl + 2, (int)DN, s->stream));
        TRY(dalloc(s, &tmp, tb));
    }
    // blocks of group g in pass r: [rstart[r][g], rstart[r][g] + rcount[r][g]) of the pass-major descriptors
    std::vector<std::vector<uint32_t>> rstart(mmax, std::vector<uint32_t>(ng, 0u)), rcount(rstart);
    uint32_t ndesc = 0, hctl[2] = {0, 0};
    std::vector<uint4> hmeta;
    std::vector<uint8_t> hflag(s->kmax);
    std::vector<int> hlv;
    std::vector<uint32_t> hb;
    for (int r = 0; r < mmax; r++) {
        hmeta.clear();
        hlv.clear();
        const uint32_t* rl = nullptr;
        if (r > 0) {  // roots: the tasks of the pass's level sets in no cone yet, in position order
            std::fill(hflag.begin(), hflag.end(), 0);
            for (const ssw_sweep::Group& gr : s->groups)
                if (gr.levels > r) {
                    hflag[gr.k0 + gr.levels - 1 - r] = 1;
                    hlv.push_back(gr.k0 + gr.levels - 1 - r);
                }
            if (hlv.empty()) break;
            HIP_TRY(hipMemcpyAsync(lvlflag, hflag.data(), hflag.size(), hipMemcpyHostToDevice, s->stream));
            HIP_TRY(hipMemcpyAsync(lv, hlv.data(), hlv.size() * sizeof(int), hipMemcpyHostToDevice, s->stream));
            k_cone_flags<<<grid_for((int64_t)DN), kBlock, 0, s->stream>>>(s->d_fstart, s->kmax, lvlflag, todo, flags,
                                                                          (uint32_t)DN);
            size_t tbr = tb;
            HIP_TRY(hipcub::DeviceSelect::Flagged(tmp, tbr, hipcub::CountingInputIterator<uint32_t>(0u), flags, roots,
                                                  ctl + 2, (int)DN, s->stream));
            k_cone_bounds<<<grid_for((int64_t)hlv.size()), kBlock, 0, s->stream>>>(roots, ctl + 2, s->d_fstart, lv,
                                                                                    (int)hlv.size(), bounds);
            HIP_TRY(hipGetLastError());
            hb.resize(2 * hlv.size());
            HIP_TRY(hipMemcpyAsync(hb.data(), bounds, hb.size() * 4, hipMemcpyDeviceToHost, s->stream));
            HIP_TRY(hipStreamSynchronize(s->stream));
            rl = roots;
        }
        size_t li = 0;
        for (size_t gi = 0; gi < ng; gi++) {
            const ssw_sweep::Group& gr = s->groups[gi];
            if (gr.levels <= r) continue;
            const int j = gr.k0 + gr.levels - 1 - r;
            uint32_t first, n;
            if (r == 0) {
                first = fs[j];
                n = fs[j + 1] - fs[j];
            } else {
                first = hb[2 * li];
                n = hb[2 * li + 1] - hb[2 * li];
                li++;
            }
            rstart[r][gi] = ndesc + (uint32_t)hmeta.size();
            for (uint32_t b = 0; b < n; b += (uint32_t)T)
                hmeta.push_back(make_uint4((uint32_t)gr.k0, (uint32_t)j, first + b, std::min<uint32_t>(T, n - b)));
            rcount[r][gi] = ndesc + (uint32_t)hmeta.size() - rstart[r][gi];
        }
        if (hmeta.empty()) continue;
        if ((size_t)ndesc + hmeta.size() > desc_cap) return fail(SSW_ERR_HIP, "grouped replay: descriptor bound exceeded");
        TRY(dalloc(s, &meta, hmeta.size()));
        HIP_TRY(hipMemcpyAsync(meta, hmeta.data(), hmeta.size() * sizeof(uint4), hipMemcpyHostToDevice, s->stream));
        const unsigned nb = (unsigned)hmeta.size();
        k_cone<<<nb, kConeThreads, 0, s->stream>>>(uoff, up, s->d_fstart, meta, rl, todo, list, (uint32_t)list_cap, ctl,
                                                   desc_rm + 2 * (size_t)ndesc, ctl + 1);
        HIP_TRY(hipGetLastError());
        HIP_TRY(hipMemcpyAsync(hctl, ctl, 8, hipMemcpyDeviceToHost, s->stream));
        HIP_TRY(hipStreamSynchronize(s->stream));  // meta is reallocated by the next pass
        ndesc += nb;
        if (hctl[1] != 0) break;
    }
    dfree(s, meta);
    dfree(s, tmp);
    dfree(s, bounds);
    dfree(s, lv);
    dfree(s, roots);
    dfree(s, lvlflag);
    dfree(s, flags);
    dfree(s, ctl);
    dfree(s, todo);
    if (hctl[1] != 0) {  // a cone or the list did not fit
        s->groups.clear();
        s->group_fallback = true;
        return SSW_OK;
    }
    // descriptors in group order (a group's workgroups contiguous)
    std::vector<uint32_t> hperm;
    hperm.reserve(ndesc);
    for (size_t gi = 0; gi < ng; gi++) {
        ssw_sweep::Group& gr = s->groups[gi];
        gr.desc0 = (uint32_t)hperm.size();
        gr.passes = PassTab{};
        for (int r = 0; r < mmax; r++) {
            if (rcount[r][gi] == 0) continue;
            gr.passes.off[gr.passes.n++] = (uint32_t)hperm.size() - gr.desc0;
            for (uint32_t k = 0; k < rcount[r][gi]; k++) hperm.push_back(rstart[r][gi] + k);
        }
        gr.ndesc = (uint32_t)hperm.size() - gr.desc0;
        gr.passes.off[gr.passes.n] = gr.ndesc;
    }
    s->group_tasks = hctl[0];
    s->ndesc = ndesc;
    std::vector<uint32_t> gmap(std::max<uint32_t>(1u, ndesc), 0u);
    for (size_t i = 0; i < s->groups.size(); i++)
        for (uint32_t k = 0; k < s->groups[i].ndesc; k++) gmap[s->groups[i].desc0 + k] = (uint32_t)i;
    TRY(dalloc(s, &s->d_gmap, gmap.size()));
    HIP_TRY(hipMemcpyAsync(s->d_gmap, gmap.data(), gmap.size() * 4, hipMemcpyHostToDevice, s->stream));
    TRY(dalloc(s, &s->d_gcount, std::max<size_t>(1, s->groups.size())));
    TRY(dalloc(s, &s->d_gblocks, std::max<size_t>(1, s->groups.size())));
    std::vector<uint32_t> gbase(std::max<size_t>(1, s->groups.size()), 0u);
    for (size_t i = 0; i < s->groups.size(); i++) gbase[i] = s->groups[i].desc0;
    TRY(dalloc(s, &s->d_gbase, gbase.size()));
    HIP_TRY(hipMemcpyAsync(s->d_gbase, gbase.data(), gbase.size() * 4, hipMemcpyHostToDevice, s->stream));
    std::vector<uint32_t> pb;
    s->pbound_start.assign(s->groups.size(), 0u);
    for (size_t i = 0; i < s->groups.size(); i++) {
        const ssw_sweep::Group& gr = s->groups[i];
        s->pbound_start[i] = (uint32_t)pb.size();
        for (int r = 0; r <= gr.passes.n; r++) pb.push_back(gr.desc0 + gr.passes.off[r]);
    }
    if (pb.empty()) pb.push_back(0u);
    TRY(dalloc(s, &s->d_pbound, pb.size()));
    HIP_TRY(hipMemcpyAsync(s->d_pbound, pb.data(), pb.size() * 4, hipMemcpyHostToDevice, s->stream));
    if (s->p.num_timestep_levels > 1) {  // restricted sweeps filter the cones
        s->gf_scan_bytes = 0;
        HIP_TRY(hipcub::DeviceScan::ExclusiveSum(nullptr, s->gf_scan_bytes, s->d_gf_kept, s->d_gf_pos, (int)ndesc + 1,
                                                 s->stream));
        TRY(dalloc(s, &s->d_gf_kept, (size_t)ndesc + 1));
        TRY(dalloc(s, &s->d_gf_pos, (size_t)ndesc + 1));
        TRY(dalloc(s, &s->d_gf_pbval, pb.size()));
        TRY(dalloc(s, &s->d_gf_scan, std::max<size_t>(s->gf_scan_bytes, 1)));
    }
    // cones in group order (a group's workgroups contiguous), counted, placed
    // and written
    TRY(dalloc(s, &desc, 2 * (size_t)ndesc));
    TRY(dalloc(s, &perm, ndesc));
    HIP_TRY(hipMemcpyAsync(perm, hperm.data(), hperm.size() * 4, hipMemcpyHostToDevice, s->stream));
    k_permute_desc<<<grid_for(ndesc), kBlock, 0, s->stream>>>(desc_rm, perm, desc, ndesc);
    std::vector<uint32_t> hw(ng);
    std::vector<uint4> ginfo(ng);
    uint32_t slots = 0;
    for (size_t i = 0; i < ng; i++) {
        ssw_sweep::Group& gr = s->groups[i];
        gr.slot0 = slots;
        slots += gr.ndesc * (uint32_t)gr.waves;
        ginfo[i] = make_uint4((uint32_t)gr.k0, (uint32_t)gr.waves, gr.slot0, gr.desc0);
    }
    TRY(dalloc(s, &s->d_ginfo, ng));
    TRY(dalloc(s, &words, ng));
    HIP_TRY(hipMemcpyAsync(s->d_ginfo, ginfo.data(), ng * sizeof(uint4), hipMemcpyHostToDevice, s->stream));
    k_fill_u32<<<grid_for((int64_t)ng), kBlock, 0, s->stream>>>(words, 0u, (int64_t)ng);
    TRY(dalloc(s, &ct, (size_t)ndesc + 1));
    TRY(dalloc(s, &ts, (size_t)ndesc + 1));
    TRY(dalloc(s, &cu, (size_t)ndesc + 1));
    TRY(dalloc(s, &us, (size_t)ndesc + 1));
    HIP_TRY(hipMemsetAsync(ct + ndesc, 0, 4, s->stream));
    HIP_TRY(hipMemsetAsync(cu + ndesc, 0, 8, s->stream));
    const double inv_aref = 1.0 / s->aref;
    TRY(dalloc(s, &fars, (size_t)hctl[0]));
    k_cone_tiles<R, false><<<ndesc, 64, 0, s->stream>>>(g, inv_aref, sorted, s->d_xpos, uoff, up, s->d_fstart,
                                                        s->d_nup, fars, desc, list, s->d_gmap, s->d_ginfo, ct, cu,
                                                        words, nullptr, nullptr, slots, nullptr, nullptr, nullptr);
    HIP_TRY(hipGetLastError());
    size_t t1 = 0, t2 = 0;
    HIP_TRY(hipcub::DeviceScan::ExclusiveSum(nullptr, t1, ct, ts, (int)ndesc + 1, s->stream));
    HIP_TRY(hipcub::DeviceScan::ExclusiveSum(nullptr, t2, cu, us, (int)ndesc + 1, s->stream));
    TRY(dalloc(s, &tmp, std::max(t1, t2)));
    HIP_TRY(hipcub::DeviceScan::ExclusiveSum(tmp, t1, ct, ts, (int)ndesc + 1, s->stream));
    HIP_TRY(hipcub::DeviceScan::ExclusiveSum(tmp, t2, cu, us, (int)ndesc + 1, s->stream));
    uint32_t more = 0;
    uint64_t units = 0;
    HIP_TRY(hipMemcpyAsync(hw.data(), words, ng * 4, hipMemcpyDeviceToHost, s->stream));
    HIP_TRY(hipMemcpyAsync(&more, ts + ndesc, 4, hipMemcpyDeviceToHost, s->stream));
    HIP_TRY(hipMemcpyAsync(&units, us + ndesc, 8, hipMemcpyDeviceToHost, s->stream));
    HIP_TRY(hipStreamSynchronize(s->stream));
    size_t lds = 0, members = 0;
    for (size_t i = 0; i < ng; i++) {
        s->groups[i].words = hw[i];
        members = std::max<size_t>(members, hw[i]);
        lds = std::max(lds, ConeShape<R>::bytes(s->groups[i].waves, hw[i]));
    }
    if (lds > 65536)  // at most 116 KB (a cone of kConeCap members and 128 roots, FP64)
        for (const bool general : {false, true}) {
            HIP_TRY(hipFuncSetAttribute((const void*)SSW_CONE_KERNEL(k_sweep_cone, R, 16, general),
                                        hipFuncAttributeMaxDynamicSharedMemorySize, 160 << 10));
            HIP_TRY(hipFuncSetAttribute((const void*)SSW_CONE_KERNEL(k_sweep_cone, R, 8, general),
                                        hipFuncAttributeMaxDynamicSharedMemorySize, 160 << 10));
            HIP_TRY(hipFuncSetAttribute((const void*)SSW_CONE_KERNEL(k_sweep_cone_pack, R, 16, general),
                                        hipFuncAttributeMaxDynamicSharedMemorySize, 160 << 10));
            HIP_TRY(hipFuncSetAttribute((const void*)SSW_CONE_KERNEL(k_sweep_cone_pack, R, 8, general),
                                        hipFuncAttributeMaxDynamicSharedMemorySize, 160 << 10));
        }
    dfree(s, tmp);
    dfree(s, desc_rm);
    dfree(s, up);
    dfree(s, uoff);
    dfree(s, cu);
    dfree(s, ct);
    // The tiles of FP32 cones can take more than the per-level replay's planes
    // (measured: up to 35 B more per task, clustered cells x 16 directions). Where
    // they and what the handle still allocates do not fit, that replay runs.
    const int64_t DP = (int64_t)s->D * s->Nper;
    const int64_t later = !s->have_state ? ssw::state_bytes(s->N, (int64_t)DN, DP, sizeof(R))
                          : !s->d_offI   ? ssw::offset_bytes((int64_t)DN, DP, sizeof(R))
                                         : 0;
    const int64_t bytes = 16 * (int64_t)((size_t)units + slots + more) + 4 * (int64_t)ndesc;
    int rc = ssw::cones_fit(bytes, later, expected_free(s)) ? dalloc(s, &s->d_coneblob, (size_t)units) : SSW_ERR_OOM;
    if (rc == SSW_OK) rc = dalloc(s, &s->d_conetiles, (size_t)slots + more);
    if (rc == SSW_OK) rc = dalloc(s, &s->d_conemore, (size_t)ndesc);
    if (rc == SSW_ERR_OOM) {
        free_groups(s);
        s->group_fallback = true;
        *retry = false;
        return SSW_OK;
    }
    TRY(rc);
    k_cone_tiles<R, true><<<ndesc, 256, members * 4, s->stream>>>(
        g, inv_aref, sorted, s->d_xpos, nullptr, nullptr, s->d_fstart, s->d_nup, fars, desc, list, s->d_gmap,
        s->d_ginfo, nullptr, nullptr, words, ts, us, slots, s->d_coneblob, s->d_conetiles, s->d_conemore);
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipStreamSynchronize(s->stream));
    return SSW_OK;
}

// Groups with kNarrowGroup, or, where a cone or the list does not fit, a
// quarter of it (cones of 8 level sets of few directions reach further: 262144
// cells x 16 directions fit with 2048 only, 2.07 ms a frame); if that does not
// fit either, sweeps keep the per-level replay.
// sorted: the tasks in schedule order; s->d_xpos, s->d_fstart and s->d_nup held.
int build_groups(ssw_sweep* s, const uint32_t* sorted) {
    for (uint32_t narrow : {kNarrowGroup, kNarrowGroup / 4}) {
        bool retry = true;
        s->group_fallback = false;
        TRY(s->fp32 ? build_groups_t<float>(s, sorted, narrow, &retry)
                    : build_groups_t<double>(s, sorted, narrow, &retry));
        if (!s->group_fallback || !retry) break;
    }
    return SSW_OK;
}

void free_groups(ssw_sweep* s) {
    s->groups.clear();
    s->group_tasks = 0;
    s->group_fallback = false;
    for (uint4** p : {&s->d_coneblob, &s->d_conetiles, &s->d_ginfo}) dfree(s, *p);
    for (uint32_t** p : {&s->d_conemore, &s->d_gmap, &s->d_gcount, &s->d_gbase, &s->d_gblocks, &s->d_pbound, &s->d_gf_kept,
                         &s->d_gf_pos, &s->d_gf_pbval})
        dfree(s, *p);
    dfree(s, s->d_gf_scan);
    s->gf_scan_bytes = 0;
    for (uint32_t*& p : s->d_gsel_l) dfree(s, p);
}

// The direction sweeps' schedule from every task's depth and upwind count:
// tasks sorted by (direction, level set, class, cell), groups of 64 of a level
// set, their tiles counted, placed and written. Takes d_depth (freed as soon as
// it is no longer needed).
template <typename R>
int build_dir_schedule_t(ssw_sweep* s, uint32_t*& d_depth) {
    using S = DirShape<R>;
    const size_t DN = (size_t)s->D * s->N, KD = (size_t)s->kmax * s->D;
    const uint32_t N = (uint32_t)s->N, D = (uint32_t)s->D, kmax = (uint32_t)s->kmax;
    uint32_t *key = nullptr, *key2 = nullptr, *val = nullptr, *val2 = nullptr, *sorted = nullptr, *start = nullptr,
             *first = nullptr, *gt = nullptr, *ts = nullptr, *at = nullptr, *tf = nullptr;
    uint64_t *gu = nullptr, *us = nullptr;
    uint8_t *tmp = nullptr, *nfar = nullptr;
    uint4* groups = nullptr;
    Defer cleanup{[&] {
        for (uint32_t** p : {&key, &key2, &val, &val2, &sorted, &start, &first, &gt, &ts, &at, &tf}) dfree(s, *p);
        dfree(s, gu);
        dfree(s, us);
        dfree(s, tmp);
        dfree(s, nfar);
        dfree(s, groups);
        dfree(s, s->d_nup);
    }};
    Geo g = make_geo(s);
    for (uint32_t** p : {&key, &key2, &val, &val2}) TRY(dalloc(s, p, DN));
    k_dir_keys<<<grid_for((int64_t)DN), kBlock, 0, s->stream>>>(d_depth, s->d_nup, N, kmax, (uint32_t)DN, key, val);
    int bits = 3;  // keys below D * kmax * 8 < 2^32 (kmax <= 2^22 + 1, D <= 127)
    while (bits < 32 && (KD >> (bits - 3))) bits++;
    hipcub::DoubleBuffer<uint32_t> kb(key, key2), vb(val, val2);
    size_t tb = 0;
    HIP_TRY(hipcub::DeviceRadixSort::SortPairs(nullptr, tb, kb, vb, (int)DN, 0, bits, s->stream));
    TRY(dalloc(s, &tmp, tb));
    HIP_TRY(hipcub::DeviceRadixSort::SortPairs(tmp, tb, kb, vb, (int)DN, 0, bits, s->stream));
    TRY(dalloc(s, &start, KD));
    TRY(dalloc(s, &s->d_xpos, DN));
    k_fill_u32<<<grid_for((int64_t)KD), kBlock, 0, s->stream>>>(start, kNone, (int64_t)KD);
    TRY(dalloc(s, &s->d_dircell, DN));
    k_dir_starts<<<grid_for((int64_t)DN), kBlock, 0, s->stream>>>(kb.Current(), vb.Current(), (uint32_t)DN, N, start,
                                                                  s->d_xpos, s->d_dircell);
    HIP_TRY(hipGetLastError());
    std::vector<uint32_t> hs(KD);
    HIP_TRY(hipMemcpyAsync(hs.data(), start, KD * 4, hipMemcpyDeviceToHost, s->stream));
    HIP_TRY(hipStreamSynchronize(s->stream));
    sorted = vb.Current();  // owned by exactly one pointer
    if (sorted == val) val = nullptr;
    else val2 = nullptr;
    dfree(s, tmp);
    for (uint32_t** p : {&key, &key2, &val, &val2}) dfree(s, *p);
    // level sets and widest level set of every direction, and the first group
    // of every (direction, level set)
    std::vector<uint32_t> hf(KD), at0(D + 1);
    std::vector<uint4> info(D);
    uint32_t ng = 0;
    for (uint32_t d = 0; d < D; d++) {
        at0[d] = ng;
        uint32_t k = 0, widest = 0;
        for (; k < kmax && hs[(size_t)d * kmax + k] != kNone; k++) {
            const uint32_t b = hs[(size_t)d * kmax + k];
            const uint32_t e = k + 1 < kmax && hs[(size_t)d * kmax + k + 1] != kNone ? hs[(size_t)d * kmax + k + 1]
                                                                                     : (d + 1) * N;
            if (e <= b) return fail(SSW_ERR_HIP, "direction sweeps: level set starts out of order");
            widest = std::max(widest, e - b);
            hf[(size_t)d * kmax + k] = ng;
            ng += (e - b + 63) / 64;
        }
        for (uint32_t j = k; j < kmax; j++)
            if (hs[(size_t)d * kmax + j] != kNone) return fail(SSW_ERR_HIP, "direction sweeps: a direction skips a level set");
        info[d] = make_uint4(0, 0, k, widest > S::kRing / 4 ? 1u : 0u);
    }
    at0[D] = ng;
    TRY(dalloc(s, &first, KD));
    TRY(dalloc(s, &groups, ng));
    HIP_TRY(hipMemcpyAsync(first, hf.data(), KD * 4, hipMemcpyHostToDevice, s->stream));
    k_dir_groups<<<grid_for((int64_t)KD), kBlock, 0, s->stream>>>(start, first, N, D, kmax, groups);
    TRY(dalloc(s, &nfar, DN));
    const unsigned nb = (unsigned)((s->N + kFluxCells - 1) / kFluxCells);
    k_dir_far<R><<<nb, kFluxCells * ((D + kFluxDirs - 1) / kFluxDirs), 0, s->stream>>>(g, s->d_xpos, d_depth, start,
                                                                                      kmax, nfar);
    TRY(dalloc(s, &gt, (size_t)ng + 1));
    TRY(dalloc(s, &ts, (size_t)ng + 1));
    TRY(dalloc(s, &gu, (size_t)ng + 1));
    TRY(dalloc(s, &us, (size_t)ng + 1));
    HIP_TRY(hipMemsetAsync(gt + ng, 0, 4, s->stream));
    HIP_TRY(hipMemsetAsync(gu + ng, 0, 8, s->stream));
    const unsigned gb = (unsigned)((ng + kBlock / 64 - 1) / (kBlock / 64));
    k_dir_tile_count<R><<<gb, kBlock, 0, s->stream>>>(groups, ng, sorted, s->d_nup, nfar, gt, gu);
    HIP_TRY(hipGetLastError());
    size_t t1 = 0, t2 = 0;
    HIP_TRY(hipcub::DeviceScan::ExclusiveSum(nullptr, t1, gt, ts, (int)ng + 1, s->stream));
    HIP_TRY(hipcub::DeviceScan::ExclusiveSum(nullptr, t2, gu, us, (int)ng + 1, s->stream));
    TRY(dalloc(s, &tmp, std::max(t1, t2)));
    HIP_TRY(hipcub::DeviceScan::ExclusiveSum(tmp, t1, gt, ts, (int)ng + 1, s->stream));
    HIP_TRY(hipcub::DeviceScan::ExclusiveSum(tmp, t2, gu, us, (int)ng + 1, s->stream));
    TRY(dalloc(s, &at, (size_t)D + 1));
    TRY(dalloc(s, &tf, (size_t)D + 1));
    HIP_TRY(hipMemcpyAsync(at, at0.data(), ((size_t)D + 1) * 4, hipMemcpyHostToDevice, s->stream));
    k_gather_u32<<<grid_for(D + 1), kBlock, 0, s->stream>>>(ts, at, tf, D + 1);
    HIP_TRY(hipGetLastError());
    std::vector<uint32_t> htf(D + 1);
    uint64_t units = 0;
    HIP_TRY(hipMemcpyAsync(htf.data(), tf, ((size_t)D + 1) * 4, hipMemcpyDeviceToHost, s->stream));
    HIP_TRY(hipMemcpyAsync(&units, us + ng, 8, hipMemcpyDeviceToHost, s->stream));
    HIP_TRY(hipStreamSynchronize(s->stream));
    for (uint32_t d = 0; d < D; d++) {
        info[d].x = htf[d];
        info[d].y = htf[d + 1] - htf[d];
    }
    dfree(s, d_depth);
    dfree(s, tmp);
    TRY(dalloc(s, (uint8_t**)&s->d_dirsa, DN * sizeof(SA<R>)));
    if (s->p.num_timestep_levels > 1) TRY(dalloc(s, &s->d_dirlev, DN));
    TRY(dalloc(s, &s->d_dirblob, (size_t)units));
    TRY(dalloc(s, &s->d_dirtiles, 2 * (size_t)htf[D]));
    TRY(dalloc(s, &s->d_dirinfo, (size_t)D));
    HIP_TRY(hipMemcpyAsync(s->d_dirinfo, info.data(), D * sizeof(uint4), hipMemcpyHostToDevice, s->stream));
    k_dir_tile_fill<R><<<gb, kBlock, 0, s->stream>>>(g, 1.0 / s->aref, groups, ng, sorted, s->d_nup, nfar, s->d_xpos, ts,
                                                     us, tf, s->d_dirblob, s->d_dirtiles);
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipStreamSynchronize(s->stream));
    return SSW_OK;
}

int init_replay(ssw_sweep* s);
int setup_overflow(ssw_sweep* s);
void free_schedule(ssw_sweep* s);

// The full schedule, once per grid: Kahn layering of the whole graph, each
// task's depth, a stable sort by depth of the tasks in (direction, cell)
// order, then the compiled or geometric per-task data in that order, and the
// chunk table of the compaction. A graph with a cycle leaves the schedule that
// was there as it is (have_schedule); from then on it is replaced.
int build_schedule(ssw_sweep* s) {
    const size_t DN = (size_t)s->D * s->N;
    // sort the tasks by depth, stable over t = d*N + c (double-buffered: four
    // DN-word arrays and a small temporary)
    uint32_t *d_depth = nullptr, *d_keys = nullptr, *d_vals = nullptr, *d_vals2 = nullptr, *d_sorted = nullptr;
    uint8_t* d_tmp = nullptr;
    Defer cleanup{[&] {
        for (uint32_t** p : {&d_depth, &d_keys, &d_vals, &d_vals2, &d_sorted}) dfree(s, *p);
        dfree(s, d_tmp);
    }};
    TRY(dalloc(s, &d_depth, DN));
    int depth = 0;
    std::vector<uint32_t> starts;
    TRY(kahn_layering(s, 0, (int64_t)DN, d_depth, &depth, &starts));
    free_schedule(s);
    s->kmax = depth;
    s->full_start = std::move(starts);
    Geo g = make_geo(s);
    if (s->compiled && s->dir_sweeps && !s->uneven_faces) {
        TRY(s->fp32 ? build_dir_schedule_t<float>(s, d_depth) : build_dir_schedule_t<double>(s, d_depth));
        return init_replay(s);
    }
    TRY(dalloc(s, &d_keys, DN));
    TRY(dalloc(s, &d_vals, DN));
    TRY(dalloc(s, &d_vals2, DN));
    k_iota<<<grid_for((int64_t)DN), kBlock, 0, s->stream>>>(d_vals, (uint32_t)DN);
    HIP_TRY(hipGetLastError());
    int bits = 1;
    while ((1ll << bits) <= s->kmax) bits++;
    hipcub::DoubleBuffer<uint32_t> kb(d_depth, d_keys), vb(d_vals, d_vals2);
    size_t tmp_bytes = 0;
    HIP_TRY(hipcub::DeviceRadixSort::SortPairs(nullptr, tmp_bytes, kb, vb, (int)DN, 0, bits, s->stream));
    TRY(dalloc(s, &d_tmp, tmp_bytes));
    HIP_TRY(hipcub::DeviceRadixSort::SortPairs(d_tmp, tmp_bytes, kb, vb, (int)DN, 0, bits, s->stream));
    HIP_TRY(hipStreamSynchronize(s->stream));
    // the sorted order moves to d_sorted: the buffer it is stays owned by
    // exactly one pointer, so that it is freed once
    d_sorted = vb.Current();
    if (d_sorted == d_vals) d_vals = nullptr;
    else d_vals2 = nullptr;
    dfree(s, d_tmp);
    dfree(s, d_keys);
    dfree(s, d_depth);
    dfree(s, d_vals);
    dfree(s, d_vals2);
    TRY(dalloc(s, &s->d_fstart, s->full_start.size()));
    HIP_TRY(hipMemcpyAsync(s->d_fstart, s->full_start.data(), s->full_start.size() * 4, hipMemcpyHostToDevice,
                           s->stream));
    const double inv_aref = 1.0 / s->aref;
    if (s->compiled) {
        TRY(dalloc(s, &s->d_xpos, DN));
        k_invert<<<grid_for((int64_t)DN), kBlock, 0, s->stream>>>(d_sorted, s->d_xpos, (uint32_t)DN);
        HIP_TRY(hipGetLastError());
        if (s->uneven_faces) {
            dfree(s, s->d_nup);
            s->group_fallback = s->group_request >= 2;
        } else if (s->group_request >= 2) {
            TRY(build_groups(s, d_sorted));
            dfree(s, s->d_nup);
            if (!s->groups.empty()) return init_replay(s);
        }
        TRY(setup_overflow(s));
        TRY(dalloc(s, &s->d_hdr, DN));
        TRY(dalloc(s, (uint8_t**)&s->d_A, DN * real_size(s)));
        TRY(dalloc(s, (uint8_t**)&s->d_planes, (size_t)kPlanes * DN * entry_size(s)));
        if (s->fp32)
            k_schedule<float><<<grid_for((int64_t)DN), kBlock, 0, s->stream>>>(
                g, inv_aref, d_sorted, s->d_fstart, s->kmax, 1, s->d_xpos, s->d_ovf_start, s->d_hdr,
                (float*)s->d_A, (Entry<float>*)s->d_planes, (Entry<float>*)s->d_ovf, nullptr);
        else
            k_schedule<double><<<grid_for((int64_t)DN), kBlock, 0, s->stream>>>(
                g, inv_aref, d_sorted, s->d_fstart, s->kmax, 1, s->d_xpos, s->d_ovf_start, s->d_hdr,
                (double*)s->d_A, (Entry<double>*)s->d_planes, (Entry<double>*)s->d_ovf, nullptr);
    } else {
        TRY(dalloc(s, &s->d_recs, DN));
        k_schedule<double><<<grid_for((int64_t)DN), kBlock, 0, s->stream>>>(
            g, inv_aref, d_sorted, s->d_fstart, s->kmax, 0, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr,
            s->d_recs);
    }
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipStreamSynchronize(s->stream));
    dfree(s, d_sorted);
    dfree(s, s->d_ovf_start);  // copied into the headers
    // chunk table: chunks of at most kChunk tasks inside one level set
    std::vector<uint4> chunks;
    std::vector<uint32_t> first(s->kmax);
    for (int k = 0; k < s->kmax; k++) {
        first[k] = (uint32_t)chunks.size();
        const uint32_t b = s->full_start[k], e = s->full_start[k + 1];
        if (b == e) chunks.push_back(make_uint4((uint32_t)k, b, e, 0u));
        for (uint32_t p = b; p < e; p += kChunk)
            chunks.push_back(make_uint4((uint32_t)k, p, std::min(e, p + (uint32_t)kChunk), 0u));
    }
    s->nchunks = (uint32_t)chunks.size();
    TRY(dalloc(s, &s->d_chunks, chunks.size()));
    TRY(dalloc(s, &s->d_first_chunk, first.size()));
    TRY(dalloc(s, &s->d_ccount, chunks.size()));
    TRY(dalloc(s, &s->d_coff, chunks.size()));
    TRY(dalloc(s, &s->d_cstart, (size_t)s->kmax + 1));
    HIP_TRY(hipMemcpyAsync(s->d_chunks, chunks.data(), chunks.size() * sizeof(uint4), hipMemcpyHostToDevice,
                           s->stream));
    HIP_TRY(hipMemcpyAsync(s->d_first_chunk, first.data(), first.size() * 4, hipMemcpyHostToDevice, s->stream));
    s->scan_tmp_bytes = 0;
    HIP_TRY(hipcub::DeviceScan::ExclusiveSum(nullptr, s->scan_tmp_bytes, s->d_ccount, s->d_coff, (int)s->nchunks,
                                             s->stream));
    TRY(dalloc(s, (uint8_t**)&s->d_scan_tmp, s->scan_tmp_bytes));
    HIP_TRY(hipStreamSynchronize(s->stream));
    return init_replay(s);
}

// Empty active-set lists, plans and graphs, and the full sweep's plan.
int init_replay(ssw_sweep* s) {
    const int L = s->p.num_timestep_levels;
    for (uint32_t*& p : s->d_idx) dfree(s, p);
    s->d_idx.assign(L, nullptr);
    s->cstart.assign(L, std::vector<uint32_t>());
    s->list_ok.assign(L, 0);
    s->list_full.assign(L, 0);
    s->replays.assign(L, 0);
    for (hipGraphExec_t ge : s->graphs)
        if (ge) (void)hipGraphExecDestroy(ge);
    s->graphs.assign(L, nullptr);
    for (uint4*& p : s->d_runtab) dfree(s, p);
    s->d_runtab.assign(L, nullptr);
    for (uint32_t*& p : s->d_gsel_l) dfree(s, p);
    s->d_gsel_l.assign(L, nullptr);
    s->gcount.assign(L, std::vector<uint32_t>());
    s->gblocks.assign(L, std::vector<uint32_t>());
    s->runtab.assign(L, std::vector<uint4>());
    s->plan.assign(L, std::vector<ssw_sweep::ReplayItem>());
    TRY(plan_replay(s, 0));
    s->have_schedule = true;
    return SSW_OK;
}

const uint4* schedule_tasks(ssw_sweep* s) { return s->compiled ? s->d_hdr : s->d_recs; }

// The active-set list of sweep level lvl >= 1: the positions of the full
// schedule whose cell has level >= lvl, per level set, and its level starts
// on the host. Sweep level 0 covers every task and needs no list.
int make_group_list(ssw_sweep* s, int lvl) {
    if (!s->d_gsel_l[lvl]) TRY(dalloc(s, &s->d_gsel_l[lvl], std::max<uint32_t>(1u, s->ndesc)));
    const size_t ng = std::max<size_t>(1, s->groups.size());
    HIP_TRY(hipMemsetAsync(s->d_gcount, 0, ng * 4, s->stream));
    HIP_TRY(hipMemsetAsync(s->d_gblocks, 0, ng * 4, s->stream));
    Geo g = make_geo(s);
    const uint32_t nd = s->ndesc;
    const size_t npb = std::max<size_t>(1, s->pbound_start.empty() ? 1 : (size_t)s->pbound_start.back() +
                                                                          s->groups.back().passes.n + 1);
    std::vector<uint32_t> pbv(npb, 0u);
    if (nd) {
        // the cones with active tasks, packed in order (scratch held since the
        // cone build)
        uint32_t *kept = s->d_gf_kept, *pos = s->d_gf_pos, *pbval = s->d_gf_pbval;
        uint8_t* scan_tmp = s->d_gf_scan;
        size_t tb = s->gf_scan_bytes;
        if (!kept || !pos || !pbval || !scan_tmp)
            return fail(SSW_ERR_INVALID, "grouped replay: restricted-sweep scratch missing");
        k_fill_u32<<<1, 1, 0, s->stream>>>(kept + nd, 0u, 1);
        k_cone_active<<<nd, 64, 0, s->stream>>>(g, lvl, s->d_coneblob, s->d_conetiles, s->d_conemore,
                                                s->d_ginfo, s->d_gmap, kept, s->d_gcount, s->d_gblocks);
        HIP_TRY(hipGetLastError());
        HIP_TRY(hipcub::DeviceScan::ExclusiveSum(scan_tmp, tb, kept, pos, (int)nd + 1, s->stream));
        k_place_cone<<<grid_for(nd), kBlock, 0, s->stream>>>(kept, pos, s->d_gmap, s->d_gbase, s->d_gsel_l[lvl], nd);
        k_gather_u32<<<grid_for((int64_t)npb), kBlock, 0, s->stream>>>(pos, s->d_pbound, pbval, (uint32_t)npb);
        HIP_TRY(hipGetLastError());
        HIP_TRY(hipMemcpyAsync(pbv.data(), pbval, npb * 4, hipMemcpyDeviceToHost, s->stream));
        HIP_TRY(hipStreamSynchronize(s->stream));
    }
    std::vector<uint32_t>& gc = s->gcount[lvl];
    gc.assign(ng, 0u);
    HIP_TRY(hipMemcpyAsync(gc.data(), s->d_gcount, ng * 4, hipMemcpyDeviceToHost, s->stream));
    std::vector<uint32_t>& gb = s->gblocks[lvl];
    gb.assign(ng, 0u);
    HIP_TRY(hipMemcpyAsync(gb.data(), s->d_gblocks, ng * 4, hipMemcpyDeviceToHost, s->stream));
    HIP_TRY(hipStreamSynchronize(s->stream));
    // pass ranges of each group's kept cones
    if ((int)s->gpass_l.size() <= lvl) s->gpass_l.resize(lvl + 1);
    s->gpass_l[lvl].assign(s->groups.size(), PassTab{});
    for (size_t i = 0; i < s->groups.size(); i++) {
        const ssw_sweep::Group& gr = s->groups[i];
        PassTab& pt = s->gpass_l[lvl][i];
        pt.n = gr.passes.n;
        const uint32_t b = pbv[s->pbound_start[i]];
        for (int r = 0; r <= gr.passes.n; r++) pt.off[r] = pbv[s->pbound_start[i] + r] - b;
    }
    int64_t kept = 0;
    for (uint32_t v : gc) kept += v;
    // every task active: the full sweep's launches are used
    s->list_full[lvl] = (kept == s->group_tasks) ? 1 : 0;
    s->list_ok[lvl] = 1;
    s->replays[lvl] = 0;
    s->epoch++;
    if (s->graphs[lvl]) {
        (void)hipGraphExecDestroy(s->graphs[lvl]);
        s->graphs[lvl] = nullptr;
    }
    TRY(plan_replay(s, lvl));
    return SSW_OK;
}

int make_list(ssw_sweep* s, int lvl) {
    if (s->d_dirinfo) {  // direction sweeps pass every task and test its level: no list
        uint32_t* d_min = nullptr;
        Defer free_min{[&] { dfree(s, d_min); }};
        TRY(dalloc(s, &d_min, 1));
        k_fill_u32<<<1, 1, 0, s->stream>>>(d_min, 255u, 1);
        k_min_level<<<std::min<unsigned>(grid_for(s->N), 1024u), kBlock, 0, s->stream>>>(s->d_level, s->N, d_min);
        HIP_TRY(hipGetLastError());
        uint32_t mn = 0;
        HIP_TRY(hipMemcpyAsync(&mn, d_min, 4, hipMemcpyDeviceToHost, s->stream));
        HIP_TRY(hipStreamSynchronize(s->stream));
        s->list_full[lvl] = mn >= (uint32_t)lvl ? 1 : 0;  // every cell active: a full sweep
        s->list_ok[lvl] = 1;
        s->replays[lvl] = 0;
        s->epoch++;
        if (s->graphs[lvl]) {
            (void)hipGraphExecDestroy(s->graphs[lvl]);
            s->graphs[lvl] = nullptr;
        }
        return plan_replay(s, lvl);
    }
    if (!s->groups.empty()) return make_group_list(s, lvl);
    const size_t DN = (size_t)s->D * s->N;
    if (!s->d_idx[lvl]) TRY(dalloc(s, &s->d_idx[lvl], DN));
    Geo g = make_geo(s);
    const uint4* tasks = schedule_tasks(s);
    k_compact_count<<<s->nchunks, kBlock, 0, s->stream>>>(g, tasks, s->d_chunks, s->nchunks, lvl, s->d_ccount);
    HIP_TRY(hipGetLastError());
    size_t tb = s->scan_tmp_bytes;
    HIP_TRY(hipcub::DeviceScan::ExclusiveSum(s->d_scan_tmp, tb, s->d_ccount, s->d_coff, (int)s->nchunks, s->stream));
    k_compact_write<<<s->nchunks, kBlock, 0, s->stream>>>(g, tasks, s->d_chunks, s->nchunks, s->d_fstart, lvl,
                                                          s->d_coff, s->d_idx[lvl]);
    HIP_TRY(hipGetLastError());
    // total = offset + count of the last chunk
    uint32_t last[2] = {0, 0};
    HIP_TRY(hipMemcpyAsync(&last[0], s->d_coff + s->nchunks - 1, 4, hipMemcpyDeviceToHost, s->stream));
    HIP_TRY(hipMemcpyAsync(&last[1], s->d_ccount + s->nchunks - 1, 4, hipMemcpyDeviceToHost, s->stream));
    HIP_TRY(hipStreamSynchronize(s->stream));
    k_compact_starts<<<grid_for((int64_t)s->kmax + 1), kBlock, 0, s->stream>>>(s->d_first_chunk, s->d_coff, s->kmax,
                                                                               last[0] + last[1], s->d_cstart);
    HIP_TRY(hipGetLastError());
    std::vector<uint32_t>& cs = s->cstart[lvl];
    cs.resize(s->kmax + 1);
    HIP_TRY(hipMemcpyAsync(cs.data(), s->d_cstart, (s->kmax + 1) * 4, hipMemcpyDeviceToHost, s->stream));
    HIP_TRY(hipStreamSynchronize(s->stream));
    TRY(plan_replay(s, lvl));
    s->list_ok[lvl] = 1;
    s->replays[lvl] = 0;
    s->epoch++;
    if (s->graphs[lvl]) {
        (void)hipGraphExecDestroy(s->graphs[lvl]);
        s->graphs[lvl] = nullptr;
    }
    return SSW_OK;
}

template <typename R, typename... Args>
void launch_cones(int waves, bool general, uint32_t blocks, uint32_t words, hipStream_t st, Args... args) {
    hipLaunchKernelGGL(SSW_CONE_KERNEL(k_sweep_cone, R, waves, general), dim3(blocks), dim3(64 * waves),
                       ConeShape<R>::bytes(waves, words), st, args...);
}

// Launches one item of sweep level lvl's replay plan on stream st: a group
// of level sets (its cones one workgroup each), a run of narrow level sets
// (one workgroup), or one level set.
template <typename R>
void launch_item_t(ssw_sweep* s, const Geo& g, const Flux<R>& fl, int lvl, const ssw_sweep::ReplayItem& it,
                   hipStream_t st) {
    const std::vector<uint32_t>& fs = s->full_start;
    const bool all = lvl == 0 || s->list_full[lvl];
    const uint32_t* idx = all ? nullptr : s->d_idx[lvl];
    const Entry<R>* ovf = (const Entry<R>*)s->d_ovf;
    if (it.group == 2) {  // direction sweeps: one workgroup per direction
        constexpr int lanes = 64 * DirShape<R>::kWaves;
        const int at = all ? 0 : lvl;
        const uint32_t DN = (uint32_t)(s->D * s->N);
        SA<R>* sas = (SA<R>*)s->d_dirsa;
        k_dir_inputs<R><<<grid_for(DN), kBlock, 0, st>>>(s->d_dircell, fl.sa, g.level, sas, at ? s->d_dirlev : nullptr,
                                                         DN);
        if (at == 0 && !fl.offI)
            k_sweep_dir<R, false><<<s->D, lanes, 0, st>>>(g, fl, s->d_dirblob, s->d_dirtiles, s->d_dirinfo, sas,
                                                          s->d_dirlev, 0);
        else
            k_sweep_dir<R, true><<<s->D, lanes, 0, st>>>(g, fl, s->d_dirblob, s->d_dirtiles, s->d_dirinfo, sas,
                                                         s->d_dirlev, at);
        return;
    }
    if (it.group) {
        const ssw_sweep::Group& gr = s->groups[it.tab];
        launch_cones<R>(gr.waves, !all || fl.offI != nullptr, all ? gr.ndesc : s->gblocks[lvl][it.tab], gr.words,
                        st, g, fl, s->d_coneblob, s->d_conetiles, s->d_conemore,
                        all ? nullptr : s->d_gsel_l[lvl] + gr.desc0, gr.slot0, gr.desc0, gr.words, all ? 0 : lvl,
                        all ? gr.passes : s->gpass_l[lvl][it.tab]);
        return;
    }
    if (it.levels > 0) {  // a run of narrow level sets, one workgroup
        k_sweep_comp_run<R><<<1, run_block<R>(), 0, st>>>(g, fl, s->d_hdr, (const R*)s->d_A,
                                                          (const Entry<R>*)s->d_planes, ovf, idx,
                                                          s->d_runtab[lvl] + it.tab, it.levels);
        return;
    }
    const std::vector<uint32_t>& cs = all ? fs : s->cstart[lvl];
    const int k = it.k;
    const uint32_t count = cs[k + 1] - cs[k];
    const uint32_t b = fs[k], W = fs[k + 1] - fs[k];
    const uint32_t* ik = idx ? idx + cs[k] : nullptr;
    if (s->compiled) {
        const uint4* hdr = s->d_hdr + b;
        const R* A = (const R*)s->d_A + b;
        const Entry<R>* planes = (const Entry<R>*)s->d_planes + (size_t)kPlanes * b;
        switch (s->rec_block) {
            case 128:
                k_sweep_comp<R, 128><<<(count + 127) / 128, 128, 0, st>>>(g, fl, hdr, A, planes, ovf, b, W, ik, count);
                break;
            case 256:
                k_sweep_comp<R, 256><<<(count + 255) / 256, 256, 0, st>>>(g, fl, hdr, A, planes, ovf, b, W, ik, count);
                break;
            default:
                k_sweep_comp<R, 64><<<(count + 63) / 64, 64, 0, st>>>(g, fl, hdr, A, planes, ovf, b, W, ik, count);
        }
    } else {
        k_sweep_rec<R><<<(count + kTasksPerBlock - 1) / kTasksPerBlock, kBlock, 0, st>>>(g, fl, s->d_recs + b, ik,
                                                                                        count);
    }
}

// Launches the replay of sweep level lvl's level sets on the handle's stream,
// one exact-size launch per plan item; with `ev` each launch is bracketed by
// events.
template <typename R>
void launch_replay_t(ssw_sweep* s, const Geo& g, int lvl, std::vector<std::pair<hipEvent_t, hipEvent_t>>* ev,
                     const std::function<hipEvent_t()>* mark) {
    const Flux<R> fl = make_flux<R>(s);
    for (const ssw_sweep::ReplayItem& it : s->plan[lvl]) {
        hipEvent_t a = ev ? (*mark)() : nullptr;
        launch_item_t<R>(s, g, fl, lvl, it, s->stream);
        if (ev) ev->push_back({a, (*mark)()});
    }
}

void launch_replay(ssw_sweep* s, const Geo& g, int lvl, std::vector<std::pair<hipEvent_t, hipEvent_t>>* ev,
                   const std::function<hipEvent_t()>* mark = nullptr) {
    if (s->fp32) launch_replay_t<float>(s, g, lvl, ev, mark);
    else launch_replay_t<double>(s, g, lvl, ev, mark);
}

// Captures the replay of sweep level lvl as one graph (nothing is executed). A
// failed capture leaves no graph; the level sets are then launched one by one
// (counted in ssw_info).
void capture(ssw_sweep* s, const Geo& g, int lvl) {
    hipGraph_t graph = nullptr;
    std::unique_lock<std::shared_mutex> lock(g_capture_mu);
    if (hipStreamBeginCapture(s->stream, hipStreamCaptureModeRelaxed) != hipSuccess) {
        (void)hipGetLastError();
        s->capture_failures++;
        return;
    }
    launch_replay(s, g, lvl, nullptr);
    hipError_t ce = hipStreamEndCapture(s->stream, &graph);
    lock.unlock();
    if (ce != hipSuccess || !graph) {
        if (graph) (void)hipGraphDestroy(graph);
        (void)hipGetLastError();
        s->capture_failures++;
        return;
    }
    hipGraphExec_t ge = nullptr;
    hipError_t ie = hipGraphInstantiate(&ge, graph, nullptr, nullptr, 0);
    (void)hipGraphDestroy(graph);
    if (ie != hipSuccess) {
        (void)hipGetLastError();
        s->capture_failures++;
        return;
    }
    s->graphs[lvl] = ge;
}

ChemArgs chem_args(ssw_sweep* s) {
    ChemArgs ca;
    ca.rho = s->d_rho;
    ca.x = s->d_x;
    ca.T = s->d_T;
    ca.src = s->d_src;
    ca.sa = s->d_sa;
    ca.species_ts = s->d_sts;
    ca.prev_rate = s->d_prev;
    ca.photon = s->d_rate;
    ca.change_ts = s->d_change;
    ca.vol = s->d_vol;
    ca.size = s->d_size;
    ca.max_ts = s->p.max_timestep;
    ca.thr = s->p.significant_rate_threshold;
    ca.safety = s->p.chemistry_timestep_safety_factor;
    ca.scale_factor = s->p.scale_factor;
    ca.prevent_cooling = s->p.prevent_cooling;
    ca.lref = s->lref;
    ca.failures = s->d_fail;
    ca.active = s->d_active;
    ca.limiting = s->d_active + 1;
    ca.queue = s->d_chemq;
    return ca;
}

// The periodic sources and the chemistry of n handles (at most kChemJobs) after
// their sweeps. The tail gets a wave per 4 cells, so that a queue of all of them
// has four quads a cell, at most two per SIMD (its quads then take further cells
// as they finish); waves that find no queued cell end at once.
template <typename R, int kJobs>
void launch_chemistry(const ChemJob<R>* j, int n, hipStream_t st) {
    ChemJobs<R, kJobs> a;
    int64_t pw = 0, cells = 0;
    for (int k = 0; k < n; k++) {
        a.job[k] = j[k];
        const Geo& g = j[k].g;
        pw = std::max(pw, (g.Nper + 63) / 64 * ((g.D + kPerDirs - 1) / kPerDirs));
        cells = std::max(cells, g.N);
    }
    k_periodic<R, kJobs><<<dim3(grid_for(64 * pw), n), kBlock, 0, st>>>(a);
    k_chemistry<R, kJobs><<<dim3(grid_for(cells), n), kBlock, 0, st>>>(a);
    k_chemistry_tail<R, kJobs><<<dim3((unsigned)std::min<int64_t>((cells + 3) / 4, 2048), n), 64, 0, st>>>(a);
}

// ssw_sweep::rates_current and rates_partial after the sweeps of `order`.
void rates_after(ssw_sweep* s, const std::vector<int>& order) {
    const int last = order.back();
    auto full = [&](int lvl) { return lvl == 0 || s->list_full[lvl]; };
    bool x = s->x_nonneg;  // before the last sweep
    for (size_t i = 0; i + 1 < order.size(); i++) x = x || full(order[i]);
    s->rates_current = s->nonneg && s->areas_nonneg && x && !s->rotated && !s->uneven_faces;
    s->x_nonneg = x || full(last);
    s->rates_partial = !full(last);
}

template <typename R>
int run_step(ssw_sweep* s, double* elapsed) {
    Geo g = make_geo(s);
    Flux<R> fl = make_flux<R>(s);
    const ChemArgs ca = chem_args(s);
    const std::vector<int> order = s->ts.sweep_order();
    const int L = s->p.num_timestep_levels;
    s->rates_current = false;  // an error below leaves a partly swept state
    k_fill_u32<<<1, 8, 0, s->stream>>>((uint32_t*)s->d_active, 0u, 8);
    const unsigned gcells = grid_for(s->N);
    s->sweeps_last = 0;
    s->builds_last = 0;
    s->t_transport_total = s->t_chem_total = s->t_build_total = 0;
    s->n_transport = 0;
    size_t evn = 0;
    std::function<hipEvent_t()> mark = [&](void) -> hipEvent_t {
        if (evn >= s->ev.size()) {
            hipEvent_t e;
            (void)hipEventCreate(&e);
            s->ev.push_back(e);
        }
        hipEvent_t e = s->ev[evn++];
        (void)hipEventRecord(e, s->stream);
        return e;
    };
    std::vector<std::pair<hipEvent_t, hipEvent_t>> tr, ch, bu;
    // sweep levels whose active set changed (device flags set by the level
    // update of the previous step)
    std::vector<uint32_t> need(L, 1u);
    if (L > 1) {
        HIP_TRY(hipMemcpyAsync(need.data(), s->d_need, L * 4, hipMemcpyDeviceToHost, s->stream));
        HIP_TRY(hipStreamSynchronize(s->stream));
    }
    for (int l = 1; l < L; l++)
        if (need[l]) drop_list(s, l);
    for (int lvl : order) {
        if (lvl > 0 && !s->list_ok[lvl]) {
            hipEvent_t b0 = s->timing ? mark() : nullptr;
            TRY(make_list(s, lvl));
            if (s->timing) bu.push_back({b0, mark()});
            s->builds_last++;
        }
        // timing: one event pair around the sweep's whole replay (per-launch
        // events would add their own packets between the launches); the
        // average launch duration is the total over the replay's launches
        hipEvent_t t0 = s->timing ? mark() : nullptr;
        if (s->graphs_on && !s->graphs[lvl] && s->replays[lvl] >= 1)
            capture(s, g, lvl);
        if (s->graphs[lvl]) HIP_TRY(hipGraphLaunch(s->graphs[lvl], s->stream));
        else launch_replay(s, g, lvl, nullptr);
        if (s->timing) {
            tr.push_back({t0, mark()});
            s->n_transport += (int64_t)s->plan[lvl].size();
        }
        HIP_TRY(hipGetLastError());
        s->replays[lvl]++;
        hipEvent_t a = s->timing ? mark() : nullptr;
        const ChemJob<R> job{g, fl, ca, lvl};
        launch_chemistry<R, 1>(&job, 1, s->stream);
        if (s->timing) ch.push_back({a, mark()});
        s->sweeps_last++;
    }
    HIP_TRY(hipGetLastError());
    rates_after(s, order);
    double el = s->ts.current_max_timestep();
    s->ts.advance();
    k_levels<<<gcells, kBlock, 0, s->stream>>>(g, s->d_change, s->d_level, s->p.max_timestep,
                                               s->p.timestep_safety_factor, s->ts.lowest);
    HIP_TRY(hipGetLastError());
    if (s->timing) {
        HIP_TRY(hipStreamSynchronize(s->stream));
        for (auto& pr : tr) {
            float ms = 0;
            (void)hipEventElapsedTime(&ms, pr.first, pr.second);
            s->t_transport_total += ms;
        }
        for (auto& pr : ch) {
            float ms = 0;
            (void)hipEventElapsedTime(&ms, pr.first, pr.second);
            s->t_chem_total += ms;
        }
        for (auto& pr : bu) {
            float ms = 0;
            (void)hipEventElapsedTime(&ms, pr.first, pr.second);
            s->t_build_total += ms;
        }
    }
    if (elapsed) *elapsed = el;
    return SSW_OK;
}

// ---------------------------------------------------------------------------
// Packed steps: one step of each of several handles, their grouped launches
// packed into shared launches (k_sweep_cone_pack).
//
// The handles' sweeps are aligned by index: sweep i of every handle whose
// step has more than i sweeps runs together. Inside sweep i, the next items of
// the handles' replay plans are launched together: grouped items of handles
// with the same transport precision and workgroups go into one packed launch
// (up to kMaxPack per launch), other items are launched alone. The handle with
// the most items left says which workgroups are next; taking the t-th items
// of all, whatever their workgroups, made two launches of many (eight handles,
// 2.44 ms a step instead of 1.65). Each handle's
// items still run in its plan's order (everything is on one stream), and a
// packed workgroup computes exactly what it computes in a launch of its own,
// so every handle's results are bitwise those of stepping it alone.

struct BatchSweep {
    ssw_sweep* s;
    std::vector<int> order;
    Geo g;
};

template <typename R>
GroupJob<R> group_job(ssw_sweep* s, int lvl, const ssw_sweep::ReplayItem& it, uint32_t* nblk) {
    const bool all = lvl == 0 || s->list_full[lvl];
    const ssw_sweep::Group& gr = s->groups[it.tab];
    const Flux<R> fl = make_flux<R>(s);
    const Geo g = make_geo(s);
    GroupJob<R> J;
    J.N = g.N;
    J.X = fl.X;
    J.I = fl.I;
    J.P = fl.P;
    J.offI = fl.offI;
    J.sa = fl.sa;
    J.thr = fl.thr;
    J.level = s->d_level;
    J.blob = s->d_coneblob;
    J.tiles = s->d_conetiles;
    J.more = s->d_conemore;
    J.slot0 = gr.slot0;
    J.cone0 = gr.desc0;
    J.sel = all ? nullptr : s->d_gsel_l[lvl] + gr.desc0;
    J.words = gr.words;
    J.lvl = all ? 0 : lvl;
    J.start = 0;
    *nblk = all ? gr.ndesc : s->gblocks[lvl][it.tab];
    J.blocks = *nblk;
    J.pt = all ? gr.passes : s->gpass_l[lvl][it.tab];
    return J;
}

// A packed launch under construction: jobs of one precision and workgroup.
template <typename R>
struct Pack {
    PackArgs<R> a{};  // value-initialised: no jobs yet
    uint32_t grid = 0;
};

template <typename R>
void flush_pack(Pack<R>& p, int waves, hipStream_t st) {
    if (p.a.n <= 0) return;
    uint32_t words = 0;
    bool general = false;
    for (int k = 0; k < p.a.n; k++) {
        words = std::max(words, p.a.job[k].words);
        general = general || p.a.job[k].lvl > 0 || p.a.job[k].offI;
    }
    hipLaunchKernelGGL(SSW_CONE_KERNEL(k_sweep_cone_pack, R, waves, general), dim3(p.grid), dim3(64 * waves),
                       ConeShape<R>::bytes(waves, words), st, p.a);
    p.a.n = 0;
    p.grid = 0;
}

template <typename R>
void add_job(Pack<R>& p, const GroupJob<R>& J, int waves, hipStream_t st) {
    if (p.a.n >= kMaxPack) flush_pack<R>(p, waves, st);
    GroupJob<R> j = J;
    j.start = p.grid;
    p.grid += (J.blocks + kXcds - 1) / kXcds * kXcds;
    p.a.job[p.a.n++] = j;
}

// Packs keyed by (precision, waves of a workgroup).
struct Packs {
    Pack<float> f[3];
    Pack<double> d[3];
    static int slot(int waves) { return waves == 4 ? 0 : waves == 8 ? 1 : 2; }
    void flush(hipStream_t st) {
        const int waves[3] = {4, 8, 16};
        for (int k = 0; k < 3; k++) {
            flush_pack<float>(f[k], waves[k], st);
            flush_pack<double>(d[k], waves[k], st);
        }
    }
};

template <typename R>
void packed_item(ssw_sweep* s, const Geo& g, int lvl, const ssw_sweep::ReplayItem& it, Pack<R>& pk, hipStream_t st) {
    if (it.group == 1) {
        uint32_t nblk = 0;
        const GroupJob<R> J = group_job<R>(s, lvl, it, &nblk);
        if (nblk) add_job<R>(pk, J, s->groups[it.tab].waves, st);
        return;
    }
    launch_item_t<R>(s, g, make_flux<R>(s), lvl, it, st);
}

// The chemistry of a packed sweep's handles of one precision, kChemJobs to a
// launch: a handle's sub-steps are a chain of their own, and one launch after
// the other would add them up.
template <typename R>
void batch_chemistry(const std::vector<ChemJob<R>>& jobs, hipStream_t st) {
    for (size_t k = 0; k < jobs.size(); k += kChemJobs) {
        const int n = (int)std::min<size_t>(kChemJobs, jobs.size() - k);
        if (n == 1) launch_chemistry<R, 1>(&jobs[k], 1, st);
        else launch_chemistry<R, kChemJobs>(&jobs[k], n, st);
    }
}

// Graphs of packed sweeps, keyed by (uid, epoch, sweep level) of every
// handle in the sweep: a key seen once is captured the second time it comes
// and replayed from then on, as a handle's own replays are. The epoch of a
// handle changes whenever one of its replay plans is rebuilt, so a graph is
// only replayed with the plans (and buffers) it was captured from; graphs of
// destroyed handles are never matched again (uids are not reused) and leave
// the cache by age.
struct PackedGraph {
    std::vector<uint64_t> key;
    int device;
    hipGraphExec_t ge;  // null: seen once, not captured yet
    uint64_t last_use;
};
std::mutex g_pack_mu;
std::vector<PackedGraph> g_pack_graphs;
uint64_t g_pack_clock = 0;
int64_t g_pack_captured = 0, g_pack_replayed = 0;
constexpr size_t kPackGraphs = 256;

// Under g_pack_mu: the entry of key on device dev, or nullptr.
PackedGraph* find_packed(const std::vector<uint64_t>& key, int dev) {
    for (PackedGraph& e : g_pack_graphs)
        if (e.device == dev && e.key == key) {
            e.last_use = ++g_pack_clock;
            return &e;
        }
    return nullptr;
}

// Under g_pack_mu: adds an entry, evicting the least recently used one when full.
void add_packed(const std::vector<uint64_t>& key, int dev, hipGraphExec_t ge) {
    if (g_pack_graphs.size() >= kPackGraphs) {
        size_t old = 0;
        for (size_t k = 1; k < g_pack_graphs.size(); k++)
            if (g_pack_graphs[k].last_use < g_pack_graphs[old].last_use) old = k;
        if (g_pack_graphs[old].ge) (void)hipGraphExecDestroy(g_pack_graphs[old].ge);
        g_pack_graphs.erase(g_pack_graphs.begin() + (std::ptrdiff_t)old);
    }
    g_pack_graphs.push_back(PackedGraph{key, dev, ge, ++g_pack_clock});
}

// Captures what `enqueue` launches on st as one graph (nothing runs). Returns
// null if the capture failed; the caller then launches the work directly.
hipGraphExec_t capture_packed(hipStream_t st, const std::function<void()>& enqueue) {
    hipGraph_t graph = nullptr;
    std::unique_lock<std::shared_mutex> lock(g_capture_mu);
    if (hipStreamBeginCapture(st, hipStreamCaptureModeRelaxed) != hipSuccess) {
        (void)hipGetLastError();
        return nullptr;
    }
    enqueue();
    hipError_t ce = hipStreamEndCapture(st, &graph);
    lock.unlock();
    if (ce != hipSuccess || !graph) {
        if (graph) (void)hipGraphDestroy(graph);
        (void)hipGetLastError();
        return nullptr;
    }
    hipGraphExec_t ge = nullptr;
    hipError_t ie = hipGraphInstantiate(&ge, graph, nullptr, nullptr, 0);
    (void)hipGraphDestroy(graph);
    if (ie != hipSuccess) {
        (void)hipGetLastError();
        return nullptr;
    }
    return ge;
}

// One packed step of the prepared handles bs[0..n) on the stream of the
// first (the others' streams wait for it before and it waits for theirs).
int step_pack(BatchSweep* bs, int n, double* elapsed) {
    const hipStream_t st = bs[0].s->stream;
    for (int h = 1; h < n; h++) {
        ssw_sweep* s = bs[h].s;
        if (!s->sync_ev) HIP_TRY(hipEventCreateWithFlags(&s->sync_ev, hipEventDisableTiming));
        HIP_TRY(hipEventRecord(s->sync_ev, s->stream));
        HIP_TRY(hipStreamWaitEvent(st, s->sync_ev, 0));
    }
    for (int h = 0; h < n; h++) {
        k_fill_u32<<<1, 8, 0, st>>>((uint32_t*)bs[h].s->d_active, 0u, 8);
    }
    size_t sweeps = 0;
    for (int h = 0; h < n; h++) sweeps = std::max(sweeps, bs[h].order.size());
    bool graphs = true;
    for (int h = 0; h < n; h++) graphs = graphs && bs[h].s->graphs_on;
    const int dev = bs[0].s->device;
    for (size_t i = 0; i < sweeps; i++) {
        // sweep i of every handle: plan items together where their workgroups
        // are of the same waves, those of the handle with the most items left
        // first, then the handles' periodic sources and chemistry together
        const std::function<void()> enqueue = [&]() {
            Packs pk;
            std::vector<size_t> at(n, 0);
            auto left = [&](int h) {
                return i < bs[h].order.size() ? bs[h].s->plan[bs[h].order[i]].size() - at[h] : (size_t)0;
            };
            auto item = [&](int h) -> const ssw_sweep::ReplayItem& { return bs[h].s->plan[bs[h].order[i]][at[h]]; };
            auto waves = [&](int h) { return item(h).group == 1 ? bs[h].s->groups[item(h).tab].waves : 0; };
            for (;;) {
                int lead = 0;
                for (int h = 1; h < n; h++)
                    if (left(h) > left(lead)) lead = h;
                if (!left(lead)) break;
                const int wv = waves(lead);
                for (int h = 0; h < n; h++) {
                    if (!left(h) || waves(h) != wv) continue;
                    BatchSweep& b = bs[h];
                    const int lvl = b.order[i], k = Packs::slot(wv);
                    if (b.s->fp32) packed_item<float>(b.s, b.g, lvl, item(h), pk.f[k], st);
                    else packed_item<double>(b.s, b.g, lvl, item(h), pk.d[k], st);
                    at[h]++;
                }
                pk.flush(st);
            }
            std::vector<ChemJob<float>> jf;
            std::vector<ChemJob<double>> jd;
            for (int h = 0; h < n; h++) {
                BatchSweep& b = bs[h];
                if (i >= b.order.size()) continue;
                if (b.s->fp32) jf.push_back({b.g, make_flux<float>(b.s), chem_args(b.s), b.order[i]});
                else jd.push_back({b.g, make_flux<double>(b.s), chem_args(b.s), b.order[i]});
            }
            batch_chemistry<float>(jf, st);
            batch_chemistry<double>(jd, st);
        };
        bool done = false;
        if (graphs) {
            std::vector<uint64_t> key;
            for (int h = 0; h < n; h++)
                if (i < bs[h].order.size())
                    key.insert(key.end(), {bs[h].s->uid, bs[h].s->epoch, (uint64_t)bs[h].order[i]});
            std::lock_guard<std::mutex> lk(g_pack_mu);
            PackedGraph* e = find_packed(key, dev);
            if (e && !e->ge) {  // the second time: capture
                e->ge = capture_packed(st, enqueue);
                if (e->ge) g_pack_captured++;
            }
            if (e && e->ge) {
                HIP_TRY(hipGraphLaunch(e->ge, st));
                g_pack_replayed++;
                done = true;
            } else if (!e) {
                add_packed(key, dev, nullptr);
            }
        }
        if (!done) enqueue();
        for (int h = 0; h < n; h++)
            if (i < bs[h].order.size()) bs[h].s->sweeps_last++;
        HIP_TRY(hipGetLastError());
    }
    for (int h = 0; h < n; h++) {
        ssw_sweep* s = bs[h].s;
        rates_after(s, bs[h].order);
        const double el = s->ts.current_max_timestep();
        s->ts.advance();
        k_levels<<<grid_for(s->N), kBlock, 0, st>>>(bs[h].g, s->d_change, s->d_level, s->p.max_timestep,
                                                   s->p.timestep_safety_factor, s->ts.lowest);
        if (elapsed) elapsed[h] = el;
    }
    HIP_TRY(hipGetLastError());
    // the handles' own streams continue after the packed step
    ssw_sweep* s0 = bs[0].s;
    if (!s0->sync_ev) HIP_TRY(hipEventCreateWithFlags(&s0->sync_ev, hipEventDisableTiming));
    HIP_TRY(hipEventRecord(s0->sync_ev, st));
    for (int h = 1; h < n; h++) HIP_TRY(hipStreamWaitEvent(bs[h].s->stream, s0->sync_ev, 0));
    return SSW_OK;
}

// Packs of about kPackSize handles, on up to kPackStreams streams: the device
// runs the launches of a few streams at once (one hardware queue per stream,
// dealt to streams in turn as they are created), so a few packs side by side
// beat one pack of all of them. Handle k goes to pack uid(k) mod npack
// (creation turn; evened out where the turns are uneven), so that the packs'
// streams sit on different queues and every pack holds a mix of problem
// sizes; within a pack the longest plan leads. Measured on 16 small problems
// (8000-27000 cells, 16-84 directions): 3.46 ms per step against 4.28 ms for
// packs of similar sizes and 5.34 ms for one stream per problem.
constexpr int kPackSize = 4;
constexpr int kPackStreams = 4;

int step_batch(ssw_sweep* const* hs, int n, double* elapsed) {
    std::vector<BatchSweep> bs((size_t)n);
    // per handle, on its own stream: the sweep levels whose active set
    // changed, and their active-set lists (the lists depend only on the
    // timestep levels, which change at the end of a step)
    for (int h = 0; h < n; h++) {
        ssw_sweep* s = hs[h];
        BatchSweep& b = bs[h];
        b.s = s;
        b.order = s->ts.sweep_order();
        b.g = make_geo(s);
        const int L = s->p.num_timestep_levels;
        s->rates_current = false;
        s->sweeps_last = 0;
        s->builds_last = 0;
        s->t_transport_total = s->t_chem_total = s->t_build_total = 0;
        s->n_transport = 0;
        std::vector<uint32_t> need(L, 1u);
        if (L > 1) {
            HIP_TRY(hipMemcpyAsync(need.data(), s->d_need, L * 4, hipMemcpyDeviceToHost, s->stream));
            HIP_TRY(hipStreamSynchronize(s->stream));
        }
        for (int l = 1; l < L; l++)
            if (need[l]) drop_list(s, l);
        for (int lvl : b.order)
            if (lvl > 0 && !s->list_ok[lvl]) {
                TRY(make_list(s, lvl));
                s->builds_last++;
            }
    }
    // handles by their full sweep's plan length (a proxy of their per-step
    // chain), longest first, dealt to the packs by creation turn
    std::vector<int> order((size_t)n);
    for (int h = 0; h < n; h++) order[h] = h;
    std::stable_sort(order.begin(), order.end(),
                     [&](int x, int y) { return bs[x].s->plan[0].size() > bs[y].s->plan[0].size(); });
    const int npack = std::min(kPackStreams, (n + kPackSize - 1) / kPackSize);
    std::vector<std::vector<int>> packs((size_t)npack);
    for (int r = 0; r < n; r++) packs[bs[order[r]].s->uid % (uint64_t)npack].push_back(order[r]);
    for (;;) {  // even out: no pack more than one above another
        auto big = std::max_element(packs.begin(), packs.end(),
                                    [](const std::vector<int>& x, const std::vector<int>& y) { return x.size() < y.size(); });
        auto small = std::min_element(packs.begin(), packs.end(),
                                      [](const std::vector<int>& x, const std::vector<int>& y) { return x.size() < y.size(); });
        if (big->size() <= small->size() + 1) break;
        small->push_back(big->back());
        big->pop_back();
    }
    // the lead (whose stream a pack runs on) of each pack: its longest member,
    // unless an evened-out pack needs another member to sit at a place in the
    // turn of the hardware queues (creation order modulo the queue count) that
    // no earlier pack's lead holds
    uint32_t used = 0;
    for (size_t k = 0; k < packs.size(); k++) {
        std::vector<int>& m = packs[k];
        for (size_t j = 0; j < m.size(); j++) {
            const uint32_t q = 1u << (bs[m[j]].s->uid % (uint64_t)kPackStreams);
            if (!(used & q)) {
                std::swap(m[0], m[j]);
                break;
            }
        }
        used |= 1u << (bs[m[0]].s->uid % (uint64_t)kPackStreams);
    }
    // each pack from a thread of its own (the first on the caller's): issuing
    // the launches of a step takes host time comparable to running them
    const int np = (int)packs.size();
    std::vector<int> rc((size_t)np, SSW_OK);
    std::vector<std::string> err((size_t)np);
    auto run = [&](int k) {
        std::vector<BatchSweep> sub;
        for (int h : packs[k]) sub.push_back(bs[h]);
        std::vector<double> el(sub.size(), 0.0);
        rc[k] = step_pack(sub.data(), (int)sub.size(), el.data());
        if (rc[k] != SSW_OK) err[k] = g_err;
        if (elapsed)
            for (size_t j = 0; j < sub.size(); j++) elapsed[packs[k][j]] = el[j];
    };
    std::vector<std::thread> th;
    int spawned = 1;
    try {
        for (; spawned < np; spawned++) th.emplace_back(run, spawned);
    } catch (const std::exception&) {  // no thread to spare: the rest on this one
    }
    run(0);
    for (int k = spawned; k < np; k++) run(k);
    for (std::thread& t : th) t.join();
    for (int k = 0; k < np; k++)
        if (rc[k] != SSW_OK) return fail(rc[k], err[k]);
    return SSW_OK;
}

// Pinned host memory through which downloads pass, one for the process:
// kernels write the outputs into it in the caller's order, chunk by chunk, and
// host threads copy finished chunks on into the caller's arrays (whose pages
// are usually touched there for the first time: 5 GB/s on one thread). Made at
// a handle's second download, freed with the last handle; a download that
// finds it in use by another thread takes the plain path. Results of 262144
// cells: 1.8 -> 0.27 ms, of 1000 cells 0.10 -> 0.03 ms (six
// copies of 25 us each before).
constexpr uint32_t kStageCells = 49152;             // cells of a chunk
constexpr int kStageChunks = 16;
constexpr size_t kStageChunkBytes = (size_t)kStageCells * (6 * 8 + 1);
constexpr int kStageThreads = 6;
struct Staging {
    std::mutex mu;
    uint8_t* host = nullptr;
    int device = -1;
    std::vector<hipEvent_t> done;
    void free() {
        if (host) (void)hipHostFree(host);
        host = nullptr;
        for (hipEvent_t e : done) (void)hipEventDestroy(e);
        done.clear();
    }
    bool make(int dev) {
        if (host) return device == dev;
        std::shared_lock<std::shared_mutex> lock(g_capture_mu);
        device = dev;
        if (hipHostMalloc((void**)&host, kStageChunkBytes * kStageChunks, hipHostMallocDefault) != hipSuccess) {
            (void)hipGetLastError();
            host = nullptr;
            return false;
        }
        for (int k = 0; k < kStageChunks; k++) {
            hipEvent_t e;
            if (hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) {
                (void)hipGetLastError();
                free();
                return false;
            }
            done.push_back(e);
        }
        return true;
    }
};
Staging g_staging;

// The device arrays `src` (and levels) into the host arrays `dst` in the
// caller's cell order. Plain path: one copy per array, permuted on the host.
int fetch_outputs(ssw_sweep* s, const std::vector<const double*>& src, const std::vector<double*>& dst,
                  const uint8_t* d_level, uint8_t* level) {
    const int64_t n = s->N;
    std::unique_lock<std::mutex> lock(g_staging.mu, std::try_to_lock);
    if (!s->downloaded || !lock.owns_lock() || !g_staging.make(s->device)) {
        s->downloaded = true;
        for (size_t k = 0; k < src.size(); k++)
            HIP_TRY(hipMemcpyAsync(dst[k], src[k], n * 8, hipMemcpyDeviceToHost, s->stream));
        if (level) HIP_TRY(hipMemcpyAsync(level, d_level, n, hipMemcpyDeviceToHost, s->stream));
        HIP_TRY(hipStreamSynchronize(s->stream));
        for (double* a : dst) to_caller(s, a, 1);
        if (level) to_caller(s, level, 1);
        return SSW_OK;
    }
    OutputArrays oa{};
    oa.n = (int)src.size();
    for (int k = 0; k < oa.n; k++) oa.a[k] = src[k];
    oa.level = level ? d_level : nullptr;
    for (int64_t r0 = 0; r0 < n; r0 += (int64_t)kStageCells * kStageChunks) {
        const int chunks = (int)std::min<int64_t>(kStageChunks, (n - r0 + kStageCells - 1) / kStageCells);
        auto first = [&](int c) { return r0 + (int64_t)c * kStageCells; };
        auto cells = [&](int c) { return std::min<int64_t>(kStageCells, n - first(c)); };
        auto copy = [&](int c) {
            const uint8_t* st = g_staging.host + (size_t)c * kStageChunkBytes;
            for (int k = 0; k < oa.n; k++)
                std::memcpy(dst[k] + first(c), st + (size_t)k * kStageCells * 8, (size_t)cells(c) * 8);
            if (level) std::memcpy(level + first(c), st + (size_t)oa.n * kStageCells * 8, (size_t)cells(c));
        };
        for (int c = 0; c < chunks; c++) {
            k_stage_outputs<<<grid_for(cells(c)), kBlock, 0, s->stream>>>(
                oa, s->permuted ? s->d_perm : nullptr, (uint32_t)first(c), (uint32_t)cells(c), kStageCells,
                (double*)(g_staging.host + (size_t)c * kStageChunkBytes));
            HIP_TRY(hipGetLastError());
            if (chunks > 1) HIP_TRY(hipEventRecord(g_staging.done[c], s->stream));
        }
        if (chunks == 1) {
            HIP_TRY(hipStreamSynchronize(s->stream));
            copy(0);
            continue;
        }
        std::atomic<int> next{0};
        std::atomic<bool> failed{false};
        auto work = [&] {
            for (int c = next++; c < chunks; c = next++) {
                if (hipEventSynchronize(g_staging.done[c]) != hipSuccess) failed = true;
                copy(c);
            }
        };
        std::vector<std::thread> th;
        try {
            for (int k = 1; k < std::min(kStageThreads, chunks); k++) th.emplace_back(work);
        } catch (const std::exception&) {  // no thread to spare: fewer
        }
        work();
        for (std::thread& t : th) t.join();
        if (failed) return fail(SSW_ERR_HIP, "a download's kernel failed");
    }
    return SSW_OK;
}

void free_state(ssw_sweep* s) {
    dfree(s, s->d_rho);
    dfree(s, s->d_x);
    dfree(s, s->d_T);
    dfree(s, s->d_src);
    dfree(s, s->d_sa);
    dfree(s, s->d_sts);
    dfree(s, s->d_prev);
    dfree(s, s->d_change);
    dfree(s, s->d_chemq);
    dfree(s, s->d_photon);
    dfree(s, s->d_rate);
    dfree(s, s->d_X);
    dfree(s, s->d_I);
    dfree(s, s->d_P);
    dfree(s, s->d_offI);
    dfree(s, s->d_offP);
}

// Everything that build_schedule makes.
void free_schedule(ssw_sweep* s) {
    s->have_schedule = false;
    drop_all_lists(s);
    for (uint32_t*& p : s->d_idx) dfree(s, p);
    for (uint4*& p : s->d_runtab) dfree(s, p);
    free_groups(s);
    dfree(s, s->d_fstart);
    dfree(s, s->d_dirblob);
    dfree(s, s->d_dirtiles);
    dfree(s, s->d_dirinfo);
    dfree(s, s->d_dircell);
    dfree(s, s->d_dirsa);
    dfree(s, s->d_dirlev);
    dfree(s, s->d_recs);
    dfree(s, s->d_hdr);
    dfree(s, s->d_A);
    dfree(s, s->d_planes);
    dfree(s, s->d_ovf_start);
    dfree(s, s->d_ovf);
    dfree(s, s->d_xpos);
    dfree(s, s->d_chunks);
    dfree(s, s->d_first_chunk);
    dfree(s, s->d_ccount);
    dfree(s, s->d_coff);
    dfree(s, s->d_cstart);
    dfree(s, s->d_scan_tmp);
}

void free_grid(ssw_sweep* s) {
    free_schedule(s);
    dfree(s, s->d_off);
    dfree(s, s->d_inv);
    dfree(s, s->d_perm);
    dfree(s, s->d_geo);
    dfree(s, s->d_nk);
    dfree(s, s->d_vol);
    dfree(s, s->d_size);
    dfree(s, s->d_pslot);
    dfree(s, s->d_pcells);
    dfree(s, s->d_pfoff);
    dfree(s, s->d_pnb);
    dfree(s, s->d_pgeo);
    dfree(s, s->d_cnt);
    dfree(s, s->d_level);
    dfree(s, s->d_nup);
}

// Overflow entries of the per-level replay's planes (s->ovf_total of them).
int setup_overflow(ssw_sweep* s) {
    const size_t DN = (size_t)s->D * s->N;
    uint32_t *d_cursor = nullptr, *d_count = nullptr;
    unsigned long long* d_stats = nullptr;
    Defer cleanup{[&] {
        dfree(s, d_cursor);
        dfree(s, d_count);
        dfree(s, d_stats);
    }};
    TRY(dalloc(s, &d_count, DN));
    TRY(dalloc(s, &d_stats, 4));
    Geo g = make_geo(s);
    k_face_stats<<<(unsigned)((s->N + kFluxCells - 1) / kFluxCells),
                   kFluxCells * ((s->D + kFluxDirs - 1) / kFluxDirs), 0, s->stream>>>(g, d_stats, d_count, nullptr);
    HIP_TRY(hipGetLastError());
    TRY(dalloc(s, &s->d_ovf_start, DN));
    TRY(dalloc(s, (uint8_t**)&s->d_ovf, (size_t)std::max<int64_t>(1, s->ovf_total) * entry_size(s)));
    TRY(dalloc(s, &d_cursor, 1));
    HIP_TRY(hipMemsetAsync(d_cursor, 0, 4, s->stream));
    k_overflow<<<grid_for((int64_t)DN), kBlock, 0, s->stream>>>(g, d_count, s->d_ovf_start, d_cursor);
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipStreamSynchronize(s->stream));
    return SSW_OK;
}

// The device address of `scratch` on device `dev`, looked up once per device
// with that device current (each device holds its own copy of the array at
// its own address) and kept for the life of the process.
std::mutex g_scratch_mu;
std::array<void*, kMaxDevices> g_scratch_ptr{};

int noalloc_scratch(int dev, uint8_t** out) {
    if (dev < 0 || dev >= kMaxDevices) return fail(SSW_ERR_INVALID, "device ordinal out of range");
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
        int cur = -1;
        HIP_TRY(hipGetDevice(&cur));
        if (cur != dev) HIP_TRY(hipSetDevice(dev));
        void* p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (cur != dev) HIP_TRY(hipSetDevice(cur));
        if (e != hipSuccess || !p)
            return fail(SSW_ERR_HIP, std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e));
        g_scratch_ptr[dev] = p;
    }
    *out = (uint8_t*)g_scratch_ptr[dev];
    return SSW_OK;
}

// One per-cell output of ssw_download_noalloc: into the caller's order through
// the staging buffer when the grid is permuted, else copied directly.
template <typename T>
int noalloc_out(ssw_sweep* s, const T* src, T* dst, uint8_t* stage) {
    const int64_t n = s->N;
    if (s->permuted) {
        k_to_caller<T><<<grid_for(n), kBlock, 0, s->stream>>>(src, s->d_inv, (T*)stage, n);
        HIP_TRY(hipGetLastError());
        src = (const T*)stage;
    }
    // the next output reuses the staging buffer: stream order puts its kernel
    // after this copy
    HIP_TRY(hipMemcpyAsync(dst, src, (size_t)n * sizeof(T), hipMemcpyDeviceToHost, s->stream));
    return SSW_OK;
}

ssw::Problem memory_problem(const ssw_sweep_parameters& p, int64_t n, int64_t faces, int64_t periodic_cells) {
    return {n, faces, periodic_cells, p.num_directions, p.num_timestep_levels,
            p.transport_precision == SSW_TRANSPORT_FP32};
}

// The per-direction dependency graph of the uploaded faces under the current
// directions: mirror check (first build), downwind statistics, overflow
// counts, the transport mode (choose_mode) and the schedule. d_cnt is held.
int build_direction_graph(ssw_sweep* s, bool choose_mode) {
    const int64_t n = s->N;
    const size_t DN = (size_t)s->D * n;
    unsigned long long* d_stats = nullptr;
    Defer cleanup{[&] { dfree(s, d_stats); }};
    TRY(dalloc(s, &d_stats, 6));
    HIP_TRY(hipMemsetAsync(d_stats, 0, 6 * 8, s->stream));
    Geo g = make_geo(s);
    if (choose_mode) k_check_mirror<<<grid_for(n), kBlock, 0, s->stream>>>(g, d_stats, d_stats + 5);
    const bool tiles = (s->dir_sweeps || s->group_request >= 2) &&
                       (choose_mode ? s->mode_request != SSW_TRANSPORT_MODE_GEOMETRIC : s->compiled);
    if (tiles) TRY(dalloc(s, &s->d_nup, DN));
    k_face_stats<<<(unsigned)((n + kFluxCells - 1) / kFluxCells),
                   kFluxCells * ((s->D + kFluxDirs - 1) / kFluxDirs), 0, s->stream>>>(g, d_stats + 1, s->d_cnt,
                                                                                      s->d_nup);
    HIP_TRY(hipGetLastError());
    unsigned long long hb[6] = {0, 0, 0, 0, 0, 0};
    HIP_TRY(hipMemcpyAsync(hb, d_stats, sizeof(hb), hipMemcpyDeviceToHost, s->stream));
    HIP_TRY(hipStreamSynchronize(s->stream));
    dfree(s, d_stats);
    if (hb[0] != 0)
        return fail(SSW_ERR_GRID, std::to_string(hb[0]) +
                                      " local faces have no mirror face with the exactly negated normal");
    if (choose_mode) s->uneven_faces = hb[5] != 0;
    for (int k = 0; k < 3; k++) s->dw[k] = (double)hb[k + 1] / ((double)n * s->D);
    s->ovf_total = (int64_t)hb[4];
    if (!choose_mode) {
        return build_schedule(s);
    }
    // transport mode: compiled when the least that a compiled replay needs (planes,
    // or the directions' tiles; cones are built where they fit as well) is at
    // most 85% of the free device memory (automatic), else geometric
    const int64_t need = ssw::replay_bytes(memory_problem(s->p, n, s->F, s->Nper),
                                           s->dir_sweeps && !s->uneven_faces ? ssw::Replay::kDirections
                                                                             : ssw::Replay::kPerLevel) +
                         std::max<int64_t>(0, s->ovf_total - (int64_t)DN / 16) * (int64_t)entry_size(s);
    if (s->mode_request == SSW_TRANSPORT_MODE_COMPILED) s->compiled = true;
    else if (s->mode_request == SSW_TRANSPORT_MODE_GEOMETRIC) s->compiled = false;
    else s->compiled = (double)need <= 0.85 * (double)expected_free(s);
    if (!s->compiled) dfree(s, s->d_nup);
    return build_schedule(s);
}

// The row-major matrix times every direction (multiply_by_matrix,
// src/sweep/direction/mod.rs:150-155), and kept[i] = kernel[i][D-1] of remap
// (:177-205): 1 if the last rotated direction is the last of the rotated
// directions most aligned with old direction i (Iterator::max_by_key keeps
// the last maximum of 1 + old_i . new_j), else 0.
void rotate_table(const double* m, std::vector<double>& dirs, std::vector<double>& kept) {
    const int D = (int)dirs.size() / 3;
    const std::vector<double> old = dirs;
    for (int d = 0; d < D; d++) {
        const double x = old[3 * d], y = old[3 * d + 1], z = old[3 * d + 2];
        dirs[3 * d] = x * m[0] + y * m[1] + z * m[2];
        dirs[3 * d + 1] = x * m[3] + y * m[4] + z * m[5];
        dirs[3 * d + 2] = x * m[6] + y * m[7] + z * m[8];
    }
    kept.assign(D, 0.0);
    for (int i = 0; i < D; i++) {
        int best = 0;
        double best_v = 0.0;
        for (int j = 0; j < D; j++) {
            const double v =
                1.0 + ((old[3 * i] * dirs[3 * j] + old[3 * i + 1] * dirs[3 * j + 1]) + old[3 * i + 2] * dirs[3 * j + 2]);
            if (j == 0 || v >= best_v) {
                best = j;
                best_v = v;
            }
        }
        kept[i] = best == D - 1 ? 1.0 : 0.0;
    }
}

template <typename R>
int rotate_state_t(ssw_sweep* s, const double* d_kept, const double* dI, const double* dO, const double* dP) {
    const int64_t DN = (int64_t)s->D * s->N;
    const size_t rs = sizeof(R);
    if (!s->d_offI) TRY(dalloc(s, (uint8_t**)&s->d_offI, (size_t)DN * rs));
    if (!s->d_offP) TRY(dalloc(s, (uint8_t**)&s->d_offP, (size_t)s->D * std::max<int64_t>(1, s->Nper) * rs));
    const Geo g = make_geo(s);
    const Flux<R> fl = make_flux<R>(s);
    k_rotate_state<R><<<grid_for(DN), kBlock, 0, s->stream>>>(g, fl, d_kept, dI, dO, dP);
    k_rotate_offsets<R><<<grid_for(DN), kBlock, 0, s->stream>>>(g, fl);
    HIP_TRY(hipGetLastError());
    return SSW_OK;
}

}  // namespace

extern "C" {

const char* ssw_last_error(void) { return g_err.c_str(); }

void ssw_default_parameters(ssw_sweep_parameters* p) {
    std::memset(p, 0, sizeof(*p));
    p->num_directions = 84;
    p->explicit_directions = nullptr;
    p->num_timestep_levels = 1;
    p->periodic = 0;
    p->max_timestep = 1e6 * 3.15576e7;
    p->significant_rate_threshold = 0.0;
    p->timestep_safety_factor = 0.01 * 10.0;  // percent(10.0)
    p->chemistry_timestep_safety_factor = 0.01 * 10.0;
    p->prevent_cooling = 1;
    p->transport_precision = SSW_TRANSPORT_FP64;
    p->scale_factor = 1.0;
}

int ssw_create(const ssw_sweep_parameters* params, ssw_sweep** out) {
    if (!params || !out) return fail(SSW_ERR_INVALID, "null argument");
    *out = nullptr;
    const ssw_sweep_parameters& p = *params;
    if (p.num_timestep_levels < 1 || p.num_timestep_levels >= 32)
        return fail(SSW_ERR_INVALID, "num_timestep_levels must be in [1, 31]");
    if (p.transport_precision != SSW_TRANSPORT_FP64 && p.transport_precision != SSW_TRANSPORT_FP32)
        return fail(SSW_ERR_INVALID, "transport_precision must be 32 or 64");
    if (!(p.max_timestep > 0.0)) return fail(SSW_ERR_INVALID, "max_timestep must be positive");
    std::vector<double> dirs;
    if (p.explicit_directions) {
        if (p.num_directions < 1 || p.num_directions > 127)
            return fail(SSW_ERR_INVALID, "explicit direction count must be in [1, 127]");
        for (int d = 0; d < p.num_directions; d++) {
            const double* v = p.explicit_directions + 3 * d;
            double len = std::sqrt((v[0] * v[0] + v[1] * v[1]) + v[2] * v[2]);
            if (!(len > 0.0)) return fail(SSW_ERR_INVALID, "zero explicit direction");
            double r = 1.0 / len;  // glam normalize: v * (1/|v|)
            dirs.push_back(v[0] * r);
            dirs.push_back(v[1] * r);
            dirs.push_back(v[2] * r);
        }
    } else {
        const double(*bins)[3] = nullptr;
        static const double one[1][3] = {{1.0, 0.0, 0.0}};
        switch (p.num_directions) {  // Directions::from_num (src/sweep/direction/mod.rs:58-75)
            case 1: bins = one; break;
            case 16: bins = SSW_DIRECTION_BINS_16; break;
            case 21: bins = SSW_DIRECTION_BINS_21; break;
            case 32: bins = SSW_DIRECTION_BINS_32; break;
            case 64: bins = SSW_DIRECTION_BINS_64; break;
            case 84: bins = SSW_DIRECTION_BINS_84; break;
            default: return fail(SSW_ERR_INVALID, "num_directions must be 1, 16, 21, 32, 64 or 84");
        }
        for (int d = 0; d < p.num_directions; d++)
            for (int k = 0; k < 3; k++) dirs.push_back(bins[d][k]);
    }
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev < 1) return fail(SSW_ERR_NO_DEVICE, "no HIP device");
    ssw_sweep* s = new ssw_sweep();
    s->uid = g_next_uid.fetch_add(1) + 1;
    g_live_handles++;
    s->p = p;
    s->p.explicit_directions = nullptr;
    s->D = p.num_directions;
    s->dirs = dirs;
    s->fp32 = p.transport_precision == SSW_TRANSPORT_FP32;
    (void)hipGetDevice(&s->device);
    hipError_t se;
    {
        std::shared_lock<std::shared_mutex> lock(g_capture_mu);
        se = hipStreamCreateWithFlags(&s->stream, hipStreamNonBlocking);
    }
    if (se != hipSuccess) {
        delete s;
        g_live_handles--;
        return fail(SSW_ERR_HIP, "hipStreamCreate failed");
    }
    int r = dalloc(s, &s->d_dirs, dirs.size());
    if (r == SSW_OK) r = dalloc(s, &s->d_need, (size_t)p.num_timestep_levels);
    if (r == SSW_OK) r = dalloc(s, &s->d_fail, 1);
    if (r == SSW_OK) r = dalloc(s, &s->d_active, 4);
    if (r != SSW_OK) {
        ssw_destroy(s);
        return r;
    }
    if (hipMemcpyAsync(s->d_dirs, dirs.data(), dirs.size() * 8, hipMemcpyHostToDevice, s->stream) != hipSuccess ||
        hipMemsetAsync(s->d_fail, 0, 8, s->stream) != hipSuccess ||
        hipMemsetAsync(s->d_active, 0, 32, s->stream) != hipSuccess || hipStreamSynchronize(s->stream) != hipSuccess) {
        ssw_destroy(s);
        return fail(SSW_ERR_HIP, "initialisation of the handle's device memory failed");
    }
    s->ts.init(p.max_timestep, p.num_timestep_levels);
    *out = s;
    return SSW_OK;
}

void ssw_destroy(ssw_sweep* s) {
    if (!s) return;
    if (s->stream) (void)hipStreamSynchronize(s->stream);
    free_state(s);
    free_grid(s);
    dfree(s, s->d_dirs);
    dfree(s, s->d_need);
    dfree(s, s->d_fail);
    dfree(s, s->d_active);
    for (hipEvent_t e : s->ev) (void)hipEventDestroy(e);
    if (s->sync_ev) (void)hipEventDestroy(s->sync_ev);
    if (s->stream) {
        std::shared_lock<std::shared_mutex> lock(g_capture_mu);
        (void)hipStreamDestroy(s->stream);
    }
    delete s;
    if (--g_live_handles == 0) {
        std::lock_guard<std::mutex> lock(g_staging.mu);
        std::shared_lock<std::shared_mutex> alloc(g_capture_mu);
        if (g_live_handles == 0) g_staging.free();
    }
}

int ssw_set_transport_mode(ssw_sweep* s, int32_t mode) {
    if (!s) return fail(SSW_ERR_INVALID, "null handle");
    if (mode != SSW_TRANSPORT_MODE_AUTO && mode != SSW_TRANSPORT_MODE_GEOMETRIC && mode != SSW_TRANSPORT_MODE_COMPILED)
        return fail(SSW_ERR_INVALID, "transport mode " + std::to_string(mode) +
                                         " is not available (0 automatic, 3 geometric, 4 compiled)");
    if (s->have_grid) return fail(SSW_ERR_INVALID, "the transport mode must be set before ssw_upload_grid");
    s->mode_request = mode;
    return SSW_OK;
}

int ssw_set_replay_block(ssw_sweep* s, int32_t block) {
    if (!s) return fail(SSW_ERR_INVALID, "null handle");
    if (block != 0 && block != 64 && block != 128 && block != 256)
        return fail(SSW_ERR_INVALID, "replay block size must be 0, 64, 128 or 256");
    s->rec_block = block ? block : 64;
    s->epoch++;
    for (hipGraphExec_t& ge : s->graphs)  // graphs hold the old launch shape
        if (ge) {
            (void)hipGraphExecDestroy(ge);
            ge = nullptr;
        }
    std::fill(s->replays.begin(), s->replays.end(), 0);
    return SSW_OK;
}

int ssw_set_cell_positions(ssw_sweep* s, int64_t n, const double* positions) {
    if (!s) return fail(SSW_ERR_INVALID, "null handle");
    if (s->have_grid) return fail(SSW_ERR_INVALID, "cell positions must be set before ssw_upload_grid");
    if (!positions || n <= 0) {
        s->pos.clear();
        return SSW_OK;
    }
    s->pos.assign(positions, positions + 3 * n);
    return SSW_OK;
}

int ssw_set_group_levels(ssw_sweep* s, int32_t levels) {
    if (!s) return fail(SSW_ERR_INVALID, "null handle");
    if (levels < 1 || levels > kMaxGroup) return fail(SSW_ERR_INVALID, "group levels must be 1 to 8");
    if (s->have_grid) return fail(SSW_ERR_INVALID, "ssw_set_group_levels must be called before ssw_upload_grid");
    s->group_request = levels;
    return SSW_OK;
}

int ssw_set_direction_sweeps(ssw_sweep* s, int32_t enabled) {
    if (!s) return fail(SSW_ERR_INVALID, "null handle");
    if (s->have_grid) return fail(SSW_ERR_INVALID, "ssw_set_direction_sweeps must be called before ssw_upload_grid");
    s->dir_sweeps = enabled != 0;
    return SSW_OK;
}

int ssw_direction_table(int32_t num_directions, double* out) {
    if (!out) return fail(SSW_ERR_INVALID, "null argument");
    const double(*bins)[3] = nullptr;
    static const double one[1][3] = {{1.0, 0.0, 0.0}};
    switch (num_directions) {  // Directions::from_num (src/sweep/direction/mod.rs:58-75)
        case 1: bins = one; break;
        case 16: bins = SSW_DIRECTION_BINS_16; break;
        case 21: bins = SSW_DIRECTION_BINS_21; break;
        case 32: bins = SSW_DIRECTION_BINS_32; break;
        case 64: bins = SSW_DIRECTION_BINS_64; break;
        case 84: bins = SSW_DIRECTION_BINS_84; break;
        default: return fail(SSW_ERR_INVALID, "num_directions must be 1, 16, 21, 32, 64 or 84");
    }
    for (int d = 0; d < num_directions; d++)
        for (int k = 0; k < 3; k++) out[3 * d + k] = bins[d][k];
    return SSW_OK;
}

int ssw_set_group_block(ssw_sweep* s, int32_t roots) {
    if (!s) return fail(SSW_ERR_INVALID, "null handle");
    if (roots != 0 && roots != 32 && roots != 64 && roots != 128)
        return fail(SSW_ERR_INVALID, "group block must be 0, 32, 64 or 128");
    if (s->have_grid) return fail(SSW_ERR_INVALID, "ssw_set_group_block must be called before ssw_upload_grid");
    s->group_block = roots ? roots : kGroupT;
    return SSW_OK;
}

int ssw_set_narrow_runs(ssw_sweep* s, int32_t enabled) {
    if (!s) return fail(SSW_ERR_INVALID, "null handle");
    if (s->have_grid) return fail(SSW_ERR_INVALID, "ssw_set_narrow_runs must be called before ssw_upload_grid");
    s->narrow_runs = enabled != 0;
    return SSW_OK;
}

int ssw_set_graph_replay(ssw_sweep* s, int32_t enabled) {
    if (!s) return fail(SSW_ERR_INVALID, "null handle");
    s->graphs_on = enabled != 0;
    s->epoch++;
    if (!s->graphs_on)
        for (hipGraphExec_t& ge : s->graphs)
            if (ge) {
                (void)hipGraphExecDestroy(ge);
                ge = nullptr;
            }
    return SSW_OK;
}

int ssw_upload_grid(ssw_sweep* s, int64_t n, const int64_t* off, const int32_t* nbr, const uint8_t* kind,
                    const double* area, const double* normal, const double* volume, const double* size) {
    if (!s || !off || !nbr || !kind || !area || !normal || !volume || !size)
        return fail(SSW_ERR_INVALID, "null argument");
    if (n <= 0 || n > (int64_t)kCellMask) return fail(SSW_ERR_INVALID, "cell count must be in [1, 2^25 - 1]");
    if ((int64_t)s->D * n >= (int64_t)0x7FFFFFFFll)
        return fail(SSW_ERR_INVALID, "cells x directions must be below 2^31");
    if (off[0] != 0) return fail(SSW_ERR_INVALID, "face_offsets[0] must be 0");
    for (int64_t c = 0; c < n; c++) {
        if (off[c + 1] < off[c]) return fail(SSW_ERR_INVALID, "face_offsets must be non-decreasing");
        if (off[c + 1] - off[c] > kMaxFaces) return fail(SSW_ERR_INVALID, "a cell has more than 127 faces");
    }
    const int64_t F = off[n];
    if (F >= (int64_t)0xFFFFFFFFll) return fail(SSW_ERR_INVALID, "too many faces");
    expect_frees(s);
    free_state(s);
    free_grid(s);
    s->have_grid = s->have_state = false;
    s->N = n;
    s->F = F;
    TRY(make_order(s, n));
    double asum = 0.0;
    s->areas_nonneg = true;
    for (int64_t f = 0; f < F; f++) {
        asum += area[f];  // caller's order: independent of the internal order
        if (!(area[f] >= 0.0)) s->areas_nonneg = false;
    }
    // Areas are carried in units of a power of two near the mean face area, so
    // that X = O / A keeps the range of O (SI areas reach 1e42 m^2); scaling
    // by a power of two is exact.
    s->aref = (F > 0 && asum > 0.0) ? std::ldexp(1.0, (int)std::lround(std::log2(asum / (double)F))) : 1.0;
    std::vector<uint32_t> coff(n + 1), off32(n + 1);  // face offsets in the caller's and the internal order
    for (int64_t c = 0; c <= n; c++) coff[c] = (uint32_t)off[c];
    off32[0] = 0;
    for (int64_t i = 0; i < n; i++) off32[i + 1] = off32[i] + (coff[s->inv[i] + 1] - coff[s->inv[i]]);
    const int L = s->p.num_timestep_levels;
    const size_t DN = (size_t)s->D * n;
    TRY(dalloc(s, &s->d_off, n + 1));
    TRY(dalloc(s, &s->d_geo, F));
    TRY(dalloc(s, &s->d_nk, F));
    TRY(dalloc(s, &s->d_vol, n));
    TRY(dalloc(s, &s->d_size, n));
    TRY(dalloc(s, &s->d_pslot, n));
    TRY(dalloc(s, &s->d_level, n));
    {
        // the caller's faces go through a staging buffer, at most what the
        // schedule's build takes later, as many cells at a time as fit
        constexpr size_t kFace = 24 + 8 + 4 + 1;
        const size_t cap = std::max<size_t>(1 << 20, 16 * DN) / kFace, room = std::min<size_t>(cap, F) + 8;
        uint8_t *stage = nullptr, *tmp = nullptr;
        uint32_t* d_coff = nullptr;
        uint64_t *pcount = nullptr, *psum = nullptr;
        unsigned long long* bad = nullptr;
        Defer cleanup{[&] {
            dfree(s, stage);
            dfree(s, tmp);
            dfree(s, d_coff);
            dfree(s, pcount);
            dfree(s, psum);
            dfree(s, bad);
        }};
        TRY(dalloc(s, &stage, std::max<size_t>(room * kFace, n * sizeof(double))));
        TRY(dalloc(s, &d_coff, n + 1));
        TRY(dalloc(s, &pcount, n + 1));
        TRY(dalloc(s, &psum, n + 1));
        TRY(dalloc(s, &bad, 1));
        HIP_TRY(hipMemcpyAsync(s->d_off, off32.data(), (n + 1) * 4, hipMemcpyHostToDevice, s->stream));
        HIP_TRY(hipMemcpyAsync(d_coff, coff.data(), (n + 1) * 4, hipMemcpyHostToDevice, s->stream));
        HIP_TRY(hipMemsetAsync(bad, 0xFF, 8, s->stream));
        HIP_TRY(hipMemsetAsync(pcount + n, 0, 8, s->stream));
        HIP_TRY(hipMemsetAsync(s->d_level, L - 1, n, s->stream));
        TRY(upload_cells(s, volume, (double*)stage, s->d_vol));
        TRY(upload_cells(s, size, (double*)stage, s->d_size));
        double* const sn = (double*)stage;
        double* const sarea = sn + 3 * room;
        int32_t* const sb = (int32_t*)(sarea + room);
        uint8_t* const sk = (uint8_t*)(sb + room);
        for (int64_t c0 = 0; c0 < n;) {
            const int64_t f0 = off[c0];
            // the last cell whose faces all fit (a cell has at most 127, a chunk holds more)
            const int64_t c1 = std::upper_bound(off + c0, off + n + 1, f0 + (int64_t)room) - off - 1;
            const int64_t m = off[c1] - f0;
            if (m > 0) {
                HIP_TRY(hipMemcpyAsync(sn, normal + 3 * f0, m * 24, hipMemcpyHostToDevice, s->stream));
                HIP_TRY(hipMemcpyAsync(sarea, area + f0, m * 8, hipMemcpyHostToDevice, s->stream));
                HIP_TRY(hipMemcpyAsync(sb, nbr + f0, m * 4, hipMemcpyHostToDevice, s->stream));
                HIP_TRY(hipMemcpyAsync(sk, kind + f0, m, hipMemcpyHostToDevice, s->stream));
            }
            k_pack_faces<<<grid_for(16 * (c1 - c0)), kBlock, 0, s->stream>>>(
                d_coff, (uint32_t)c0, (uint32_t)c1, (uint32_t)f0, sn, sarea, sb, sk, s->permuted ? s->d_perm : nullptr,
                s->d_off, s->p.periodic ? 1 : 0, (uint32_t)n, s->d_geo, s->d_nk, pcount, bad);
            HIP_TRY(hipGetLastError());
            c0 = c1;
        }
        size_t tb = 0;
        HIP_TRY(hipcub::DeviceScan::ExclusiveSum(nullptr, tb, pcount, psum, (int)n + 1, s->stream));
        TRY(dalloc(s, &tmp, tb));
        HIP_TRY(hipcub::DeviceScan::ExclusiveSum(tmp, tb, pcount, psum, (int)n + 1, s->stream));
        unsigned long long hbad = 0;
        uint64_t total = 0;
        HIP_TRY(hipMemcpyAsync(&hbad, bad, 8, hipMemcpyDeviceToHost, s->stream));
        HIP_TRY(hipMemcpyAsync(&total, psum + n, 8, hipMemcpyDeviceToHost, s->stream));
        HIP_TRY(hipStreamSynchronize(s->stream));
        if (hbad != ~0ull) {
            free_grid(s);
            return fail(SSW_ERR_INVALID, (hbad & 1ull) ? "face_neighbour out of range" : "face_kind must be 0, 1 or 2");
        }
        s->Nper = (int64_t)(total >> 32);
        const size_t pf = (size_t)(total & 0xFFFFFFFFull);
        TRY(dalloc(s, &s->d_pcells, std::max<int64_t>(1, s->Nper)));
        TRY(dalloc(s, &s->d_pfoff, s->Nper + 1));
        TRY(dalloc(s, &s->d_pnb, std::max<size_t>(1, pf)));
        TRY(dalloc(s, &s->d_pgeo, std::max<size_t>(1, pf)));
        k_pack_periodic<<<grid_for(n + 1), kBlock, 0, s->stream>>>(pcount, psum, s->d_off, s->d_geo, s->d_nk,
                                                                   (uint32_t)n, s->d_pslot, s->d_pcells, s->d_pfoff,
                                                                   s->d_pgeo, s->d_pnb);
        HIP_TRY(hipGetLastError());
        s->h_pcells.resize(s->Nper);
        if (s->Nper)
            HIP_TRY(hipMemcpyAsync(s->h_pcells.data(), s->d_pcells, s->Nper * 4, hipMemcpyDeviceToHost, s->stream));
        HIP_TRY(hipStreamSynchronize(s->stream));
    }
    TRY(dalloc(s, &s->d_cnt, DN));
    TRY(build_direction_graph(s, true));
    s->have_grid = true;
    return SSW_OK;
}

int ssw_upload_state(ssw_sweep* s, const double* density, const double* xhii, const double* temp,
                     const double* source) {
    if (!s || !density || !xhii || !temp || !source) return fail(SSW_ERR_INVALID, "null argument");
    if (!s->have_grid) return fail(SSW_ERR_INVALID, "ssw_upload_grid must be called first");
    drop_all_lists(s);
    s->have_state = false;
    dfree(s, s->d_offI);
    dfree(s, s->d_offP);
    const int64_t n = s->N;
    const int L = s->p.num_timestep_levels;
    std::vector<double> sod(n);
    double lmax = 0.0;
    s->rates_current = false;
    s->nonneg = s->x_nonneg = true;
    for (int64_t c = 0; c < n; c++) {
        if (!(source[c] >= 0.0)) s->nonneg = false;
        sod[c] = source[c] / (double)s->D;  // Site::source_per_direction_bin
        lmax = std::max(lmax, std::fabs(sod[c]));
    }
    // FP32 transport carries rates in units of a power of two near the largest
    // source per direction bin (photon rates reach 1e52 s^-1, above FP32 range).
    s->lref = (s->fp32 && lmax > 0.0) ? std::ldexp(1.0, (int)std::lround(std::log2(lmax))) : 1.0;
    const size_t es = real_size(s);
    // the buffers of the grid's last state are kept, their sizes are the grid's
    // (1000 cells x 16 directions: 0.17 ms a call when they were allocated anew
    // and freed, 0.095 like this)
    auto keep = [](ssw_sweep* h, auto** p, size_t count) -> int { return *p ? SSW_OK : dalloc(h, p, count); };
    TRY(keep(s, &s->d_rho, n));
    TRY(keep(s, &s->d_x, n));
    TRY(keep(s, &s->d_T, n));
    TRY(keep(s, &s->d_src, n));
    TRY(keep(s, (uint8_t**)&s->d_sa, n * sa_size(s)));
    TRY(keep(s, &s->d_sts, n));
    TRY(keep(s, &s->d_prev, n));
    TRY(keep(s, &s->d_rate, n));
    TRY(keep(s, &s->d_change, n));
    TRY(keep(s, &s->d_chemq, (size_t)n + 2));
    TRY(keep(s, (uint8_t**)&s->d_X, (size_t)s->D * n * es));
    TRY(keep(s, (uint8_t**)&s->d_I, (size_t)s->D * n * es));
    if (s->Nper) TRY(keep(s, (uint8_t**)&s->d_P, (size_t)s->D * s->Nper * es));
    TRY(upload_cells(s, density, s->d_sts, s->d_rho));
    TRY(upload_cells(s, xhii, s->d_sts, s->d_x));
    TRY(upload_cells(s, temp, s->d_sts, s->d_T));
    TRY(upload_cells(s, sod.data(), s->d_sts, s->d_src));
    HIP_TRY(hipMemsetAsync(s->d_sts, 0, n * 8, s->stream));
    HIP_TRY(hipMemsetAsync(s->d_prev, 0, n * 8, s->stream));
    HIP_TRY(hipMemsetAsync(s->d_change, 0, n * 8, s->stream));
    HIP_TRY(hipMemsetAsync(s->d_X, 0, (size_t)s->D * n * es, s->stream));
    HIP_TRY(hipMemsetAsync(s->d_I, 0, (size_t)s->D * n * es, s->stream));
    if (s->Nper) HIP_TRY(hipMemsetAsync(s->d_P, 0, (size_t)s->D * s->Nper * es, s->stream));
    HIP_TRY(hipMemsetAsync(s->d_fail, 0, 8, s->stream));
    HIP_TRY(hipMemsetAsync(s->d_active, 0, 32, s->stream));
    HIP_TRY(hipMemsetAsync(s->d_level, L - 1, n, s->stream));  // src/sweep/mod.rs:206
    // the transport reads source/D in its storage scale (FP32: divided by the
    // power of two lref, exact)
    if (s->fp32)
        k_attenuation<float><<<grid_for(n), kBlock, 0, s->stream>>>(s->d_src, s->lref, s->d_rho, s->d_x, s->d_size,
                                                                    (float2*)s->d_sa, n);
    else
        k_attenuation<double><<<grid_for(n), kBlock, 0, s->stream>>>(s->d_src, s->lref, s->d_rho, s->d_x, s->d_size,
                                                                     (double2*)s->d_sa, n);
    HIP_TRY(hipGetLastError());
    TRY(set_need_all(s, 1u));
    HIP_TRY(hipStreamSynchronize(s->stream));
    s->ts.init(s->p.max_timestep, L);
    s->have_state = true;
    return SSW_OK;
}

int ssw_step(ssw_sweep* s, double* elapsed) {
    if (!s) return fail(SSW_ERR_INVALID, "null handle");
    if (!s->have_state) return fail(SSW_ERR_INVALID, "ssw_upload_state must be called first");
    return s->fp32 ? run_step<float>(s, elapsed) : run_step<double>(s, elapsed);
}

int ssw_packed_graph_stats(int64_t* captured, int64_t* replayed) {
    std::lock_guard<std::mutex> lk(g_pack_mu);
    if (captured) *captured = g_pack_captured;
    if (replayed) *replayed = g_pack_replayed;
    return SSW_OK;
}

int ssw_step_batch(ssw_sweep* const* handles, int32_t n, double* elapsed) {
    if (!handles || n < 1) return fail(SSW_ERR_INVALID, "no handles");
    for (int h = 0; h < n; h++) {
        if (!handles[h]) return fail(SSW_ERR_INVALID, "null handle");
        if (!handles[h]->have_state) return fail(SSW_ERR_INVALID, "ssw_upload_state must be called first");
        if (handles[h]->device != handles[0]->device)
            return fail(SSW_ERR_INVALID, "the handles of a packed step must be on one device");
        for (int k = 0; k < h; k++)
            if (handles[k] == handles[h]) return fail(SSW_ERR_INVALID, "a handle appears twice in a packed step");
    }
    return step_batch(handles, n, elapsed);
}

int ssw_rotate_directions(ssw_sweep* s, const double* matrix) {
    if (!s || !matrix) return fail(SSW_ERR_INVALID, "null argument");
    if (!s->have_grid) return fail(SSW_ERR_INVALID, "ssw_upload_grid must be called first");
    for (int k = 0; k < 9; k++)
        if (!std::isfinite(matrix[k])) return fail(SSW_ERR_INVALID, "rotation matrix must be finite");
    expect_frees(s);
    const int64_t n = s->N;
    const size_t DN = (size_t)s->D * n;
    // the rates before the rotation, as the reference's sites hold them
    double *dI = nullptr, *dO = nullptr, *dP = nullptr, *d_kept = nullptr;
    Defer cleanup{[&] {
        for (double** p : {&dI, &dO, &dP, &d_kept}) dfree(s, *p);
    }};
    if (s->have_state) {
        TRY(dalloc(s, &dI, DN));
        TRY(dalloc(s, &dO, DN));
        TRY(dalloc(s, &dP, DN));
        const Geo g = make_geo(s);
        launch_fluxes(s, g, dI, dO, dP);
        HIP_TRY(hipGetLastError());
        HIP_TRY(hipStreamSynchronize(s->stream));
    }
    const std::vector<double> before = s->dirs;
    const std::array<double, 3> dw{s->dw[0], s->dw[1], s->dw[2]};
    const int64_t ovf_total = s->ovf_total;
    std::vector<double> kept;
    rotate_table(matrix, s->dirs, kept);
    // the dependency graph and schedule of the rotated directions
    auto build = [&]() -> int {
        HIP_TRY(hipMemcpyAsync(s->d_dirs, s->dirs.data(), s->dirs.size() * 8, hipMemcpyHostToDevice, s->stream));
        TRY(dalloc(s, &s->d_cnt, DN));
        return build_direction_graph(s, false);
    };
    int rc = build();
    if (rc != SSW_OK && s->have_schedule) {
        // the rotated graph has a cycle, or its layering did not fit: the
        // handle stays as it was
        const std::string why = g_err;
        dfree(s, s->d_cnt);
        dfree(s, s->d_nup);
        s->dirs = before;
        for (int k = 0; k < 3; k++) s->dw[k] = dw[k];
        s->ovf_total = ovf_total;
        HIP_TRY(hipMemcpyAsync(s->d_dirs, s->dirs.data(), s->dirs.size() * 8, hipMemcpyHostToDevice, s->stream));
        HIP_TRY(hipStreamSynchronize(s->stream));
        return fail(rc, why);
    }
    auto turn = [&]() -> int {  // the state with them
        s->rotated = true;
        s->rates_current = false;
        if (s->have_state) {
            TRY(dalloc(s, &d_kept, kept.size()));
            HIP_TRY(hipMemcpyAsync(d_kept, kept.data(), kept.size() * 8, hipMemcpyHostToDevice, s->stream));
            TRY(s->fp32 ? rotate_state_t<float>(s, d_kept, dI, dO, dP) : rotate_state_t<double>(s, d_kept, dI, dO, dP));
            TRY(set_need_all(s, 1u));
        }
        HIP_TRY(hipStreamSynchronize(s->stream));
        return SSW_OK;
    };
    if (rc == SSW_OK) rc = turn();
    if (rc != SSW_OK) {  // no schedule, or a state that is not its own: later calls are refused
        const std::string why = g_err;
        (void)hipStreamSynchronize(s->stream);
        free_state(s);
        free_grid(s);
        s->have_grid = s->have_state = false;
        return fail(rc, why);
    }
    return SSW_OK;
}

int ssw_rotation_matrix(const double* axis, double angle, double* out) {
    if (!axis || !out) return fail(SSW_ERR_INVALID, "null argument");
    // get_rotation_matrix (src/sweep/direction/mod.rs:112-135)
    const double x = axis[0], y = axis[1], z = axis[2];
    const double c = std::cos(angle), sn = std::sin(angle);
    const double m[9] = {c + x * x * (1.0 - c),     x * y * (1.0 - c) - z * sn, x * z * (1.0 - c) + y * sn,
                         y * x * (1.0 - c) + z * sn, c + y * y * (1.0 - c),     y * z * (1.0 - c) - x * sn,
                         z * x * (1.0 - c) - y * sn, z * y * (1.0 - c) + x * sn, c + z * z * (1.0 - c)};
    std::memcpy(out, m, sizeof(m));
    return SSW_OK;
}

int ssw_random_rotation_matrix(double phi, double u, double psi, double* out) {
    if (!out) return fail(SSW_ERR_INVALID, "null argument");
    // get_random_rotation_matrix (src/sweep/direction/mod.rs:137-148) for its
    // three draws: phi in [0, 2 pi), u in [0, 1), psi in [0, 2 pi)
    const double theta = std::acos(2.0 * u - 1.0);
    const double axis[3] = {std::cos(phi) * std::sin(theta), std::sin(phi) * std::sin(theta), std::cos(theta)};
    return ssw_rotation_matrix(axis, psi, out);
}

int ssw_synchronize(ssw_sweep* s) {
    if (!s) return fail(SSW_ERR_INVALID, "null handle");
    HIP_TRY(hipStreamSynchronize(s->stream));
    return SSW_OK;
}

int ssw_download(ssw_sweep* s, double* x, double* T, double* sts, double* photon, uint8_t* level, double* change) {
    if (!s) return fail(SSW_ERR_INVALID, "null handle");
    if (!s->have_state) return fail(SSW_ERR_INVALID, "ssw_upload_state must be called first");
    std::vector<const double*> src;
    std::vector<double*> dst;
    auto want = [&](const double* d, double* h) {
        if (!h) return;
        src.push_back(d);
        dst.push_back(h);
    };
    want(s->d_x, x);
    want(s->d_T, T);
    want(s->d_sts, sts);
    want(s->d_change, change);
    if (photon) {
        if (!s->rates_current && !s->d_photon) TRY(dalloc(s, &s->d_photon, s->N));
        TRY(photon_rates(s, make_geo(s), s->d_photon, nullptr));
        want(s->rates_current ? s->d_rate : s->d_photon, photon);
    }
    return fetch_outputs(s, src, dst, s->d_level, level);
}

int ssw_download_noalloc(ssw_sweep* s, double* x, double* T, double* sts, double* photon, uint8_t* level,
                         double* change) {
    if (!s) return fail(SSW_ERR_INVALID, "null handle");
    if (!s->have_state) return fail(SSW_ERR_INVALID, "ssw_upload_state must be called first");
    const int64_t n = s->N;
    if ((size_t)n * 8 > kNoAllocBytes)
        return fail(SSW_ERR_INVALID, "ssw_download_noalloc: " + std::to_string(n) + " cells exceed its limit of " +
                                         std::to_string(kNoAllocBytes / 8) + " cells (use ssw_download)");
    uint8_t* stage = nullptr;
    TRY(noalloc_scratch(s->device, &stage));
    if (x) TRY(noalloc_out(s, s->d_x, x, stage));
    if (T) TRY(noalloc_out(s, s->d_T, T, stage));
    if (sts) TRY(noalloc_out(s, s->d_sts, sts, stage));
    if (change) TRY(noalloc_out(s, s->d_change, change, stage));
    if (level) TRY(noalloc_out(s, s->d_level, level, stage));
    if (photon) {
        // pulled: the photon rate of every cell lands at its caller index in the staging buffer
        TRY(photon_rates(s, make_geo(s), (double*)stage, s->permuted ? s->d_inv : nullptr));
        if (s->rates_current) TRY(noalloc_out(s, s->d_rate, photon, stage));
        else HIP_TRY(hipMemcpyAsync(photon, stage, (size_t)n * 8, hipMemcpyDeviceToHost, s->stream));
    }
    HIP_TRY(hipStreamSynchronize(s->stream));
    return SSW_OK;
}

int ssw_download_chemistry_outputs(ssw_sweep* s, double* photoionization, double* heating, double* recombination,
                                   double* collisional_ionization) {
    if (!s) return fail(SSW_ERR_INVALID, "null handle");
    if (!s->have_state) return fail(SSW_ERR_INVALID, "ssw_upload_state must be called first");
    const int64_t n = s->N;
    double* outs[4] = {photoionization, heating, recombination, collisional_ionization};
    double* d_out = nullptr;
    Defer cleanup{[&] { dfree(s, d_out); }};
    TRY(dalloc(s, &d_out, 4 * n));
    double* d[4];
    std::vector<const double*> src;
    std::vector<double*> dst;
    for (int k = 0; k < 4; k++) {
        d[k] = outs[k] ? d_out + k * n : nullptr;
        if (!outs[k]) continue;
        src.push_back(d[k]);
        dst.push_back(outs[k]);
    }
    if (src.empty()) return SSW_OK;
    const Geo g = make_geo(s);
    const ChemArgs ca = chem_args(s);
    const unsigned nb = (unsigned)((n + 63) / 64);
    if (s->fp32) k_chem_outputs<float><<<nb, 64, 0, s->stream>>>(g, make_flux<float>(s), ca, d[0], d[1], d[2], d[3]);
    else k_chem_outputs<double><<<nb, 64, 0, s->stream>>>(g, make_flux<double>(s), ca, d[0], d[1], d[2], d[3]);
    HIP_TRY(hipGetLastError());
    return fetch_outputs(s, src, dst, nullptr, nullptr);
}

int ssw_download_counts(ssw_sweep* s, int32_t lvl, uint32_t* counts) {
    if (!s || !counts) return fail(SSW_ERR_INVALID, "null argument");
    if (!s->have_grid) return fail(SSW_ERR_INVALID, "ssw_upload_grid must be called first");
    if (lvl < 0 || lvl >= s->p.num_timestep_levels) return fail(SSW_ERR_INVALID, "sweep_level out of range");
    Defer cleanup{[&] { dfree(s, s->d_cnt); }};
    if (!s->d_cnt) TRY(dalloc(s, &s->d_cnt, (size_t)s->D * s->N));
    const Geo g = make_geo(s);
    k_count<<<grid_for((int64_t)s->N * s->D), kBlock, 0, s->stream>>>(g, lvl);
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipMemcpyAsync(counts, s->d_cnt, (size_t)s->D * s->N * 4, hipMemcpyDeviceToHost, s->stream));
    HIP_TRY(hipStreamSynchronize(s->stream));
    dfree(s, s->d_cnt);
    to_caller(s, counts, s->D);
    return SSW_OK;
}

int ssw_download_levelsets(ssw_sweep* s, int32_t lvl, uint32_t* depth) {
    if (!s || !depth) return fail(SSW_ERR_INVALID, "null argument");
    if (!s->have_grid) return fail(SSW_ERR_INVALID, "ssw_upload_grid must be called first");
    if (lvl < 0 || lvl >= s->p.num_timestep_levels) return fail(SSW_ERR_INVALID, "sweep_level out of range");
    // Kahn layering of the restricted graph (the replay schedule is not touched)
    std::vector<uint8_t> lev(s->N);
    HIP_TRY(hipMemcpyAsync(lev.data(), s->d_level, s->N, hipMemcpyDeviceToHost, s->stream));
    HIP_TRY(hipStreamSynchronize(s->stream));
    int64_t active = 0;
    for (uint8_t v : lev) active += v >= lvl;
    int k = 0;
    uint32_t* d_depth = nullptr;
    Defer cleanup{[&] { dfree(s, d_depth); }};
    const int64_t DN = (int64_t)s->D * s->N;
    TRY(dalloc(s, &d_depth, (size_t)DN));
    k_fill_u32<<<grid_for(DN), kBlock, 0, s->stream>>>(d_depth, kNone, DN);
    TRY(kahn_layering(s, lvl, active * s->D, d_depth, &k, nullptr));
    HIP_TRY(hipMemcpyAsync(depth, d_depth, (size_t)DN * 4, hipMemcpyDeviceToHost, s->stream));
    HIP_TRY(hipStreamSynchronize(s->stream));
    dfree(s, d_depth);
    to_caller(s, depth, s->D);
    return SSW_OK;
}

int ssw_download_fluxes(ssw_sweep* s, double* incoming, double* outgoing, double* periodic) {
    if (!s) return fail(SSW_ERR_INVALID, "null handle");
    if (!s->have_state) return fail(SSW_ERR_INVALID, "ssw_upload_state must be called first");
    const size_t m = (size_t)s->D * s->N;
    double *dI = nullptr, *dO = nullptr, *dP = nullptr;
    Defer cleanup{[&] {
        for (double** p : {&dI, &dO, &dP}) dfree(s, *p);
    }};
    TRY(dalloc(s, &dI, m));
    TRY(dalloc(s, &dO, m));
    TRY(dalloc(s, &dP, m));
    Geo g = make_geo(s);
    launch_fluxes(s, g, dI, dO, dP);
    HIP_TRY(hipGetLastError());
    if (incoming) HIP_TRY(hipMemcpyAsync(incoming, dI, m * 8, hipMemcpyDeviceToHost, s->stream));
    if (outgoing) HIP_TRY(hipMemcpyAsync(outgoing, dO, m * 8, hipMemcpyDeviceToHost, s->stream));
    if (periodic) HIP_TRY(hipMemcpyAsync(periodic, dP, m * 8, hipMemcpyDeviceToHost, s->stream));
    HIP_TRY(hipStreamSynchronize(s->stream));
    dfree(s, dI);
    dfree(s, dO);
    dfree(s, dP);
    if (incoming) to_caller(s, incoming, s->D);
    if (outgoing) to_caller(s, outgoing, s->D);
    if (periodic) to_caller(s, periodic, s->D);
    return SSW_OK;
}

int ssw_download_transport(ssw_sweep* s, void* X, void* I) {
    if (!s) return fail(SSW_ERR_INVALID, "null handle");
    if (!s->have_state) return fail(SSW_ERR_INVALID, "ssw_upload_state must be called first");
    const int64_t DN = (int64_t)s->D * s->N;
    const size_t m = (size_t)DN * real_size(s);
    uint8_t* dtmp = nullptr;
    Defer cleanup{[&] { dfree(s, dtmp); }};
    // X, and in direction sweeps I, is stored in schedule-position order
    auto get = [&](void* out, const void* in, bool ordered) -> int {
        if (!out) return SSW_OK;
        if (ordered) {
            if (!dtmp) TRY(dalloc(s, &dtmp, m));
            if (s->fp32)
                k_gather_x<float><<<grid_for(DN), kBlock, 0, s->stream>>>((const float*)in, s->d_xpos, (float*)dtmp, DN);
            else
                k_gather_x<double><<<grid_for(DN), kBlock, 0, s->stream>>>((const double*)in, s->d_xpos, (double*)dtmp,
                                                                           DN);
            HIP_TRY(hipGetLastError());
            in = dtmp;
        }
        HIP_TRY(hipMemcpyAsync(out, in, m, hipMemcpyDeviceToHost, s->stream));
        return SSW_OK;
    };
    TRY(get(X, s->d_X, s->compiled));
    TRY(get(I, s->d_I, s->d_dirinfo != nullptr));  // into dtmp only after X has left it: stream order
    HIP_TRY(hipStreamSynchronize(s->stream));
    dfree(s, dtmp);
    for (void* a : {X, I}) {
        if (!a) continue;
        if (s->fp32) to_caller(s, (float*)a, s->D);
        else to_caller(s, (double*)a, s->D);
    }
    return SSW_OK;
}

// ---------------------------------------------------------------------------
// checkpoint of the dynamic state (no counterpart in the reference, which
// restarts from snapshots of the ECS components): a header, then per cell in
// the caller's order density, x, T, source per direction, attenuation,
// species timestep, previous rate, change timescale and level, then X and I
// direction-major in the caller's cell order and the periodic sources per
// direction for the periodic cells in increasing caller index, all in the
// storage precision and scale of the transport.

}  // extern "C"

namespace {

struct CkptHeader {
    uint64_t magic;
    uint32_t version, precision;
    int64_t N, Nper;
    int32_t D, L;
    double lref, max_ts;
    int32_t lowest, first_done;
};
constexpr uint64_t kCkptMagic = 0x31544b5057535353ull;  // "SSSWPKT1"

int64_t ckpt_bytes(const ssw_sweep* s) {
    const int64_t n = s->N, DN = (int64_t)s->D * n, rs = (int64_t)real_size(s);
    return (int64_t)sizeof(CkptHeader) + n * 8 * 8 + ((n + 7) / 8) * 8 + 2 * DN * rs + (int64_t)s->D * s->Nper * rs;
}

// Periodic slots ordered by the caller index of their cell.
std::vector<uint32_t> slots_by_caller(const ssw_sweep* s) {
    std::vector<std::pair<uint32_t, uint32_t>> v(s->h_pcells.size());
    for (size_t k = 0; k < v.size(); k++) {
        const uint32_t ci = s->h_pcells[k];
        v[k] = {s->permuted ? s->inv[ci] : ci, (uint32_t)k};
    }
    std::sort(v.begin(), v.end());
    std::vector<uint32_t> out(v.size());
    for (size_t k = 0; k < v.size(); k++) out[k] = v[k].second;
    return out;
}

template <typename R>
int save_t(ssw_sweep* s, uint8_t* buf) {
    const int64_t n = s->N, DN = (int64_t)s->D * n;
    CkptHeader h{kCkptMagic, 1u, (uint32_t)(s->fp32 ? 32 : 64), n, s->Nper, s->D, s->p.num_timestep_levels,
                 s->lref, s->p.max_timestep, s->ts.lowest, s->ts.first_done ? 1 : 0};
    std::memcpy(buf, &h, sizeof(h));
    uint8_t* p = buf + sizeof(h);
    std::vector<double2> sa(n);
    double* cell = reinterpret_cast<double*>(p);
    HIP_TRY(hipMemcpyAsync(cell + 0 * n, s->d_rho, n * 8, hipMemcpyDeviceToHost, s->stream));
    HIP_TRY(hipMemcpyAsync(cell + 1 * n, s->d_x, n * 8, hipMemcpyDeviceToHost, s->stream));
    HIP_TRY(hipMemcpyAsync(cell + 2 * n, s->d_T, n * 8, hipMemcpyDeviceToHost, s->stream));
    HIP_TRY(hipMemcpyAsync(cell + 3 * n, s->d_src, n * 8, hipMemcpyDeviceToHost, s->stream));
    TRY(download_sa(s, sa));
    HIP_TRY(hipMemcpyAsync(cell + 5 * n, s->d_sts, n * 8, hipMemcpyDeviceToHost, s->stream));
    HIP_TRY(hipMemcpyAsync(cell + 6 * n, s->d_prev, n * 8, hipMemcpyDeviceToHost, s->stream));
    HIP_TRY(hipMemcpyAsync(cell + 7 * n, s->d_change, n * 8, hipMemcpyDeviceToHost, s->stream));
    uint8_t* lev = p + n * 8 * 8;
    HIP_TRY(hipMemcpyAsync(lev, s->d_level, n, hipMemcpyDeviceToHost, s->stream));
    R* X = reinterpret_cast<R*>(lev + ((n + 7) / 8) * 8);
    R* I = X + DN;
    R* P = I + DN;
    R* tmp = nullptr;
    Defer cleanup{[&] { dfree(s, tmp); }};
    if (s->compiled) {
        TRY(dalloc(s, &tmp, (size_t)DN));
        k_gather_x<R><<<grid_for(DN), kBlock, 0, s->stream>>>((const R*)s->d_X, s->d_xpos, tmp, DN);
        HIP_TRY(hipGetLastError());
    }
    HIP_TRY(hipMemcpyAsync(X, tmp ? (void*)tmp : s->d_X, DN * sizeof(R), hipMemcpyDeviceToHost, s->stream));
    if (s->d_dirinfo) {  // I in X's order, after the copy of X in stream order
        k_gather_x<R><<<grid_for(DN), kBlock, 0, s->stream>>>((const R*)s->d_I, s->d_xpos, tmp, DN);
        HIP_TRY(hipGetLastError());
    }
    HIP_TRY(hipMemcpyAsync(I, s->d_dirinfo ? (void*)tmp : s->d_I, DN * sizeof(R), hipMemcpyDeviceToHost, s->stream));
    std::vector<R> Pd((size_t)s->D * s->Nper);
    if (s->Nper)
        HIP_TRY(hipMemcpyAsync(Pd.data(), s->d_P, Pd.size() * sizeof(R), hipMemcpyDeviceToHost, s->stream));
    HIP_TRY(hipStreamSynchronize(s->stream));
    dfree(s, tmp);
    for (int64_t c = 0; c < n; c++) cell[4 * n + c] = sa[c].y;
    for (int k = 0; k < 8; k++) to_caller(s, cell + k * n, 1);
    to_caller(s, lev, 1);
    to_caller(s, X, s->D);
    to_caller(s, I, s->D);
    const std::vector<uint32_t> order = slots_by_caller(s);
    for (int d = 0; d < s->D; d++)
        for (size_t j = 0; j < order.size(); j++) P[(size_t)d * s->Nper + j] = Pd[(size_t)d * s->Nper + order[j]];
    return SSW_OK;
}

template <typename R>
int load_t(ssw_sweep* s, const uint8_t* buf) {
    const int64_t n = s->N, DN = (int64_t)s->D * n;
    CkptHeader h;
    std::memcpy(&h, buf, sizeof(h));
    const uint8_t* p = buf + sizeof(h);
    std::vector<double> cell((size_t)n * 8);
    std::memcpy(cell.data(), p, (size_t)n * 8 * 8);
    std::vector<uint8_t> lev(p + n * 8 * 8, p + n * 8 * 9);
    const R* Xc = reinterpret_cast<const R*>(p + n * 8 * 8 + ((n + 7) / 8) * 8);
    std::vector<R> X(Xc, Xc + DN), I(Xc + DN, Xc + 2 * DN);
    const R* Pc = Xc + 2 * DN;
    std::vector<double> tmpc;
    for (int k = 0; k < 8; k++) {
        const double* in = to_internal(s, cell.data() + k * n, tmpc);
        if (in != cell.data() + k * n) std::copy(in, in + n, cell.begin() + k * n);
    }
    {
        std::vector<uint8_t> tl;
        const uint8_t* in = to_internal(s, lev.data(), tl);
        if (in != lev.data()) lev.assign(in, in + n);
    }
    for (int d = 0; d < s->D; d++) {
        std::vector<R> tr;
        const R* inx = to_internal(s, X.data() + (size_t)d * n, tr);
        if (inx != X.data() + (size_t)d * n) std::copy(inx, inx + n, X.begin() + (size_t)d * n);
        const R* ini = to_internal(s, I.data() + (size_t)d * n, tr);
        if (ini != I.data() + (size_t)d * n) std::copy(ini, ini + n, I.begin() + (size_t)d * n);
    }
    const std::vector<uint32_t> order = slots_by_caller(s);
    std::vector<R> Pd((size_t)s->D * s->Nper);
    for (int d = 0; d < s->D; d++)
        for (size_t j = 0; j < order.size(); j++) Pd[(size_t)d * s->Nper + order[j]] = Pc[(size_t)d * s->Nper + j];
    auto negative = [](auto v) { return !(v >= 0); };  // NaN counts
    s->rates_current = s->x_nonneg = false;
    s->nonneg = std::none_of(cell.begin() + 3 * n, cell.begin() + 4 * n, negative) &&
                std::none_of(Pd.begin(), Pd.end(), negative);
    s->lref = h.lref;
    std::vector<double2> sa(n);
    for (int64_t c = 0; c < n; c++)
        sa[c] = make_double2(s->fp32 ? cell[3 * n + c] / s->lref : cell[3 * n + c], cell[4 * n + c]);
    HIP_TRY(hipMemcpyAsync(s->d_rho, cell.data() + 0 * n, n * 8, hipMemcpyHostToDevice, s->stream));
    HIP_TRY(hipMemcpyAsync(s->d_x, cell.data() + 1 * n, n * 8, hipMemcpyHostToDevice, s->stream));
    HIP_TRY(hipMemcpyAsync(s->d_T, cell.data() + 2 * n, n * 8, hipMemcpyHostToDevice, s->stream));
    HIP_TRY(hipMemcpyAsync(s->d_src, cell.data() + 3 * n, n * 8, hipMemcpyHostToDevice, s->stream));
    TRY(upload_sa(s, sa));
    HIP_TRY(hipMemcpyAsync(s->d_sts, cell.data() + 5 * n, n * 8, hipMemcpyHostToDevice, s->stream));
    HIP_TRY(hipMemcpyAsync(s->d_prev, cell.data() + 6 * n, n * 8, hipMemcpyHostToDevice, s->stream));
    HIP_TRY(hipMemcpyAsync(s->d_change, cell.data() + 7 * n, n * 8, hipMemcpyHostToDevice, s->stream));
    HIP_TRY(hipMemcpyAsync(s->d_level, lev.data(), n, hipMemcpyHostToDevice, s->stream));
    R* tmp = nullptr;
    Defer cleanup{[&] { dfree(s, tmp); }};
    if (s->compiled) {
        TRY(dalloc(s, &tmp, (size_t)DN));
        HIP_TRY(hipMemcpyAsync(tmp, X.data(), DN * sizeof(R), hipMemcpyHostToDevice, s->stream));
        k_scatter_x<R><<<grid_for(DN), kBlock, 0, s->stream>>>((R*)s->d_X, s->d_xpos, tmp, DN);
        HIP_TRY(hipGetLastError());
    } else {
        HIP_TRY(hipMemcpyAsync(s->d_X, X.data(), DN * sizeof(R), hipMemcpyHostToDevice, s->stream));
    }
    if (s->d_dirinfo) {  // I in X's order
        HIP_TRY(hipMemcpyAsync(tmp, I.data(), DN * sizeof(R), hipMemcpyHostToDevice, s->stream));
        k_scatter_x<R><<<grid_for(DN), kBlock, 0, s->stream>>>((R*)s->d_I, s->d_xpos, tmp, DN);
        HIP_TRY(hipGetLastError());
    } else {
        HIP_TRY(hipMemcpyAsync(s->d_I, I.data(), DN * sizeof(R), hipMemcpyHostToDevice, s->stream));
    }
    if (s->Nper)
        HIP_TRY(hipMemcpyAsync(s->d_P, Pd.data(), Pd.size() * sizeof(R), hipMemcpyHostToDevice, s->stream));
    HIP_TRY(hipStreamSynchronize(s->stream));
    dfree(s, tmp);
    s->ts.lowest = h.lowest;
    s->ts.first_done = h.first_done != 0;
    drop_all_lists(s);
    TRY(set_need_all(s, 1u));
    HIP_TRY(hipStreamSynchronize(s->stream));
    return SSW_OK;
}

}  // namespace

extern "C" {

int64_t ssw_checkpoint_bytes(ssw_sweep* s) {
    if (!s || !s->have_state) return 0;
    return ckpt_bytes(s);
}

int ssw_save_checkpoint(ssw_sweep* s, void* buf, int64_t bytes) {
    if (!s || !buf) return fail(SSW_ERR_INVALID, "null argument");
    if (!s->have_state) return fail(SSW_ERR_INVALID, "ssw_upload_state must be called first");
    if (bytes < ckpt_bytes(s)) return fail(SSW_ERR_INVALID, "checkpoint buffer too small");
    if (s->rotated) return fail(SSW_ERR_INVALID, "checkpoints of a handle with rotated directions are not supported");
    return s->fp32 ? save_t<float>(s, (uint8_t*)buf) : save_t<double>(s, (uint8_t*)buf);
}

int ssw_load_checkpoint(ssw_sweep* s, const void* buf, int64_t bytes) {
    if (!s || !buf) return fail(SSW_ERR_INVALID, "null argument");
    if (!s->have_state) return fail(SSW_ERR_INVALID, "ssw_upload_state must be called first");
    if (bytes < (int64_t)sizeof(CkptHeader)) return fail(SSW_ERR_INVALID, "checkpoint too small");
    if (s->rotated) return fail(SSW_ERR_INVALID, "checkpoints of a handle with rotated directions are not supported");
    CkptHeader h;
    std::memcpy(&h, buf, sizeof(h));
    if (h.magic != kCkptMagic || h.version != 1u) return fail(SSW_ERR_INVALID, "not a checkpoint of this library");
    if (h.N != s->N || h.D != s->D || h.L != s->p.num_timestep_levels || h.Nper != s->Nper ||
        h.precision != (uint32_t)(s->fp32 ? 32 : 64) || h.max_ts != s->p.max_timestep)
        return fail(SSW_ERR_INVALID, "checkpoint of a different problem (cells, directions, levels, periodic "
                                     "cells, precision or maximum timestep differ)");
    if (bytes < ckpt_bytes(s)) return fail(SSW_ERR_INVALID, "checkpoint truncated");
    return s->fp32 ? load_t<float>(s, (const uint8_t*)buf) : load_t<double>(s, (const uint8_t*)buf);
}

extern "C++" {
namespace {
// Workgroups of the grouped replay kernel one CU holds at once (0 if unknown),
// for the group of the most cones.
template <typename R>
int group_blocks_per_cu(const ssw_sweep* s) {
    const ssw_sweep::Group* most = &s->groups[0];
    for (const ssw_sweep::Group& gr : s->groups)
        if (gr.ndesc > most->ndesc) most = &gr;
    int n = 0;
    const hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(
        &n, SSW_CONE_KERNEL(k_sweep_cone, R, most->waves, false), 64 * most->waves,
        ConeShape<R>::bytes(most->waves, most->words));
    return e == hipSuccess ? n : 0;
}
}  // namespace
}

int ssw_get_info(ssw_sweep* s, ssw_info* info) {
    if (!s || !info) return fail(SSW_ERR_INVALID, "null argument");
    std::memset(info, 0, sizeof(*info));
    info->num_cells = s->N;
    info->num_faces = s->F;
    info->num_directions = s->D;
    info->max_depth = s->kmax;
    info->sweeps_last_step = s->sweeps_last;
    info->downwind_local = s->dw[0];
    info->downwind_periodic = s->dw[1];
    info->downwind_boundary = s->dw[2];
    info->device_bytes = s->bytes;
    info->peak_device_bytes = s->peak_bytes;
    info->transport_mode = s->have_grid ? (s->compiled ? SSW_TRANSPORT_MODE_COMPILED : SSW_TRANSPORT_MODE_GEOMETRIC)
                                        : s->mode_request;
    info->list_builds_last_step = (int32_t)s->builds_last;
    info->overflow_entries = s->ovf_total;
    info->graph_capture_failures = s->capture_failures;
    info->replay_block = s->rec_block;
    info->graph_replay = s->graphs_on ? 1 : 0;
    info->narrow_runs = (s->compiled && s->narrow_runs) ? 1 : 0;
    info->direction_sweeps = s->d_dirinfo ? 1 : 0;
    info->group_levels = s->groups.empty() ? 1 : s->group_request;
    info->group_fallback = s->group_fallback ? 1 : 0;
    info->group_tasks = s->group_tasks;
    info->group_block = s->group_block;
    if (!s->groups.empty()) {
        info->group_launches = (int64_t)s->groups.size();
        for (const ssw_sweep::Group& gr : s->groups) info->group_workgroups += gr.ndesc;
        info->group_blocks_per_cu =
            s->fp32 ? group_blocks_per_cu<float>(s) : group_blocks_per_cu<double>(s);
    }
    {
        int cus = 0;
        if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, s->device) == hipSuccess)
            info->compute_units = cus;
    }
    info->locality_order = s->permuted ? 1 : 0;
    if (s->have_state) {
        unsigned long long f = 0, a = 0, lim[3] = {0, 0, 0};
        HIP_TRY(hipMemcpyAsync(&f, s->d_fail, 8, hipMemcpyDeviceToHost, s->stream));
        HIP_TRY(hipMemcpyAsync(&a, s->d_active, 8, hipMemcpyDeviceToHost, s->stream));
        HIP_TRY(hipMemcpyAsync(lim, s->d_active + 1, 24, hipMemcpyDeviceToHost, s->stream));
        HIP_TRY(hipStreamSynchronize(s->stream));
        info->chemistry_failures = (int64_t)f;
        info->updates_last_step = (int64_t)a * s->D;
        info->limiting_temperature = (int64_t)lim[0];
        info->limiting_ionization_fraction = (int64_t)lim[1];
        info->limiting_photon_rate = (int64_t)lim[2];
    }
    return SSW_OK;
}

int32_t ssw_timestep_level(int32_t num_levels, double max_timestep, double desired_timestep) {
    if (num_levels < 1) return 0;
    return ssw::level_from_ratio(max_timestep / desired_timestep, num_levels);
}

double ssw_chemistry_timestep(double* state, double density, double volume, double length, double rate,
                              double scale_factor, int32_t prevent_cooling, double timestep, double safety,
                              int32_t* process, int32_t* failed) {
    ssw::Cell c;
    c.x = state[0];
    c.T = state[1];
    c.rho = density;
    c.vol = volume;
    c.len = length;
    c.rate = rate;
    c.a = scale_factor;
    ssw::Floor f{prevent_cooling != 0, c.T, c.x};
    int proc = 0;
    bool fl = false;
    double ts = ssw::perform_timestep(c, f, timestep, safety, proc, fl);
    state[0] = c.x;
    state[1] = c.T;
    if (process) *process = proc;
    if (failed) *failed = fl ? 1 : 0;
    return ts;
}

int64_t ssw_estimate_device_bytes(const ssw_sweep_parameters* p, int64_t n, int64_t F, int64_t num_periodic_cells,
                                  int32_t mode) {
    if (!p || n <= 0) return 0;
    // compiled: the default launch shape
    return ssw::handle_bytes(memory_problem(*p, n, F, num_periodic_cells), mode == SSW_TRANSPORT_MODE_COMPILED
                                                                               ? ssw::Replay::kGrouped
                                                                               : ssw::Replay::kGeometric);
}

int ssw_set_timing(ssw_sweep* s, int32_t enabled) {
    if (!s) return fail(SSW_ERR_INVALID, "null handle");
    s->timing = enabled != 0;
    return SSW_OK;
}

int ssw_get_timing(ssw_sweep* s, double* avg, double* total, int64_t* launches, double* chem, double* build) {
    if (!s) return fail(SSW_ERR_INVALID, "null handle");
    if (avg) *avg = s->n_transport ? s->t_transport_total / (double)s->n_transport : 0.0;
    if (total) *total = s->t_transport_total;
    if (launches) *launches = s->n_transport;
    if (chem) *chem = s->t_chem_total;
    if (build) *build = s->t_build_total;
    return SSW_OK;
}

}  // extern "C"
