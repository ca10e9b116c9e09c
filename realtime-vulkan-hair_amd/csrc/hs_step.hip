// hs_step.hip - the step kernels (k_step, k_step_batch) for one tile shape.
//
// A tile shape is the workgroup's strands (kW) and the points of one segment
// of the root-to-tip walk (kL); kThreads threads share a segment's points.
//
// What bounds it: with one lane per strand the kernel ran 1.5 wavefronts per
// SIMD at 100,000 strands and fewer below, and waited on its own dependent
// chains.  Now only the follow-the-leader recurrence is walked one lane per
// strand (28 instructions a point, a seventh of the step); the rest has four
// threads per strand at 128 x 16 and two at the 256-strand shapes, 4
// wavefronts per SIMD.  Measured (before -> after, exports included): 8 steps
// of 100,000 x 32, 128 x 16, 1,029 -> 838 us; 4 steps of 37,501 x 57, 256 x 8,
// 857 -> 555 us; one step of eight grooms of 512-2,048 strands 300 -> 208 us;
// 4 steps of 1,000,000 x 64 with the head mesh, 256 x 8, 19.3 -> 16.1 ms.  It
// issues 27.6M vector instructions a step at 100,000 x 32 (47 us at one per 4
// cycles); the rest is LDS time (same-address atomics of dense hair),
// barriers and load latency.
//
// This file is compiled once per shape the library offers, each build in its own
// namespace (HS_SHAPE_NS) with HS_TILE_STRANDS / HS_TILE_POINTS set; results
// are the same bits for every shape, only the speed differs.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "hs_device.hpp"

#ifndef HS_TILE_STRANDS
#define HS_TILE_STRANDS 128
#endif
#ifndef HS_TILE_POINTS
#define HS_TILE_POINTS 16
#endif
#ifndef HS_SHAPE_NS
#define HS_SHAPE_NS t128x16
#endif

namespace hs {
namespace HS_SHAPE_NS {

constexpr uint32_t kW = HS_TILE_STRANDS;  // strands per step workgroup
constexpr uint32_t kL = HS_TILE_POINTS;   // points per segment of the root-to-tip sweep
#ifndef HS_TILE_THREADS
#define HS_TILE_THREADS 512
#endif
// Threads per workgroup: 512 put two workgroups (16 wavefronts) on a CU, what
// 128 registers and the LDS allow.
constexpr uint32_t kThreads = HS_TILE_THREADS;
constexpr uint32_t kQ = kThreads / kW;          // threads per strand
constexpr uint32_t kT = kL / kQ;                // points of a segment per thread
// Most windows a segment's box is splatted through; more goes to device
// atomics.  A window costs a workgroup about 6-10 us, whatever the rest of the
// device does; device atomics reach 27 G/s over the whole device, 2.7 us per
// segment, and with every workgroup of a 900-strand groom using them beyond 4
// windows its step measured 100 us against 85.
constexpr int kMaxChunks = 32;
constexpr uint32_t kMaxSegments = (256 - 1 + kL - 1) / kL;  // of the longest strand
constexpr uint32_t kR = 64 / kQ;                // strands per wavefront
constexpr uint32_t kStage = 1;                  // gather-window cells a thread loads ahead of their segment
static_assert(kQ * kW == kThreads && kQ * kT == kL && kQ >= 2 && kThreads <= 1024, "whole points per thread");
static_assert(kQ * kR == 64, "a wavefront holds all threads of its strands");
static_assert(kT >= 2, "a thread's first position slot is reused to hand its last point on");

static_assert((uint64_t)kW * (kL + 1) * 1000000ull < (1ull << 32),
              "packed (vx<<32 | density) LDS sums need the density of one window below 2^32");
static_assert(kW % 64 == 0, "workgroup is whole wavefronts");
static_assert(kW % kLeafStrands == 0, "a workgroup is whole k-d leaves");
static_assert(kW <= kMaxTileStrands, "the strand planes are padded to kMaxTileStrands");
static_assert(kL <= 31, "per-point flags live in one 32-bit mask");

// ---------------------------------------------------------------------------
// Workgroup reductions and window planning
// ---------------------------------------------------------------------------

// Minimum over the wavefront (every lane active): DPP steps within each row
// of 16 lanes (VALU moves, no LDS traffic), then the four row results.
__device__ __forceinline__ int wave_min(int v)
{
    v = min(v, __builtin_amdgcn_update_dpp(v, v, 0xB1, 0xF, 0xF, false));   // quad_perm [1,0,3,2]
    v = min(v, __builtin_amdgcn_update_dpp(v, v, 0x4E, 0xF, 0xF, false));   // quad_perm [2,3,0,1]
    v = min(v, __builtin_amdgcn_update_dpp(v, v, 0x141, 0xF, 0xF, false));  // row_half_mirror
    v = min(v, __builtin_amdgcn_update_dpp(v, v, 0x140, 0xF, 0xF, false));  // row_mirror
    return min(min(__builtin_amdgcn_readlane(v, 0), __builtin_amdgcn_readlane(v, 16)),
               min(__builtin_amdgcn_readlane(v, 32), __builtin_amdgcn_readlane(v, 48)));
}

// Box of voxels (inclusive bounds).  Empty: lo = INT_MAX, hi = INT_MIN.
struct Box {
    int lo[3], hi[3];
};

// Grows the box by the bounds of a range.
__device__ __forceinline__ void box_add(Box& b, const Rng& r)
{
    b.lo[0] = min(b.lo[0], r.x0);
    b.hi[0] = max(b.hi[0], r.x1);
    b.lo[1] = min(b.lo[1], r.y0);
    b.hi[1] = max(b.hi[1], r.y1);
    b.lo[2] = min(b.lo[2], r.z0);
    b.hi[2] = max(b.hi[2], r.z1);
}

__device__ __forceinline__ Box box_empty()
{
    Box b;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        b.lo[k] = INT32_MAX;
        b.hi[k] = INT32_MIN;
    }
    return b;
}

__device__ __forceinline__ bool box_is_empty(const Box& b)
{
    return b.lo[0] > b.hi[0] || b.lo[1] > b.hi[1] || b.lo[2] > b.hi[2];
}

// Joins every lane's box into the workgroup's `bx` (lo, then -hi; INT_MAX when
// empty): a wavefront minimum per bound, then one LDS minimum per wavefront.
// The result is there after the next barrier.
__device__ __forceinline__ void block_box_min(const Box& b, int* bx)
{
    int v[6];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        v[k] = wave_min(b.lo[k]);
        v[3 + k] = wave_min(b.hi[k] == INT32_MIN ? INT32_MAX : -b.hi[k]);
    }
    if ((threadIdx.x & 63) == 0) {
#pragma unroll
        for (int k = 0; k < 6; ++k) atomicMin(bx + k, v[k]);
    }
}

// Column of strand sl's point t in the position array: threads of one strand
// (kR lanes apart, kT points apart) are shifted against each other so that a
// wavefront's lanes fall on different banks.
__device__ __forceinline__ uint32_t pn_at(uint32_t t, uint32_t sl)
{
    return t * 3 * kW + ((sl + kR * (t / kT)) & (kW - 1));
}

// Three-component values of one strand in an LDS array laid out [..][x y z][kW].
__device__ __forceinline__ f3 ld_lds(const float* p) { return mk(p[0], p[kW], p[2 * kW]); }
__device__ __forceinline__ void st_lds(float* p, f3 v)
{
    p[0] = v.x;
    p[kW] = v.y;
    p[2 * kW] = v.z;
}

// Chunking of a box into LDS windows of at most `cap` voxels: full x extent,
// chunks in y and z overlapping by one voxel so that every 2x2x2 block of the
// box lies whole inside at least one chunk.
struct Plan {
    int ex, ey, ez;   // box extents
    int cy, cz;       // chunk extents in y and z (cells)
    int ny, nz;       // chunk counts
    bool ok;          // false: no chunking fits (or empty box)
};

__device__ __forceinline__ Plan plan_box(const Box& b, int cap)
{
    Plan p;
    if (box_is_empty(b)) {
        p.ex = p.ey = p.ez = 0;
        p.cy = p.cz = 2;
        p.ny = p.nz = 0;
        p.ok = false;
        return p;
    }
    p.ex = b.hi[0] - b.lo[0] + 1;
    p.ey = b.hi[1] - b.lo[1] + 1;
    p.ez = b.hi[2] - b.lo[2] + 1;
    p.ok = true;
    p.cy = p.ey;
    p.cz = p.ez;
    p.ny = p.nz = 1;
    if (p.ex * p.ey * p.ez <= cap) return p;  // one window
    if (p.ex * p.ey * 2 <= cap) {
        p.cy = p.ey;
        p.cz = cap / (p.ex * p.ey);
    } else if (p.ex * 4 <= cap) {
        p.cz = 2;
        p.cy = cap / (p.ex * 2);
    } else {
        p.ok = false;
        p.cy = p.cz = 2;
    }
    p.ny = p.cy >= p.ey ? 1 : 1 + (p.ey - 2) / (p.cy - 1);
    p.nz = p.cz >= p.ez ? 1 : 1 + (p.ez - 2) / (p.cz - 1);
    return p;
}

__device__ __forceinline__ Win chunk_of(const Box& b, const Plan& p, int iy, int iz)
{
    Win w;
    w.x0 = b.lo[0];
    w.ex = p.ex;
    w.y0 = b.lo[1] + iy * (p.cy - 1);
    w.z0 = b.lo[2] + iz * (p.cz - 1);
    w.ey = min(p.cy, b.hi[1] - w.y0 + 1);
    w.ez = min(p.cz, b.hi[2] - w.z0 + 1);
    return w;
}

// ---------------------------------------------------------------------------
// Partial boxes: an LDS window is summed over its copies and dumped into the
// pool, and its box is listed with every reduce brick it overlaps.
// ---------------------------------------------------------------------------
// A workgroup-segment's own box goes to its own pool slot and descriptor (no
// allocator); further windows to the shared part, taken with atomics.
// Every thread of the workgroup calls these after the window is complete.

// Lists box cw, descriptor di, with every brick it overlaps: one device atomic
// each, in parallel.  `meanwhile` runs between a thread's first atomic and the
// use of its result.  Brick indices come from bit fields (x and y extents
// rounded up to powers of two): no divisions.
template <class F>
__device__ __forceinline__ void list_box(const StepArgs& a, const Win& cw, uint32_t di, F&& meanwhile)
{
    const int bx0 = cw.x0 / (int)kBX, by0 = cw.y0 / (int)kBY, bz0 = cw.z0 / (int)kBZ;
    const int nbx = (cw.x0 + cw.ex - 1) / (int)kBX - bx0 + 1;
    const int nby = (cw.y0 + cw.ey - 1) / (int)kBY - by0 + 1;
    const int nbz = (cw.z0 + cw.ez - 1) / (int)kBZ - bz0 + 1;
    const uint32_t half = a.parity * (a.gw.nbx * a.gw.nby * a.gw.nbz);
    const int lx = 32 - __clz(nbx - 1), ly = 32 - __clz(nby - 1);
    const int n = nbz << (lx + ly);
    auto brick = [&](int t, uint32_t& b) {
        const int ix = t & ((1 << lx) - 1), iy = (t >> lx) & ((1 << ly) - 1), iz = t >> (lx + ly);
        b = half + ((uint32_t)(bz0 + iz) * a.gw.nby + (uint32_t)(by0 + iy)) * a.gw.nbx + (uint32_t)(bx0 + ix);
        return (t < n) & (ix < nbx) & (iy < nby);
    };
    auto enter = [&](uint32_t b, uint32_t at) {
        if (at < kBrickList) a.gw.brick_list[(size_t)b * kBrickList + at] = di;
    };
    uint32_t b, at = 0;
    const bool mine = brick((int)threadIdx.x, b);
    if (mine) at = atomicAdd(a.gw.brick_cnt + b, 1u);
    meanwhile();
    if (mine) enter(b, at);
    for (int t = (int)(threadIdx.x + kThreads); t < n; t += (int)kThreads)
        if (brick(t, b)) enter(b, atomicAdd(a.gw.brick_cnt + b, 1u));
}

__device__ __forceinline__ void write_desc(const StepArgs& a, const Win& cw, uint32_t di, uint32_t off, bool fits)
{
    int4* d = reinterpret_cast<int4*>(a.gw.desc + ((size_t)a.parity * a.gw.desc_cap + di) * kDescInts);
    d[0] = make_int4(cw.x0, cw.y0, cw.z0, fits ? cw.ex : 0);  // ex == 0: empty descriptor
    d[1] = make_int4(cw.ey, cw.ez, (int)off, 0);
}

// store(c, cell) for every cell of the window, its copies summed.
template <class F>
__device__ __forceinline__ void each_cell(const int4* win, int cells, int nc, F&& store)
{
    auto all = [&](auto n) {
        for (int c = threadIdx.x; c < cells; c += kThreads) store(c, splat_sum<decltype(n)::value>(win, c));
    };
    switch (nc) {
    case 1: all(std::integral_constant<int, 1>{}); break;
    case 2: all(std::integral_constant<int, 2>{}); break;
    case 4: all(std::integral_constant<int, 4>{}); break;
    case 8: all(std::integral_constant<int, 8>{}); break;
    default: all(std::integral_constant<int, 16>{}); break;
    }
}
static_assert(kMaxCopies == 16, "each_cell handles 1, 2, 4, 8 and 16 copies");

// The window of workgroup-segment ws, into its own slot and descriptor.
__device__ __forceinline__ void dump_own(const StepArgs& a, const Win& cw, int cells, int nc, uint32_t ws, const int4* win)
{
    const uint32_t off = ws * kSlotCells;
    if (threadIdx.x == kThreads - 1) write_desc(a, cw, ws, off, true);
    int4* dst = a.gw.pool + (size_t)a.parity * a.gw.pool_cap + off;
    list_box(a, cw, ws, [&] { each_cell(win, cells, nc, [&](int c, int4 cell) { dst[c] = cell; }); });
}

// One window of several, into the shared part of the pool.
__device__ __forceinline__ void dump_shared(const StepArgs& a, const Win& cw, int cells, int nc, const int4* win, uint32_t* bcast)
{
    uint32_t* ctr = a.gw.counters + a.parity * 4;
    if (threadIdx.x == 0) {
        const uint32_t off = a.gw.nws * kSlotCells + atomicAdd(ctr + 0, (uint32_t)cells);
        const uint32_t di = a.gw.nws + atomicAdd(ctr + 1, 1u);
        const bool fits = (uint64_t)off + cells <= a.gw.pool_cap && di < a.gw.desc_cap;
        if (di < a.gw.desc_cap) write_desc(a, cw, di, off, fits);
        if (!fits) atomicOr(ctr + 2, kOverflowUsed | kFellBack);
        bcast[0] = off;
        bcast[1] = fits ? 1u : 0u;
        bcast[2] = di;
    }
    __syncthreads();
    const uint32_t off = bcast[0];
    const bool fits = bcast[1] != 0;
    const int G = (int)a.G;
    if (fits) list_box(a, cw, bcast[2], [] {});
    int4* dst = a.gw.pool + (size_t)a.parity * a.gw.pool_cap + off;
    each_cell(win, cells, nc, [&](int c, int4 cell) {
        if (fits) {
            dst[c] = cell;
        } else if (cell.x | cell.y | cell.z | cell.w) {
            // no room in the pool: device atomics into the overflow grid
            const int ax = c % cw.ex;
            const int rest = c / cw.ex;
            const size_t gi = (size_t)(cw.x0 + ax) + (size_t)(cw.y0 + rest % cw.ey) * G +
                              (size_t)(cw.z0 + rest / cw.ey) * G * G;
            int* gcell = reinterpret_cast<int*>(a.gw.overflow + gi);
            atomicAdd(gcell + 0, cell.x);
            atomicAdd(gcell + 1, cell.y);
            atomicAdd(gcell + 2, cell.z);
            atomicAdd(gcell + 3, cell.w);
        }
    });
    __syncthreads();
}

// ---------------------------------------------------------------------------
// Boxes of several windows
// ---------------------------------------------------------------------------
// Whether chunk (iy, iz) takes a point of this range: the chunk whose y/z
// range starts at or before its block and reaches past it (chunk starts step
// by window size - 1, so that is the quotient).  Each point goes to exactly
// one chunk, and integer voxel sums commute: the grid is the one a window
// without limits would give.
__device__ __forceinline__ bool in_chunk(const Rng& r, const Box& b, const Plan& p, int iy, int iz)
{
    const int jy = p.ny > 1 ? min(p.ny - 1, (r.y0 - b.lo[1]) / (p.cy - 1)) : 0;
    const int jz = p.nz > 1 ? min(p.nz - 1, (r.z0 - b.lo[2]) / (p.cz - 1)) : 0;
    return jy == iy && jz == iz;
}

// Chunk c of workgroup-segment (wg, sg), whose box takes several windows: zero
// the window, splat the segment's finished (stored) points whose blocks fall
// in this chunk, dump.
__device__ __forceinline__ void splat_chunk(const StepArgs& a, uint32_t wg, uint32_t sg, const Box& box, const Plan& pl, int c,
                                            int4* win, uint32_t* bcast)
{
    const int iy = c % pl.ny, iz = c / pl.ny;
    const Win cw = chunk_of(box, pl, iy, iz);
    const int cells = cw.ex * cw.ey * cw.ez;
    const SplatLane sl = splat_lane(cells);
    for (uint32_t e = threadIdx.x; e < kWinCells; e += kThreads) win[e] = make_int4(0, 0, 0, 0);
    __syncthreads();
    const uint32_t s = wg * kW + threadIdx.x % kW;
    const uint32_t q = threadIdx.x / kW;  // every kQ-th point from q on
    const uint32_t N = a.N, Sp = a.Sp;
    const uint32_t f = 1 + sg * kL;
    const uint32_t cnt = min(kL, N - f);
    const bool last_seg = f + cnt == N;
    if (s < a.S) {
        const uint32_t P4 = N * Sp * 4u, P8 = N * Sp * 8u;
        const f3 origin = mk(a.ox, a.oy, a.oz);
        // finished points of the segment: f-1 (carried), f..f+cnt-2, and the
        // tip; four at a time, their loads in flight together
        const uint32_t i0 = (f >= 2 ? f - 1 : f) + q;
        const uint32_t i1 = last_seg ? f + cnt - 1 : f + cnt - 2;
        constexpr uint32_t kGrp = 4;
#pragma unroll 1
        for (uint32_t g0 = i0; g0 <= i1; g0 += kGrp * kQ) {
        f3 XP[kGrp], VP[kGrp];
#pragma unroll
        for (uint32_t t = 0; t < kGrp; ++t) {
            if (g0 + t * kQ > i1) continue;
            const uint32_t bo = ((g0 + t * kQ) * Sp + s) * 4u;
            XP[t] = ld3(a.pos, bo, P4, P8);
            VP[t] = ld3(a.vel, bo, P4, P8);
        }
#pragma unroll
        for (uint32_t t = 0; t < kGrp; ++t) {
            if (g0 + t * kQ > i1) continue;
            const f3 x = XP[t];
            const f3 v = VP[t];
            const f3 q = grid_coord(x, origin, a.inv_h);
            const Rng rg = point_range(q, (int)a.G);
            if (rng_empty(rg)) continue;
            if (!in_chunk(rg, box, pl, iy, iz)) continue;
            Loc l;
            if (locate(q, cw, l))
                splat_block(win, cw, l, q, v, sl);
            else
                splat_any(win, cw, true, sl, a.gw.overflow, rg, q, v, (int)a.G);
        }
        }
    }
    __syncthreads();
    dump_shared(a, cw, cells, sl.nc, win, bcast);
}

// ---------------------------------------------------------------------------
// The step kernel
// ---------------------------------------------------------------------------
// XCD-aware order: dispatch places consecutive blockIdx on different XCDs
// (round robin over 8); give each XCD a contiguous run of logical workgroups
// (Morton-ordered strand blocks) so neighbouring windows share that XCD's L2.
__device__ __forceinline__ uint32_t xcd_swizzle(uint32_t block, uint32_t nblocks)
{
    const uint32_t per = (nblocks + 7) / 8;
    return (block % 8) * per + block / 8;
}

// The launch's arguments live in constant memory (the kernel-argument segment,
// or the batch's argument blob).  Held across the whole step they cost more
// scalar registers than there are, and the compiler keeps the excess in VGPR
// lanes, read back one v_readlane at a time; so each phase loads the fields it
// uses again (scalar loads, cached) through a pointer the compiler cannot see
// through.
using ArgsPtr = const __attribute__((address_space(4))) StepArgs*;
__device__ __forceinline__ StepArgs fresh_args(ArgsPtr p)
{
    asm volatile("" : "+s"(p));
    return global_args(*(const StepArgs*)p);
}

// One workgroup's share of a step: strands [wg*kW, wg*kW + kW) of the groom,
// kQ threads per strand.  Only the follow-the-leader chain is serial along the
// strand: the first kW threads walk it over predicted positions in LDS, and
// everything else (gather, force and prediction; velocities and corrections;
// splat) is done by a strand's kQ threads for kT points each.
template <bool GATHER, bool SPLAT, int COL>
__device__ __forceinline__ void step_body(ArgsPtr args, uint32_t wg)
{
    __shared__ __align__(16) int4 win[kWinCells];
    __shared__ float pn[3 * kL * kW];  // predicted, then new positions of the segment: [point][x y z][strand]
    __shared__ float carry[6 * kW];    // last point of the previous segment: position, velocity before DFTL
    __shared__ int bx[2][6];           // the segment's voxel box (lo, -hi), by segment parity
    __shared__ uint32_t bcast[3];
    __shared__ int big[kMaxSegments][7];  // boxes (lo, hi) and segments that take several windows
    if (SPLAT && threadIdx.x < 12) bx[threadIdx.x / 6][threadIdx.x % 6] = INT32_MAX;

    // A wavefront takes kR strands, all kQ threads of each: its lanes are then
    // at kQ places along the strands, several voxels apart, and fewer of them
    // meet in one voxel than with 64 neighbouring strands at one place.
    const uint32_t q = (threadIdx.x & 63u) / kR;
    const uint32_t sl = (threadIdx.x >> 6) * kR + threadIdx.x % kR;
    const uint32_t t0 = q * kT;  // this thread's first point of a segment
    const uint32_t s = wg * kW + sl;
    const uint32_t S = args->S, Sp = args->Sp, N = args->N, nseg = args->nseg;
    const bool active = s < S;
    const uint32_t plane = N * Sp;
    // byte offsets into the [3][N][Sp] arrays stay below 2^32 (checked on the
    // host), so every access is an SGPR base plus a 32-bit VGPR offset
    const uint32_t P4 = plane * 4u, P8 = plane * 8u;
    const uint32_t bS = Sp * 4u;  // byte stride between points

    f3 X[kT], U[kT];      // position and velocity; the velocity becomes the prediction, then the new velocity
    float4 cell[kStage];  // the gather window's first cells, on their way to LDS
    // The voxel window the previous step recorded for segment sg, if it fits
    // in LDS.  Read as constants (scalar loads): this step's own box replaces
    // it only after the segment's last use of it.
    auto gather_window = [&](const StepArgs& a, uint32_t sg, Win& w) {
        if (!GATHER) return false;
        const __attribute__((address_space(4))) int* gb =
            (const __attribute__((address_space(4))) int*)(uintptr_t)(a.gw.gbox + ((size_t)wg * nseg + sg) * 6);
        w = Win{gb[0], gb[1], gb[2], gb[3] - gb[0] + 1, gb[4] - gb[1] + 1, gb[5] - gb[2] + 1};
        // (after a change of tile shape the boxes are laid out for the old
        // shape: the points then gather straight from the float grid)
        return a.gbox_ok && gb[0] <= gb[3] && gb[1] <= gb[4] && gb[2] <= gb[5] &&
               w.ex * w.ey * w.ez <= (int)min(a.win_gather, kWinCells);
    };
    auto window_cell = [&](const StepArgs& a, const Win& gwin, int c) {
        // cell c's row and plane: (c + 1/2) / ex is at least 1/(2 ex) away from
        // any integer and c < 2^12, so the reciprocal's rounding cannot carry
        // the quotient past one
        const uint32_t ex = (uint32_t)gwin.ex, ey = (uint32_t)gwin.ey, G = a.G;
        const float rx = __builtin_amdgcn_rcpf((float)ex), ry = __builtin_amdgcn_rcpf((float)ey);
        const uint32_t cc = (uint32_t)min(c, gwin.ex * gwin.ey * gwin.ez - 1);  // clamped: loads are unconditional
        const uint32_t rest = (uint32_t)(((float)cc + 0.5f) * rx);
        const uint32_t az = (uint32_t)(((float)rest + 0.5f) * ry);
        const uint32_t ax = cc - __umul24(rest, ex), ay = rest - __umul24(az, ey);
        const uint32_t at = (uint32_t)gwin.x0 + ax + ((uint32_t)gwin.y0 + ay) * G + ((uint32_t)gwin.z0 + az) * (G * G);
        return a.gw.grid_f[at];
    };
    // Starts segment sg's loads: its points, and the first cells of the voxel
    // window the previous step recorded for it.
    auto load_segment = [&](const StepArgs& a, uint32_t sg) {
        const uint32_t f = 1 + sg * kL;
        const uint32_t cnt = min(kL, N - f);
        const uint32_t b0 = ((f + t0) * Sp + s) * 4u;
#pragma unroll
        for (uint32_t u = 0; u < kT; ++u) {
            X[u] = mk(0.0f, 0.0f, 0.0f);
            U[u] = mk(0.0f, 0.0f, 0.0f);
            if (active & (t0 + u < cnt)) {
                X[u] = ld3(a.pos, b0 + u * bS, P4, P8);
                U[u] = ld3(a.vel, b0 + u * bS, P4, P8);
            }
        }
        Win gwin;
        if (gather_window(a, sg, gwin)) {
#pragma unroll
            for (uint32_t k = 0; k < kStage; ++k) cell[k] = window_cell(a, gwin, (int)(k * kThreads + threadIdx.x));
        }
    };

    // the first kW threads walk the chain of strand threadIdx.x: its last
    // position and rest length
    const uint32_t cs = wg * kW + threadIdx.x;
    const bool chain = threadIdx.x < kW && cs < S;
    f3 par = mk(0.0f, 0.0f, 0.0f);
    float r = 0.0f;
    f3 fs;
    {
        const StepArgs a = fresh_args(args);
        load_segment(a, 0);
        if (chain) {
            par = ld3(a.pos, cs * 4u, P4, P8);
            r = a.seg[cs];
        }
        fs = mk(a.fx, a.fy, a.fz);
        if (active && a.noise) fs = add(fs, smul(a.noise[s], mk(a.ndx, a.ndy, a.ndz)));
    }

    uint32_t n_big = 0;  // this workgroup's segments of several windows
    for (uint32_t sg = 0; sg < nseg; ++sg) {
        const uint32_t f = 1 + sg * kL;
        const uint32_t cnt = min(kL, N - f);
        const bool last_seg = f + cnt == N;
        const uint32_t b0 = ((f + t0) * Sp + s) * 4u;  // byte offset of this thread's first point
        {
            const StepArgs a = fresh_args(args);
            const f3 origin = mk(a.ox, a.oy, a.oz);
            // ---------------- G: the previous step's voxel window, into LDS ----------------
            Win gwin{0, 0, 0, 0, 0, 0};
            const bool gwin_ok = gather_window(a, sg, gwin);
            if (gwin_ok) {
                const int cells = gwin.ex * gwin.ey * gwin.ez;
                float4* fw = reinterpret_cast<float4*>(win);
#pragma unroll
                for (uint32_t k = 0; k < kStage; ++k) {
                    const int c = (int)(k * kThreads + threadIdx.x);
                    if (c < cells) fw[c] = cell[k];
                }
                for (int c = (int)(kStage * kThreads + threadIdx.x); c < cells; c += (int)kThreads)
                    fw[c] = window_cell(a, gwin, c);
                __syncthreads();
            }

            // ------- P: friction, force and predicted position of every point -------
            // Previous step's phase 3 (compute.comp:257-298) for each point: from
            // the LDS window, or (a workgroup whose box exceeds any window)
            // straight from the float grid, the 8 cells of a block loaded together.
            auto predict = [&](uint32_t u, f3 gv) {
                const f3 x = X[u];
                f3 v = U[u];
                if (GATHER) v = friction(v, gv, a.mu_prev, a.omu_prev);
                // predict (compute.comp:187)
                float4 mf = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
                if (COL & kColMesh) mf = a.mesh_f[(size_t)(f + t0 + u) * Sp + s];
                const f3 fc = force_at<COL>(x, fs, a, mf);
                U[u] = add(add(x, smul(a.dt, v)), smul(a.dt2, fc));
                st_lds(pn + pn_at(t0 + u, sl), U[u]);
            };
            if (active) {
                if (!GATHER || gwin_ok) {
#pragma unroll
                    for (uint32_t u = 0; u < kT; ++u) {
                        if (t0 + u >= cnt) continue;
                        f3 gv = mk(0.0f, 0.0f, 0.0f);
                        if (GATHER) {
                            const f3 qc = grid_coord(X[u], origin, a.inv_h);
                            Loc l;
                            if (locate(qc, gwin, l)) {
                                gv = gather_block(reinterpret_cast<const float4*>(win), gwin, l, qc);
                            } else {
                                const Rng rg = point_range(qc, (int)a.G);
                                if (!rng_empty(rg))
                                    gv = gather_any(reinterpret_cast<const float4*>(win), gwin, in_win(rg, gwin),
                                                    a.gw.grid_f, rg, qc, (int)a.G);
                            }
                        }
                        predict(u, gv);
                    }
                } else {
#pragma unroll
                    for (uint32_t u = 0; u < kT; ++u) {
                        if (t0 + u >= cnt) continue;
                        predict(u, gather_grid(a.gw.grid_f, (int)a.G, grid_coord(X[u], origin, a.inv_h)));
                    }
                }
            }
        }
        __syncthreads();  // predictions stored; the window is no longer read

        // ---------------- F: follow the leader (compute.comp:191-192), root to tip ----------------
        if (threadIdx.x < kW) {
            if (chain) {
#pragma unroll
                for (uint32_t t = 0; t < kL; ++t) {
                    if (t >= cnt) continue;
                    float* at = pn + pn_at(t, threadIdx.x);
                    par = add(par, smul(r, normalize(sub(ld_lds(at), par))));
                    st_lds(at, par);
                }
            }
        } else if (SPLAT) {
            // meanwhile the other wavefronts clear the splat window
            for (uint32_t c = threadIdx.x - kW; c < kWinCells; c += kThreads - kW) win[c] = make_int4(0, 0, 0, 0);
        }
        __syncthreads();

        const StepArgs a = fresh_args(args);
        const f3 origin = mk(a.ox, a.oy, a.oz);
        const int G = (int)a.G;
        float* __restrict__ posb = a.pos;
        float* __restrict__ velb = a.vel;
        // ------- V: damped velocity, clamp, correction (compute.comp:195-201) -------
        // Voxels of the segment's new positions, which the next step's gather
        // needs, and of the carried point, which this segment's splat takes.
        // (One box for both: two cost a second reduction over the workgroup,
        // 48 instructions per wavefront and segment, and measured 2-3% slower.)
        Box box = box_empty();
        // hi gathers the upper bounds less one (a full block's lower corner); the one is added below
        auto box_point = [&](f3 x) {
            const f3 qc = grid_coord(x, origin, a.inv_h);
            const int ix = sat_i32(floorf(qc.x)), iy = sat_i32(floorf(qc.y)), iz = sat_i32(floorf(qc.z));
            const uint32_t g1 = (uint32_t)(G - 1);  // a full block's lower corner is in [0, G-2] on every axis
            if (((uint32_t)ix < g1) & ((uint32_t)iy < g1) & ((uint32_t)iz < g1)) {
                box_add(box, Rng{ix, ix, iy, iy, iz, iz});
            } else {
                const Rng rn = point_range(qc, G);
                if (!rng_empty(rn)) box_add(box, Rng{rn.x0, rn.x1 - 1, rn.y0, rn.y1 - 1, rn.z0, rn.z1 - 1});
            }
        };
        f3 dc[kT];  // what each point's correction takes from its predecessor's velocity
#pragma unroll
        for (uint32_t u = 0; u < kT; ++u) {
            dc[u] = mk(0.0f, 0.0f, 0.0f);
            if (!(active & (t0 + u < cnt))) continue;
            const uint32_t bo = b0 + u * bS;
            const f3 x = X[u];
            const f3 p = ld_lds(pn + pn_at(t0 + u, sl));
            // dot > vmax2 is exactly sqrt(dot) > vmax
            f3 vel = smul(a.D, muls(sub(p, x), a.inv_dt));
            if (dot(vel, vel) > a.vmax2) vel = muls(normalize(vel), a.vmax);
            const f3 corr = smul(a.D, sub(p, U[u]));
            st3(posb, bo, P4, P8, p);
            if (a.corr) st3(a.corr, bo, P4, P8, corr);
            dc[u] = muls(corr, a.inv_dt);
            X[u] = p;
            U[u] = vel;
            if (SPLAT) box_point(p);
        }
        // A thread finishes the point before its first one (its predecessor's
        // last, or the carried one: their correction is that of the thread's
        // first point) and all its points but the last.
        const bool has_prev = active & (q > 0 ? t0 - 1 < cnt : sg > 0);
        f3 xp = mk(0.0f, 0.0f, 0.0f), vp = mk(0.0f, 0.0f, 0.0f);
        if (has_prev) {
            if (q > 0) {
                xp = ld_lds(pn + pn_at(t0 - 1, sl));
            } else {
                xp = ld_lds(carry + sl);
                vp = ld_lds(carry + 3 * kW + sl);
            }
        }
        // handed on in this thread's own first slot, which only it has read
        if (active) st_lds(pn + pn_at(t0, sl), U[kT - 1]);
        // the tip of a segment that the strand fills has no thread after it
        const bool full_tip = last_seg & (cnt == kL);
        if (SPLAT) {
            if (has_prev && q == 0) box_point(xp);
            block_box_min(box, bx[sg & 1]);
        }
        __syncthreads();

        // ------- DFTL of every point whose successor is known (compute.comp:211-215) -------
        if (has_prev) {
            if (q > 0) vp = ld_lds(pn + pn_at(t0 - kT, sl));
            if (t0 < cnt) vp = sub(vp, dc[0]);  // (the tip has no correction, compute.comp:213)
            st3(velb, b0 - bS, P4, P8, vp);
        }
        if (active) {
            if (q == kQ - 1 && !last_seg) {
                st_lds(carry + sl, X[kT - 1]);
                st_lds(carry + 3 * kW + sl, U[kT - 1]);
            }
#pragma unroll
            for (uint32_t u = 0; u < kT; ++u) {
                if (u + 1 < kT) {
                    if (t0 + u + 1 < cnt) U[u] = sub(U[u], dc[u + 1 < kT ? u + 1 : u]);
                    if (t0 + u < cnt) st3(velb, b0 + u * bS, P4, P8, U[u]);
                } else if (full_tip && q == kQ - 1) {
                    st3(velb, b0 + u * bS, P4, P8, U[u]);
                }
            }
        }

        if (!SPLAT) {
            __syncthreads();  // handed-on points read before the next segment's predictions
            if (!last_seg) load_segment(fresh_args(args), sg + 1);
            continue;
        }
        // ---------------- S: splat of the finished points ----------------
        // finished: point f-1 (carried), points f..f+cnt-2, and the tip
        Box ub;
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            ub.lo[k] = __builtin_amdgcn_readfirstlane(bx[sg & 1][k]);
            const int h = __builtin_amdgcn_readfirstlane(bx[sg & 1][3 + k]);
            ub.hi[k] = h == INT32_MAX ? INT32_MIN : 1 - h;
        }
        if (threadIdx.x < 6) {
            bx[(sg & 1) ^ 1][threadIdx.x] = INT32_MAX;  // last read before the barrier above
            const int v = bx[sg & 1][threadIdx.x];
            a.gw.gbox[((size_t)wg * nseg + sg) * 6 + threadIdx.x] =
                threadIdx.x < 3 ? v : (v == INT32_MAX ? INT32_MIN : 1 - v);
        }
        const Plan pl = plan_box(ub, min((int)a.win_splat, (int)kWinCells));
        const int chunks = pl.ny * pl.nz;
        const uint32_t ws = wg * nseg + sg;
        // every finished point of this thread
        auto each_finished = [&](auto&& splat) {
            if (has_prev) splat(xp, vp);
#pragma unroll
            for (uint32_t u = 0; u < kT; ++u) {
                const bool done = u + 1 < kT ? t0 + u < cnt : full_tip && q == kQ - 1;
                if (active & done) splat(X[u], U[u]);
            }
        };
        const bool one_window = pl.ok && chunks == 1;
        // A box larger than one window takes one pass over the segment's
        // points per chunk, from the positions and velocities just stored, or
        // device atomics when they are more than kMaxChunks.
        const bool windows = pl.ok && chunks <= kMaxChunks;
        const Win cw{ub.lo[0], ub.lo[1], ub.lo[2], pl.ex, pl.ey, pl.ez};
        const int cells = pl.ex * pl.ey * pl.ez;
        const SplatLane sp = splat_lane(one_window ? cells : (int)kWinCells);
        if (one_window) {
            // the whole box in one window (cleared during F)
            each_finished([&](f3 x, f3 v) {
                const f3 qc = grid_coord(x, origin, a.inv_h);
                Loc l;
                if (locate(qc, cw, l)) {
                    splat_block(win, cw, l, qc, v, sp);
                } else {
                    const Rng rg = point_range(qc, G);
                    if (!rng_empty(rg)) splat_any(win, cw, true, sp, a.gw.overflow, rg, qc, v, G);
                }
            });
        } else if (!box_is_empty(ub)) {
            if (threadIdx.x == 0) atomicAdd(a.gw.counters + a.parity * 4 + 3, 1u);
            if (windows) {
                // kept for the end, where no segment's registers are live
                if (threadIdx.x < 6)
                    big[n_big][threadIdx.x] = threadIdx.x < 3 ? ub.lo[threadIdx.x] : ub.hi[threadIdx.x - 3];
                if (threadIdx.x == 6) big[n_big][6] = (int)sg;
                ++n_big;
            } else {
                // device atomics into the overflow grid
                each_finished([&](f3 x, f3 v) {
                    const f3 qc = grid_coord(x, origin, a.inv_h);
                    const Rng rg = point_range(qc, G);
                    if (!rng_empty(rg)) splat_any(win, cw, false, sp, a.gw.overflow, rg, qc, v, G);
                });
                if (threadIdx.x == 0) atomicOr(a.gw.counters + a.parity * 4 + 2, pl.ok ? kOverflowUsed : kOverflowUsed | kFellBack);
            }
        }
        __syncthreads();  // window complete; handed-on points read
        if (!last_seg) load_segment(fresh_args(args), sg + 1);
        if (one_window) {
            dump_own(a, cw, cells, sp.nc, ws, win);
            __syncthreads();
        } else if (threadIdx.x == 0) {
            // the slot's descriptor from two steps ago must not be read
            a.gw.desc[((size_t)a.parity * a.gw.desc_cap + ws) * kDescInts + 3] = 0;
        }
    }
    if (SPLAT && n_big > 0) {
        __threadfence_block();  // this workgroup's stored positions and velocities
        __syncthreads();
        const StepArgs a = fresh_args(args);
#pragma unroll 1
        for (uint32_t i = 0; i < n_big; ++i) {
            Box b;
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                b.lo[k] = __builtin_amdgcn_readfirstlane(big[i][k]);
                b.hi[k] = __builtin_amdgcn_readfirstlane(big[i][3 + k]);
            }
            const uint32_t sg = __builtin_amdgcn_readfirstlane(big[i][6]);
            const Plan pl = plan_box(b, min((int)a.win_splat, (int)kWinCells));
#pragma unroll 1
            for (int c = 0; c < pl.ny * pl.nz; ++c) splat_chunk(a, wg, sg, b, pl, c, win, bcast);
        }
    }
}

// Wavefronts per SIMD the compiler budgets registers for: two workgroups per
// CU, which the LDS holds.
constexpr int kStepWaves = 2 * kThreads / 256;

template <bool GATHER, bool SPLAT, int COL>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(kStepWaves))) void k_step(StepArgs a)
{
    const uint32_t wg = a.swz ? xcd_swizzle(blockIdx.x, a.nwg) : blockIdx.x;
    if (wg >= a.nwg) return;
    // `a` is the only by-value struct: it starts the kernel-argument segment
    step_body<GATHER, SPLAT, COL>((ArgsPtr)__builtin_amdgcn_kernarg_segment_ptr(), wg);
}

template <bool GATHER, bool SPLAT, int COL>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(kStepWaves))) void k_step_batch(const StepArgs* __restrict__ args,
                                                   const uint32_t* __restrict__ wg_start, uint32_t ngroom,
                                                   uint32_t swz)
{
    const uint32_t total = wg_start[ngroom];
    const uint32_t gwg = swz ? xcd_swizzle(blockIdx.x, total) : blockIdx.x;
    if (gwg >= total) return;
    const uint32_t g = find_groom(wg_start, ngroom, gwg);
    step_body<GATHER, SPLAT, COL>((ArgsPtr)(uintptr_t)(args + __builtin_amdgcn_readfirstlane(g)), gwg - wg_start[g]);
}

// ---------------------------------------------------------------------------
// Host-side launchers
// ---------------------------------------------------------------------------
template <bool G, bool S>
static void launch_step_e(const StepArgs& a, int col, uint32_t blocks, hipStream_t st)
{
    switch (col) {
    case 0: hipLaunchKernelGGL((k_step<G, S, 0>), dim3(blocks), dim3(kThreads), 0, st, a); break;
    case kColEll: hipLaunchKernelGGL((k_step<G, S, kColEll>), dim3(blocks), dim3(kThreads), 0, st, a); break;
    case kColMesh: hipLaunchKernelGGL((k_step<G, S, kColMesh>), dim3(blocks), dim3(kThreads), 0, st, a); break;
    default:
        hipLaunchKernelGGL((k_step<G, S, kColEll | kColMesh>), dim3(blocks), dim3(kThreads), 0, st, a);
        break;
    }
}

hipError_t launch_step(const StepArgs& a, bool gather, bool splat, hipStream_t st)
{
    const uint32_t blocks = ((a.nwg + 7) / 8) * 8;
    if (a.mesh.tris && !a.mesh_f) return hipErrorInvalidValue;
    const int col = (a.ncol > 1 ? kColEll : 0) | (a.mesh.tris ? kColMesh : 0);
    if (gather) {
        if (splat)
            launch_step_e<true, true>(a, col, blocks, st);
        else
            launch_step_e<true, false>(a, col, blocks, st);
    } else {
        if (splat)
            launch_step_e<false, true>(a, col, blocks, st);
        else
            launch_step_e<false, false>(a, col, blocks, st);
    }
    return hipGetLastError();
}

template <bool G, bool S>
static void launch_batch_e(const StepArgs* args, const uint32_t* wg_start, uint32_t ngroom, int col,
                           uint32_t swz, uint32_t blocks, hipStream_t st)
{
    switch (col) {
    case 0:
        hipLaunchKernelGGL((k_step_batch<G, S, 0>), dim3(blocks), dim3(kThreads), 0, st, args, wg_start, ngroom, swz);
        break;
    case kColEll:
        hipLaunchKernelGGL((k_step_batch<G, S, kColEll>), dim3(blocks), dim3(kThreads), 0, st, args, wg_start, ngroom, swz);
        break;
    case kColMesh:
        hipLaunchKernelGGL((k_step_batch<G, S, kColMesh>), dim3(blocks), dim3(kThreads), 0, st, args, wg_start, ngroom, swz);
        break;
    default:
        hipLaunchKernelGGL((k_step_batch<G, S, kColEll | kColMesh>), dim3(blocks), dim3(kThreads), 0, st, args, wg_start,
                           ngroom, swz);
        break;
    }
}

hipError_t launch_step_batch(const StepArgs* args_dev, const uint32_t* wg_start_dev, uint32_t ngroom,
                             uint32_t total_wg, bool gather, bool splat, int col, uint32_t swz, hipStream_t st)
{
    const uint32_t blocks = ((total_wg + 7) / 8) * 8;
    if (gather) {
        if (splat)
            launch_batch_e<true, true>(args_dev, wg_start_dev, ngroom, col, swz, blocks, st);
        else
            launch_batch_e<true, false>(args_dev, wg_start_dev, ngroom, col, swz, blocks, st);
    } else {
        if (splat)
            launch_batch_e<false, true>(args_dev, wg_start_dev, ngroom, col, swz, blocks, st);
        else
            launch_batch_e<false, false>(args_dev, wg_start_dev, ngroom, col, swz, blocks, st);
    }
    return hipGetLastError();
}

}  // namespace HS_SHAPE_NS
}  // namespace hs
