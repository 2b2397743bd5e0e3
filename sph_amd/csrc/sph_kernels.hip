// sph_kernels.hip - gfx950 kernels of the TinySPH step (AdamSimpson/SPH).
//
// Data layout: one SoA particle array in HBM, kept sorted by (cell, id)
// after every hash, with paired fields interleaved (pos = (x, y),
// vel = (v_x, v_y), prev = (x_prev, y_prev), rho = (density,
// density_near)) so a gather reads a pair with one 8-byte load.
//
// Physics kernels are gathers over the 3x3 cells around each particle's
// cell.  A workgroup owns 256 consecutive sorted particles; their
// candidates are at most six contiguous ranges of the sorted arrays (three
// rows around each of the one or two cell rows the group touches), which
// the group stages into LDS with coalesced loads before each particle walks
// its own candidates in canonical order (rows ascending, sorted order within
// a row).  A group whose tile would not fit (it spans more than two cell
// rows, or the staged ranges exceed the tile) reads the same candidates from
// global memory in the same order, so both paths give identical results.
// No kernel writes another particle's state: no atomics on particle data.
//
// The cell sort is a counting sort: the producing kernel computes each
// particle's new key and claims a slot in its cell with an atomic counter;
// a two-kernel scan turns counts into cell starts (and clears the counts
// for the next sort); a scatter drops (id, source) pairs into the cell
// ranges; the reorder kernel ranks each particle by id inside its cell and
// gathers its fields there - the canonical (cell, id) order of
// src/hash.c:153-163.  In a small context one kernel does all that follows the
// claims (k_sort_small).
//
// Several independent scenes can share one launch: each scene owns a
// 256-aligned range of slots of the sorted arrays and a range of global
// cells (plus a padding cell that takes the slack of its slot range in the
// sort), so a workgroup always belongs to exactly one scene and reads that
// scene's parameters as uniform values (BS maps workgroup -> scene).
//
// Workgroups are numbered XCD-aware: the hardware deals workgroups to the
// 8 XCDs round-robin, and logical tiles are remapped so that each XCD takes
// runs of 16 consecutive tiles (which share candidate rows in its L2), the
// runs dealt to the XCDs in turn.  Whole eighths per XCD would keep more rows
// in one L2, but the work per tile follows the fluid's density, which varies
// with height: in a settling column the densest eighth costs twice the mean,
// and that XCD would finish last.
#include "sph_kernels.h"

#include <hip/hip_ext.h>

#include <type_traits>

namespace {

constexpr int kWave = 64;
constexpr int kTPB = 256;
// The gathers ask the compiler for at least 6 resident workgroups per CU
// (6 waves per SIMD, at most 80 VGPRs): it then schedules them in 67-80
// VGPRs without scratch, where left alone it took 72-84 (5-6 waves).  LDS
// tiles allow 7 workgroups.  Measured on the 1M dam break at steps 221-230:
// density -2%, relaxation -4%, the capped variants -3 to -7%, viscosity
// unchanged.  The capped relaxation asks for 5 (86-94 VGPRs): with 6 its
// uncommon-pair path spills 60 bytes, and the capped 513k-particle dam break
// takes 11.89 ms for 64 steps and their download against 11.59.
// The four-lanes-per-particle variants (contexts of at most two tiles per
// CU, so at most eight of their 64-particle workgroups per CU) set no bound:
// their 66-87 VGPRs still allow 5-7 waves per SIMD, without scratch; nor do
// the sixteen-lane ones (35-64 VGPRs).
constexpr int kGatherMinBlocks = 6;
#ifndef SPH_TILE_CAP
#define SPH_TILE_CAP 1280
#endif
constexpr int kTileCap = SPH_TILE_CAP; // staged candidates per workgroup
constexpr unsigned kXcds = 8;
#ifndef SPH_XCD_CHUNK
#define SPH_XCD_CHUNK 16
#endif
constexpr unsigned kXcdChunk = SPH_XCD_CHUNK; // consecutive tiles per XCD run

__device__ __forceinline__ unsigned wave_max_u32(unsigned v)
{
#pragma unroll
    for (int o = kWave / 2; o > 0; o >>= 1)
        v = max(v, (unsigned)__shfl_xor((int)v, o, kWave));
    return v;
}

__device__ __forceinline__ unsigned wave_sum_u32(unsigned v)
{
#pragma unroll
    for (int o = kWave / 2; o > 0; o >>= 1)
        v += (unsigned)__shfl_xor((int)v, o, kWave);
    return v;
}

__device__ __forceinline__ bool lane0() { return (threadIdx.x & (kWave - 1)) == 0; }

// Logical workgroup index: runs of kXcdChunk consecutive tiles go to one
// XCD, and consecutive runs to consecutive XCDs.
// `skip` workgroups (a multiple of the XCDs) before them do something else.
__device__ __forceinline__ unsigned xcd_block(unsigned skip = 0)
{
    const unsigned b = blockIdx.x - skip, nb = gridDim.x - skip;
    const unsigned full = nb / (kXcds * kXcdChunk) * (kXcds * kXcdChunk);
    if (b >= full)
        return b; // the last, partial round keeps dispatch order
    const unsigned xcd = b % kXcds, local = b / kXcds;
    return ((local / kXcdChunk) * kXcds + xcd) * kXcdChunk + local % kXcdChunk;
}

// Raise a running maximum.  Every wave of a launch reports to the same
// address, so the atomic is issued only when the value would change it:
// same-address atomics serialise in L2, and the maximum settles after the
// first few waves.
__device__ __forceinline__ void raise_max(unsigned long long *p, unsigned long long v)
{
    if (v > *(volatile unsigned long long *)p)
        atomicMax(p, v);
}

// Count-only record of a particle's neighbourhood (overflow guard for the
// reference's 400-slot half lists, and the largest full set seen).
__device__ __forceinline__ void report_neighbors(unsigned full, unsigned half,
                                                 sph_dev_counters *C)
{
    if (half > SPH_REF_MAX_NEIGHBORS)
        atomicAdd(&C->neighbor_overflow, 1ull);
    unsigned m = wave_max_u32(full);
    if (lane0())
        raise_max(&C->max_neighbors, m);
}

// A scene's slot range is padded to whole workgroups; the padding slots are
// counted into the scene's padding cell by its first workgroup, so the
// scan places every scene's particles at its fixed slot offset.
__device__ __forceinline__ void add_pad(const sph_dev_params &P, unsigned s0, unsigned *cnt)
{
    if (threadIdx.x == 0 && s0 == P.poff && P.pad)
        atomicAdd(&cnt[P.cell_base + P.ncells], P.pad);
}

// ---------------------------------------------------------------------------
// Tiles: the candidate ranges of one workgroup of sorted particles.  The plan
// (sph_tile_plan) is uniform over the workgroup, so all of this stays in
// scalar registers.
// Middle contexts (sph_lists_crowded) have few workgroups, and their launches
// last as long as the slowest: in a settling column a twentieth of the tiles
// has 220 - 300 candidates a particle where the mean is 50.  There the planner
// lists the tiles of at least kCrowdedAt candidates a particle, and workgroups
// that start first walk their quarters with four lanes per particle.  us a step
// of 250k particles, steps 21-84 / 41-104 / 101-164 / 251-314 / 451-514: 70 / 76
// / 96 / 141 / 194 without, 69 / 70 / 75 / 99 / 139 with (from 80 candidates on 70
// / 71 / 76 / 99 / 140, from 100 72 / 74 / 77 / 100 / 139).  Sixteen lanes: 2 - 4%
// slower.  The quarters after a workgroup's own tile instead of in workgroups of
// their own: 128 where it is 99 now.
constexpr unsigned kCrowdedAt = 64;
// These kernels hold both walks, in 84 - 101 VGPRs without scratch.
constexpr int kMixedMinBlocks = 5;
constexpr unsigned kCrowded = 2; // in a plan's `wide`: the tile is listed
struct Tile {
    int off[6];       // LDS index = sorted position + off[segment]
    unsigned tb[6];   // LDS index of the segment's first record
    unsigned g0[6], len[6];
    unsigned total;   // staged records
    bool ok;          // staged in LDS; else read candidates from global memory
    bool rows_ok;     // (when not ok) each candidate row (dy) fits on its own
};

// A group is staged when its rows hold at most `cap` records.
__device__ __forceinline__ Tile make_tile(const sph_tile_plan &p, unsigned cap)
{
    Tile T;
    T.total = 0;
#pragma unroll
    for (int q = 0; q < 6; q++) {
        T.g0[q] = p.g0[q];
        T.len[q] = p.len[q];
        T.tb[q] = T.total;
        T.off[q] = (int)T.total - (int)p.g0[q];
        T.total += p.len[q];
    }
    T.ok = !(p.wide & 1u) && T.total <= cap;
    T.rows_ok = !(p.wide & 1u) && T.len[0] + T.len[3] <= cap && T.len[1] + T.len[4] <= cap &&
                T.len[2] + T.len[5] <= cap;
    return T;
}

// Plan p of a context of `tiles` 256-slot tiles, by the eight lanes of a wave
// that share p: plans 0 .. tiles - 1 are the whole tiles', the rest those of
// their quarters (where the context has them).  Lane q < 6 makes segment q,
// lane 6 the rest.
__device__ __forceinline__ void make_plan(unsigned p, unsigned tiles,
                                          const sph_dev_params *__restrict__ Pp,
                                          const int *__restrict__ BS,
                                          const unsigned *__restrict__ skey,
                                          const unsigned *__restrict__ start,
                                          const sph_tile_plans &plans)
{
    const unsigned q = threadIdx.x % 8u;
    const bool quarter = p >= tiles;
    const unsigned n = quarter ? p - tiles : p, size = quarter ? 64u : (unsigned)kTPB;
    if (quarter && (!plans.t64 || n >= 4u * tiles))
        return;
    const int scene = BS[quarter ? n / 4u : n];
    const sph_dev_params &P = Pp[scene];
    const unsigned f = n * size, end = P.poff + (unsigned)P.n; // f: the plan's first particle
    if (f >= end)
        return;
    sph_tile_plan *out = (quarter ? plans.t64 : plans.t256) + n;
    const unsigned sx = P.sx, sy = P.sy;
    const unsigned kf = skey[f] - P.cell_base, kl = skey[min(f + size, end) - 1u] - P.cell_base;
    const unsigned jA = kf / sx, jB = kl / sx;
    const bool wide = jB > jA + 1;
    // the most candidates of the first, the middle and the last particle of the
    // whole tile: lane q < 6 counts row q % 3 of the first (q < 3)
    // or the last, and of the middle
    unsigned most = 0;
    if (plans.crowded) {
        const unsigned f0 = f / kTPB * kTPB, l0 = min(f0 + kTPB, end) - 1u;
        auto row_of = [&](unsigned s) {
            const unsigned k = skey[s] - P.cell_base, x = k % sx;
            const long r = (long)(k / sx) + (long)(q % 3u) - 1;
            if (q >= 6u || r < 0 || r >= (long)sy)
                return 0u;
            const unsigned row = P.cell_base + (unsigned)r * sx;
            return start[row + (x + 1u < sx ? x + 2u : sx)] - start[row + (x > 0 ? x - 1u : 0u)];
        };
        const unsigned e = row_of(q < 3u ? f0 : l0), m = row_of((f0 + l0) / 2u);
        const int base = (int)(threadIdx.x & 63u & ~7u);
        auto rows3 = [&](unsigned v, int at) {
            return (unsigned)(__shfl((int)v, base + at) + __shfl((int)v, base + at + 1) +
                              __shfl((int)v, base + at + 2));
        };
        most = max(max(rows3(e, 0), rows3(e, 3)), rows3(m, 0));
        if (quarter && most < kCrowdedAt)
            return; // a quarter that no workgroup takes
    }
    if (q < 6u) {
        const unsigned rho = q / 3u, j = jA + rho;
        const long r = (long)j + (long)(q % 3u) - 1;
        unsigned a = 0, b = 0;
        if (!wide && j <= jB && r >= 0 && r < (long)sy) {
            const unsigned lo = rho == 0 ? kf - jA * sx : 0;
            const unsigned hi = j == jB ? kl - jB * sx : sx - 1;
            const unsigned row = P.cell_base + (unsigned)r * sx;
            a = start[row + (lo > 0 ? lo - 1 : 0)];
            b = start[row + (hi + 1 < sx ? hi + 1 : sx - 1) + 1];
        }
        out->g0[q] = a;
        out->len[q] = b - a;
    } else if (q == 6u) {
        out->jA = jA;
        out->split = jB > jA ? start[P.cell_base + (jA + 1) * sx] : ~0u;
        out->wide = wide ? 1u : 0u;
        if (size == kTPB && most >= kCrowdedAt) {
            const unsigned at = atomicAdd(plans.crowded_n, 1u);
            if (at < plans.crowded_max) {
                plans.crowded[at] = n;
                out->wide |= kCrowded;
            }
        }
    }
}

// Workgroups that make all plans, eight lanes each; a multiple of the XCDs.
constexpr unsigned kPlansPerGroup = kTPB / 8;
unsigned plan_groups(unsigned slots, const sph_tile_plans &plans)
{
    const unsigned n = slots / kTPB * (plans.t64 ? 5u : 1u);
    const unsigned g = (n + kPlansPerGroup - 1) / kPlansPerGroup;
    return (g + kXcds - 1) / kXcds * kXcds;
}

// Slot of this lane's particle within its cell `key` for the counting sort.
// The wavefront's live lanes are grouped by key first (ballots, no memory),
// then each group's first lane reserves the group's slots with one atomic,
// all groups in the same instruction: one round trip per wavefront instead
// of one per particle (or per key).  Lanes of a group take consecutive slots
// in lane order; the reorder ranks a cell by particle id, so any assignment
// of distinct slots gives the same sorted order.  Call with every live lane.
// The grouping loop reads each group's key with a scalar lane read (the lane
// index is wave-uniform) and keeps only the lane's own group mask, from which
// rank, count and leader follow after the loop.
__device__ __forceinline__ unsigned wave_slot(unsigned *cnt, unsigned key)
{
    const unsigned lane = threadIdx.x & 63u;
    unsigned long long pending = __ballot(1);
    unsigned long long mine = 0; // live lanes with this lane's key
    while (pending) {
        const int first = __ffsll((long long)pending) - 1;
        const unsigned k = (unsigned)__builtin_amdgcn_readlane((int)key, first);
        const unsigned long long same = __ballot(key == k);
        mine = key == k ? same : mine;
        pending &= ~same;
    }
    const int leader = __ffsll((long long)mine) - 1; // the group's lowest lane
    const unsigned rank = (unsigned)__popcll(mine & ((1ull << lane) - 1ull));
    unsigned base = 0;
    if ((int)lane == leader)
        base = atomicAdd(&cnt[key], (unsigned)__popcll(mine));
    return __shfl(base, leader, 64) + rank;
}

// Claim a slot of cell `key` for the next sort: the slot itself, or the
// particle's id in the cell's member list (ids beyond the row are found by the
// sort).
__device__ __forceinline__ void claim_slot(unsigned s, unsigned key, int id, unsigned *cnt,
                                           unsigned *out_slot, const sph_buckets &lists)
{
    const unsigned slot = wave_slot(cnt, key);
    if (!lists.rows)
        out_slot[s] = slot;
    else if (slot < kBucketRow)
        lists.rows[(size_t)key * kBucketRow + slot] = id;
}

// LDS storage of a tile of CAPACITY records (plus the walk's padding): as
// the records are, or - float4 records, SPH_SPLIT_TILES - as two planes of
// float2, (x, y) and (z, w), in the same bytes, so that the candidate tests
// read 8-byte positions at an 8-byte stride.
#ifndef SPH_SPLIT_TILES
#define SPH_SPLIT_TILES 1
#endif
template <class R>
struct TileMem {
    using Rec = R;
    R *p;
    __device__ void put(unsigned i, R v) const { p[i] = v; }
    __device__ R get(unsigned i) const { return p[i]; }
};
struct TileMemSplit {
    using Rec = float4;
    float2 *xy, *zw;
    __device__ void put(unsigned i, float4 v) const
    {
        xy[i] = make_float2(v.x, v.y);
        zw[i] = make_float2(v.z, v.w);
    }
    __device__ float4 get(unsigned i) const
    {
        const float2 a = xy[i], b = zw[i];
        return make_float4(a.x, a.y, b.x, b.y);
    }
};
template <int CAPACITY, class R>
__device__ __forceinline__ TileMem<R> tile_mem(R *tile)
{
    return TileMem<R>{tile};
}
template <int CAPACITY>
__device__ __forceinline__ auto tile_mem(float4 *tile)
{
    if constexpr (SPH_SPLIT_TILES) {
        float2 *xy = reinterpret_cast<float2 *>(tile);
        return TileMemSplit{xy, xy + (CAPACITY + kSphWalkPad)};
    } else {
        return TileMem<float4>{tile};
    }
}

// Copy the planned segments into LDS (all threads), then barrier.  The
// segments lie back to back in the tile, so thread t stages tile records
// t, t + 256, ...: it finds each record's segment (the last one beginning at
// or before it), issues all of its loads, and only then stores them - one
// memory round trip per workgroup, not one per segment.
template <int CAPACITY, class Mem, class Load>
__device__ __forceinline__ void stage_tile(const Tile &T, const Mem &tile, Load load)
{
    using Rec = typename Mem::Rec;
    constexpr int kPer = (CAPACITY + kTPB - 1) / kTPB;
    const unsigned total = T.total;
    Rec v[kPer];
#pragma unroll
    for (int u = 0; u < kPer; u++) {
        const unsigned i = threadIdx.x + (unsigned)u * kTPB;
        if (i < total) {
            int off = T.off[0];
#pragma unroll
            for (int q = 1; q < 6; q++)
                off = T.tb[q] <= i ? T.off[q] : off;
            v[u] = load((unsigned)((int)i - off));
        }
    }
#pragma unroll
    for (int u = 0; u < kPer; u++) {
        const unsigned i = threadIdx.x + (unsigned)u * kTPB;
        if (i < total)
            tile.put(i, v[u]);
    }
    __syncthreads();
}

// Stage only candidate row dy (segments dy + 1 of the first cell row and
// dy + 4 of the second, back to back) into the tile, then barrier: for groups
// whose rows fit one at a time but not all together.
template <int CAPACITY, class Mem, class Load>
__device__ __forceinline__ void stage_row(const Tile &T, int dy, const Mem &tile, Load load)
{
    using Rec = typename Mem::Rec;
    constexpr int kPer = (CAPACITY + kTPB - 1) / kTPB;
    const int qa = dy + 1, qb = dy + 4;
    const unsigned la = T.len[qa], total = la + T.len[qb];
    const unsigned ga = T.g0[qa], gb = T.g0[qb];
    Rec v[kPer];
#pragma unroll
    for (int u = 0; u < kPer; u++) {
        const unsigned i = threadIdx.x + (unsigned)u * kTPB;
        if (i < total)
            v[u] = load(i < la ? ga + i : gb + (i - la));
    }
#pragma unroll
    for (int u = 0; u < kPer; u++) {
        const unsigned i = threadIdx.x + (unsigned)u * kTPB;
        if (i < total)
            tile.put(i, v[u]);
    }
    __syncthreads();
}

// Candidate source reading the LDS tile: the tile index of sorted position
// k of row dy is k + row(dy).
template <class Mem>
struct LdsSrc {
    Mem tile;
    const Tile &T;
    bool rowB; // the lane is in the group's second cell row
    __device__ int row(int dy) const { return rowB ? T.off[dy + 4] : T.off[dy + 1]; }
    __device__ typename Mem::Rec at(unsigned idx) const { return tile.get(idx); }
};

template <class Mem>
__device__ __forceinline__ LdsSrc<Mem> lds_src(const Mem &tile, const Tile &T, bool rowB)
{
    return LdsSrc<Mem>{tile, T, rowB};
}

// The source of a tile staged by stage_row(dy): its first cell row's segment
// begins at index 0, its second one's follows.
template <class Mem>
struct LdsRowSrc {
    Mem tile;
    const Tile &T;
    bool rowB;
    __device__ int row(int dy) const
    {
        const int qa = dy + 1, qb = dy + 4;
        return rowB ? (int)T.len[qa] - (int)T.g0[qb] : -(int)T.g0[qa];
    }
    __device__ typename Mem::Rec at(unsigned idx) const { return tile.get(idx); }
};

template <class Mem>
__device__ __forceinline__ LdsRowSrc<Mem> lds_row_src(const Mem &tile, const Tile &T, bool rowB)
{
    return LdsRowSrc<Mem>{tile, T, rowB};
}

// Candidate source reading global memory.
template <class Rec, class Load>
struct GlobalSrc {
    Load load;
    __device__ int row(int) const { return 0; }
    __device__ Rec at(unsigned idx) const { return load(idx); }
};

template <class Rec, class Load>
__device__ __forceinline__ GlobalSrc<Rec, Load> global_src(Load l)
{
    return GlobalSrc<Rec, Load>{l};
}

// The cell row of the lane's particle (a pad lane's: row 0, its stand-in
// cell's), from the plan unless there is none (NO_PLAN) or the tile spans more
// than two.
template <bool NO_PLAN>
__device__ __forceinline__ unsigned cell_row(const sph_tile_plan &T, bool live, unsigned s,
                                             unsigned key, const sph_dev_params &P)
{
    if (NO_PLAN || (T.wide & 1u))
        return (key - P.cell_base) / P.sx;
    return live ? T.jA + (s >= T.split ? 1u : 0u) : 0u;
}

// Walk a workgroup's candidates from its LDS tile (CAPACITY records) if the
// plan staged one, else from global memory (same order, same results).  Every
// thread of the workgroup calls this (the staging and its barrier need all of
// them); `live` lanes walk.
template <bool CAP, int CAPACITY, int LP = 1, class Rec, class Load, class Test, class Body,
          class Masks>
__device__ __forceinline__ uint2 walk_group(const sph_tile_plan &plan, Rec *tile, Load load,
                                            bool live, unsigned self, const sph_rows &R,
                                            unsigned key, unsigned j, const sph_dev_params &P,
                                            const unsigned *__restrict__ start, Test &test,
                                            Body &body, Masks &mk)
{
    const Tile T = make_tile(plan, CAPACITY);
    const bool rowB = self >= plan.split;
    uint2 fh = make_uint2(0u, 0u);
    const auto mem = tile_mem<CAPACITY>(tile);
    auto rows = [&] { return sph_row_bounds(key, j, P, start); };
    if (T.ok) {
        stage_tile<CAPACITY>(T, mem, load);
        if (live)
            fh = sph_walk_masked<CAP, LP>(self, R, lds_src(mem, T, rowB), P.h2, P.bucket_cap,
                                          test, body, mk, rows);
    } else if (T.rows_ok) {
        // one candidate row at a time: same chunks, same order
        unsigned ci = 0;
        auto pass = [&](auto row) {
            constexpr int dy = decltype(row)::value;
            stage_row<CAPACITY>(T, dy, mem, load);
            if (live) {
                const uint2 r = sph_walk_rows<CAP, dy, dy, LP>(self, R,
                                                               lds_row_src(mem, T, rowB), P.h2,
                                                               P.bucket_cap, test, body, mk, rows,
                                                               ci);
                fh.x += r.x;
                fh.y += r.y;
            }
            __syncthreads(); // the next row overwrites the tile
        };
        pass(std::integral_constant<int, -1>{});
        pass(std::integral_constant<int, 0>{});
        pass(std::integral_constant<int, 1>{});
    } else if (live) {
        fh = sph_walk_masked<CAP, LP>(self, R, global_src<Rec>(load), P.h2, P.bucket_cap, test,
                                      body, mk, rows);
    }
    return fh;
}

} // namespace

// ---------------------------------------------------------------------------
// Gravity + viscosity + prediction (src/fluid.c:398-413, 416-478, 507-523)
//
// GRAV: apply v_y += (-g)*dt first (to self and, on the fly, to every
//       neighbour read, so the result equals a separate gravity pass).
// VISC: gather the viscosity impulses over the neighbour set of the last
//       hash (positions have not moved since, so the set is the
//       reference's half lists seen from both ends).
// PRED: x_prev = x; x += v*dt; boundary; then the new cell key and a slot
//       in that cell (histogram of the next sort).  Without PRED the
//       post-viscosity velocity is written to out_pos.
template <bool GRAV, bool VISC, bool PRED, bool CAP, int LP = 1, bool LISTED = false>
__device__ __forceinline__ void
visc_predict_tile(const sph_dev_params *__restrict__ Pp, const int *__restrict__ BS,
                  const sph_tile_plan *__restrict__ plans, const float2 *__restrict__ POS,
                  const float2 *__restrict__ VEL, const unsigned *__restrict__ K,
                  const unsigned *__restrict__ start, float2 *__restrict__ out_pos,
                  unsigned *__restrict__ out_key,
                  unsigned *__restrict__ out_slot, unsigned *__restrict__ cnt,
                  sph_dev_counters *__restrict__ C, const unsigned long long *__restrict__ clock,
                  float2 *__restrict__ held_vel, float4 *tile, unsigned blk,
                  const sph_buckets &lists = {})
{
    constexpr unsigned kPer = kTPB / LP; // particles per workgroup
    const unsigned s0 = blk * kPer;
    const unsigned s = s0 + threadIdx.x / LP;
    // loads that need no scene parameter go out before the parameters (every
    // slot of the grid is inside the arrays; a value is used where its slot
    // is live)
    const float2 a0 = POS[s], av0 = VEL[s];
    const unsigned ks = VISC ? K[s] : 0u;
    const int id = lists.rows ? lists.ids[s] : 0;
    const sph_tile_plan T = VISC && LP != 16 ? plans[blk] : sph_tile_plan{};
    const sph_dev_params P = Pp[BS[blk / LP]];
    const unsigned s1 = min(s0 + kPer, P.poff + (unsigned)P.n);
    const bool lead = threadIdx.x % LP == 0; // the lane that stores the particle's results
    const float gdt = P.g_neg * P.dt;
    if (LISTED && s0 < s1 && (T.wide & kCrowded))
        return; // four lanes per particle walk it (a tile of no particle has no plan)
    if (PRED)
        add_pad(P, s0, cnt);
    if (s0 >= s1)
        return; // a padding workgroup
    if (PRED && P.frozen) {
        // frozen scene: same position, same cell; its velocity waits in
        // held_vel for the relaxation kernel (the sort of a frozen scene is
        // the identity)
        if (s < s1 && lead) {
            const float2 a = POS[s];
            out_pos[s] = a;
            held_vel[s] = VEL[s];
            const unsigned key = sph_cell_key(a.x, a.y, P, &C->key_out_of_range);
            out_key[s] = key;
            claim_slot(s, key, id, cnt, out_slot, lists);
        }
        return;
    }
    // sloshing: horizontal box acceleration, applied like gravity
    const bool slosh = GRAV && P.slosh_amp != 0.0f;
    const float sdt = slosh ? sph_slosh_accel(P, *clock) * P.dt : 0.0f;
    // the lane's own particle and candidate rows, loaded before the staging
    const float2 a = a0, av = av0;
    const bool live = s < s1;
    const unsigned key = VISC && live ? ks : P.cell_base; // pad lanes: any valid cell
    const unsigned j = VISC ? cell_row<LP == 16>(T, live, s, key, P) : 0u;
    const sph_rows R = VISC ? sph_row_bounds(key, j, P, start) : sph_rows{};
    const float avx = slosh ? av.x + sdt : av.x;
    const float avy = GRAV ? av.y + gdt : av.y;
    float nvx = avx, nvy = avy;
    unsigned full = 0, half = 0;
    if (VISC) {
        // a neighbour's record carries its velocity after gravity and
        // sloshing (the same expressions as the particle's own), applied
        // once per record rather than once per pair
        auto load = [&](unsigned g) {
            const float2 p = POS[g], v = VEL[g];
            return make_float4(p.x, p.y, slosh ? v.x + sdt : v.x, GRAV ? v.y + gdt : v.y);
        };
        auto test = [&](float4 b) {
            const float dx = b.x - a.x, ddy = b.y - a.y;
            return dx * dx + ddy * ddy;
        };
        const sph_visc_consts V{sph_vgpr(P.h_recip), sph_vgpr(P.dt), sph_vgpr(P.sigma),
                                sph_vgpr(P.beta)};
        auto half_impulse = [&](float4 b) {
            const float dx = b.x - a.x, ddy = b.y - a.y;
            return sph_visc_half(dx, ddy, dx * dx + ddy * ddy, avx, avy, b.z, b.w, V, P);
        };
        sph_masks_none mk;
        uint2 fh;
        if constexpr (LP == 1) {
            auto body = [&](unsigned, float4 b, auto &&) {
                const float2 t = half_impulse(b);
                nvx = nvx - t.x;
                nvy = nvy - t.y;
            };
            fh = walk_group<CAP, kTileCap>(T, tile, load, live, s, R, key, j, P, start, test, body,
                                           mk);
        } else if constexpr (LP == 16) {
            auto pair = [&](float4 b, bool cand, auto &&, bool &accepted, bool &) {
                const float dx = b.x - a.x, ddy = b.y - a.y;
                const float r2 = dx * dx + ddy * ddy;
                accepted = cand && !(r2 > P.h2);
                const float2 t = sph_visc_half(dx, ddy, accepted ? r2 : 0.5f * P.h2, avx, avy,
                                               b.z, b.w, V, P);
                return sph_pair_term{accepted ? t.x : 0.0f, accepted ? t.y : 0.0f};
            };
            auto apply = [&](const sph_pair_term &t) {
                nvx = nvx - t.a;
                nvy = nvy - t.b;
            };
            fh = sph_walk_wide<CAP>(s, live, R, P.bucket_cap, load, pair, apply, [](bool) {});
            fh.x = sph_row_sum(fh.x);
            fh.y = sph_row_sum(fh.y);
        } else {
            auto term = [&](unsigned, float4 b, auto &&, bool &) {
                const float2 t = half_impulse(b);
                return sph_pair_term{t.x, t.y};
            };
            auto apply = [&](const sph_pair_term &t) {
                nvx = nvx - t.a;
                nvy = nvy - t.b;
            };
            auto never = [](bool) {};
            sph_split_body<decltype(term), decltype(apply), decltype(never)> sb{term, apply,
                                                                                never};
            fh = walk_group<CAP, kTileCap, LP>(T, tile, load, live, s, R, key, j, P, start, test,
                                               sb, mk);
        }
        full = fh.x;
        half = lead ? fh.y : 0u; // a particle's half list counted once
    }
    if (live && lead) {
        if (PRED) {
            float x = a.x + nvx * P.dt;
            float y = a.y + nvy * P.dt;
            sph_boundary(x, y, P);
            out_pos[s] = make_float2(x, y);
            const unsigned nk = sph_cell_key(x, y, P, &C->key_out_of_range);
            out_key[s] = nk;
            claim_slot(s, nk, id, cnt, out_slot, lists);
        } else {
            out_pos[s] = make_float2(nvx, nvy);
        }
    }
    if (VISC)
        report_neighbors(full, half, C);
}

template <bool GRAV, bool VISC, bool PRED, bool CAP>
__global__ void __launch_bounds__(kTPB, kGatherMinBlocks)
k_visc_predict(const sph_dev_params *__restrict__ Pp, const int *__restrict__ BS,
               const sph_tile_plan *__restrict__ plans, const float2 *__restrict__ POS,
               const float2 *__restrict__ VEL, const unsigned *__restrict__ K,
               const unsigned *__restrict__ start,
               float2 *__restrict__ out_pos, unsigned *__restrict__ out_key,
               unsigned *__restrict__ out_slot, unsigned *__restrict__ cnt,
               sph_dev_counters *__restrict__ C, const unsigned long long *__restrict__ clock,
               float2 *__restrict__ held_vel)
{
    __shared__ float4 tile[VISC ? kTileCap + kSphWalkPad : 1];
    visc_predict_tile<GRAV, VISC, PRED, CAP, 1>(Pp, BS, plans, POS, VEL, K, start, out_pos,
                                                out_key, out_slot, cnt, C, clock, held_vel, tile,
                                                xcd_block());
}

// The fused step's variant with one lane per particle, and four in crowded
// tiles.
template <bool CAP>
__global__ void __launch_bounds__(kTPB, kMixedMinBlocks)
k_visc_predict_mixed(const sph_dev_params *__restrict__ Pp, const int *__restrict__ BS,
                     sph_tile_plans plans,
                     const float2 *__restrict__ POS, const float2 *__restrict__ VEL,
                     const unsigned *__restrict__ K, const unsigned *__restrict__ start,
                     float2 *__restrict__ out_pos, unsigned *__restrict__ out_key,
                     unsigned *__restrict__ out_slot, unsigned *__restrict__ cnt,
                     sph_dev_counters *__restrict__ C,
                     const unsigned long long *__restrict__ clock, float2 *__restrict__ held_vel)
{
    __shared__ float4 tile[kTileCap + kSphWalkPad];
    const unsigned listed = plans.crowded_max * 4u;
    if (blockIdx.x < listed) {
        const unsigned k = blockIdx.x / 4u;
        if (k < *plans.crowded_n)
            visc_predict_tile<true, true, true, CAP, 4>(
                Pp, BS, plans.t64, POS, VEL, K, start, out_pos, out_key, out_slot, cnt, C, clock,
                held_vel, tile, plans.crowded[k] * 4u + blockIdx.x % 4u);
        return;
    }
    visc_predict_tile<true, true, true, CAP, 1, true>(Pp, BS, plans.t256, POS, VEL, K, start,
                                                      out_pos, out_key, out_slot, cnt, C, clock,
                                                      held_vel, tile, xcd_block(listed));
}

// With four lanes per particle (sph_gather_lanes).
template <bool CAP>
__global__ void __launch_bounds__(kTPB, 1)
k_visc_predict_quad(const sph_dev_params *__restrict__ Pp, const int *__restrict__ BS,
                    const sph_tile_plan *__restrict__ plans, const float2 *__restrict__ POS,
                    const float2 *__restrict__ VEL, const unsigned *__restrict__ K,
                    const unsigned *__restrict__ start, float2 *__restrict__ out_pos,
                    unsigned *__restrict__ out_key, unsigned *__restrict__ out_slot,
                    unsigned *__restrict__ cnt, sph_dev_counters *__restrict__ C,
                    const unsigned long long *__restrict__ clock, float2 *__restrict__ held_vel)
{
    __shared__ float4 tile[kTileCap + kSphWalkPad];
    visc_predict_tile<true, true, true, CAP, 4>(Pp, BS, plans, POS, VEL, K, start, out_pos,
                                                out_key, out_slot, cnt, C, clock, held_vel, tile,
                                                xcd_block());
}

// Sixteen lanes per particle.
template <bool CAP>
__global__ void __launch_bounds__(kTPB, 1)
k_visc_predict_row(const sph_dev_params *__restrict__ Pp, const int *__restrict__ BS,
                   const float2 *__restrict__ POS, const float2 *__restrict__ VEL,
                   const unsigned *__restrict__ K, const unsigned *__restrict__ start,
                   float2 *__restrict__ out_pos, unsigned *__restrict__ out_key,
                   unsigned *__restrict__ out_slot, unsigned *__restrict__ cnt,
                   sph_dev_counters *__restrict__ C, const unsigned long long *__restrict__ clock,
                   float2 *__restrict__ held_vel, sph_buckets lists)
{
    visc_predict_tile<true, true, true, CAP, 16>(Pp, BS, nullptr, POS, VEL, K, start, out_pos,
                                                 out_key, out_slot, cnt, C, clock, held_vel,
                                                 nullptr, xcd_block(), lists);
}

// src/fluid.c:398-413 as a separate pass (phase API).
__global__ void __launch_bounds__(kTPB)
k_gravity(const sph_dev_params *__restrict__ Pp, const int *__restrict__ BS,
          float2 *__restrict__ VEL, float2 *__restrict__ RHO)
{
    const unsigned blk = xcd_block();
    const sph_dev_params P = Pp[BS[blk]];
    const unsigned s = blk * kTPB + threadIdx.x;
    if (s >= P.poff + (unsigned)P.n)
        return;
    VEL[s].y += P.g_neg * P.dt;
    RHO[s] = make_float2(0.0f, 0.0f);
}

// src/fluid.c:507-523 as a separate, in-place pass (phase API).
__global__ void __launch_bounds__(kTPB)
k_predict(const sph_dev_params *__restrict__ Pp, const int *__restrict__ BS,
          float2 *__restrict__ POS, const float2 *__restrict__ VEL, float2 *__restrict__ PREV)
{
    const unsigned blk = xcd_block();
    const sph_dev_params P = Pp[BS[blk]];
    const unsigned s = blk * kTPB + threadIdx.x;
    if (s >= P.poff + (unsigned)P.n)
        return;
    const float2 p = POS[s], v = VEL[s];
    PREV[s] = p;
    float x = p.x + v.x * P.dt;
    float y = p.y + v.y * P.dt;
    sph_boundary(x, y, P);
    POS[s] = make_float2(x, y);
}

// src/fluid.c:642-653 as a separate, in-place pass (phase API).
__global__ void __launch_bounds__(kTPB)
k_update_velocities(const sph_dev_params *__restrict__ Pp, const int *__restrict__ BS,
                    float2 *__restrict__ POS, float2 *__restrict__ VEL,
                    const float2 *__restrict__ PREV)
{
    const unsigned blk = xcd_block();
    const sph_dev_params P = Pp[BS[blk]];
    const unsigned s = blk * kTPB + threadIdx.x;
    if (s >= P.poff + (unsigned)P.n)
        return;
    float2 p = POS[s];
    const float2 q = PREV[s];
    sph_boundary(p.x, p.y, P);
    float vx = (p.x - q.x) / P.dt;
    float vy = (p.y - q.y) / P.dt;
    sph_check_velocity(vx, vy);
    POS[s] = p;
    VEL[s] = make_float2(vx, vy);
}

// Keys and slots of the current positions (histogram pass of a standalone
// hash, phase API; the fused step folds this into its producers).
__global__ void __launch_bounds__(kTPB)
k_key_hist(const sph_dev_params *__restrict__ Pp, const int *__restrict__ BS,
           const float2 *__restrict__ POS, unsigned *__restrict__ out_key,
           unsigned *__restrict__ out_slot, unsigned *__restrict__ cnt,
           sph_dev_counters *__restrict__ C)
{
    const unsigned blk = xcd_block();
    const sph_dev_params P = Pp[BS[blk]];
    const unsigned s = blk * kTPB + threadIdx.x;
    add_pad(P, blk * kTPB, cnt);
    if (s >= P.poff + (unsigned)P.n)
        return;
    const float2 p = POS[s];
    const unsigned key = sph_cell_key(p.x, p.y, P, &C->key_out_of_range);
    out_key[s] = key;
    out_slot[s] = wave_slot(cnt, key);
}

// ---------------------------------------------------------------------------
// Cell-count scan: start[c] = sum of cnt[0..c), over m = cells + 1 entries
// (cnt[cells] is always 0, so start[cells] = n).  Reduce-then-scan over tiles
// of kScanTile counts; the apply kernel adds the sum of all earlier tiles,
// writes the starts and clears the counts for the next sort.  Both arrays hold
// whole tiles (sph_scan_padded(m) entries, the padding's counts zero), so
// nothing is bounds-checked: a tile is two halves of 1024 counts, thread t
// holding counts [4t, 4t+4) of each half, and every wave's load or store
// covers 1 KiB of consecutive memory.
constexpr int kScanThreads = 256;
constexpr int kScanTile = 2 * 4 * kScanThreads;

__device__ __forceinline__ unsigned sum4(uint4 v) { return v.x + v.y + v.z + v.w; }

__global__ void __launch_bounds__(kScanThreads)
k_scan_reduce(const uint4 *__restrict__ cnt, unsigned *__restrict__ bsum)
{
    __shared__ unsigned red[kScanThreads / kWave];
    const uint4 *t = cnt + blockIdx.x * (kScanTile / 4);
    unsigned sum = sum4(t[threadIdx.x]) + sum4(t[threadIdx.x + kScanThreads]);
    sum = wave_sum_u32(sum);
    if (lane0())
        red[threadIdx.x / kWave] = sum;
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned a = 0;
        for (int i = 0; i < kScanThreads / kWave; i++)
            a += red[i];
        bsum[blockIdx.x] = a;
    }
}

__global__ void __launch_bounds__(kScanThreads)
k_scan_apply(uint4 *__restrict__ cnt, const unsigned *__restrict__ bsum,
             uint4 *__restrict__ start)
{
    constexpr int kW = kScanThreads / kWave;
    __shared__ unsigned wpre[kW], wa[kW], wb[kW];
    const int w = threadIdx.x / kWave, lane = threadIdx.x & (kWave - 1);
    uint4 *t = cnt + blockIdx.x * (kScanTile / 4);
    const uint4 a = t[threadIdx.x], b = t[threadIdx.x + kScanThreads];
    // prefix of all earlier tiles
    unsigned pre = 0;
    for (unsigned i = threadIdx.x; i < blockIdx.x; i += kScanThreads)
        pre += bsum[i];
    pre = wave_sum_u32(pre);
    // inclusive wave scans of both halves' per-thread totals
    const unsigned ta = sum4(a), tb = sum4(b);
    unsigned ia = ta, ib = tb;
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
        const unsigned ya = (unsigned)__shfl_up((int)ia, o, kWave);
        const unsigned yb = (unsigned)__shfl_up((int)ib, o, kWave);
        ia += lane >= o ? ya : 0u;
        ib += lane >= o ? yb : 0u;
    }
    if (lane == kWave - 1) {
        wpre[w] = pre;
        wa[w] = ia;
        wb[w] = ib;
    }
    __syncthreads();
    unsigned tile_pre = 0, half_a = 0, pa = 0, pb = 0;
#pragma unroll
    for (int i = 0; i < kW; i++) {
        tile_pre += wpre[i];
        half_a += wa[i];
        pa += i < w ? wa[i] : 0u;
        pb += i < w ? wb[i] : 0u;
    }
    const unsigned ra = tile_pre + pa + (ia - ta);
    const unsigned rb = tile_pre + half_a + pb + (ib - tb);
    uint4 *o = start + blockIdx.x * (kScanTile / 4);
    o[threadIdx.x] = make_uint4(ra, ra + a.x, ra + a.x + a.y, ra + a.x + a.y + a.z);
    o[threadIdx.x + kScanThreads] = make_uint4(rb, rb + b.x, rb + b.x + b.y, rb + b.x + b.y + b.z);
    t[threadIdx.x] = make_uint4(0u, 0u, 0u, 0u);
    t[threadIdx.x + kScanThreads] = make_uint4(0u, 0u, 0u, 0u);
}

// The whole scan of a small count array (sph_scan_single_fits: at most
// kScanSingle counts, whole tiles) in one workgroup: the same starts and the
// same cleared counts as k_scan_reduce and k_scan_apply, in one launch where
// they take two.  Thread t holds counts [4t, 4t + 4).
constexpr unsigned kScanSingleThreads = 1024;
constexpr unsigned kScanSingle = 4 * kScanSingleThreads;

__global__ void __launch_bounds__(kScanSingleThreads)
k_scan_single(uint4 *__restrict__ cnt, unsigned mp, uint4 *__restrict__ start)
{
    constexpr unsigned kWaves = kScanSingleThreads / kWave;
    __shared__ unsigned wsum[kWaves];
    const unsigned t = threadIdx.x, lane = t & (kWave - 1u), w = t / kWave;
    const bool live = 4u * t < mp;
    const uint4 c = live ? cnt[t] : make_uint4(0u, 0u, 0u, 0u);
    const unsigned tot = sum4(c);
    unsigned inc = tot;
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
        const unsigned y = (unsigned)__shfl_up((int)inc, o, kWave);
        inc += lane >= (unsigned)o ? y : 0u;
    }
    if (lane == kWave - 1u)
        wsum[w] = inc;
    __syncthreads();
    unsigned r = inc - tot;
    for (unsigned i = 0; i < w; i++)
        r += wsum[i];
    if (live) {
        start[t] = make_uint4(r, r + c.x, r + c.x + c.y, r + c.x + c.y + c.z);
        cnt[t] = make_uint4(0u, 0u, 0u, 0u); // cleared for the next sort
    }
}

// Drop (id, source index) into the cell ranges in slot order.
__global__ void __launch_bounds__(kTPB)
k_scatter(const sph_dev_params *__restrict__ Pp, const int *__restrict__ BS,
          const unsigned *__restrict__ key, const unsigned *__restrict__ slot,
          const unsigned *__restrict__ start, const int *__restrict__ id_src,
          int *__restrict__ perm_src, int *__restrict__ perm_id, unsigned *__restrict__ key_dst,
          unsigned *__restrict__ crowded_n)
{
    const unsigned blk = xcd_block();
    if (blockIdx.x == 0 && threadIdx.x == 0 && crowded_n)
        *crowded_n = 0; // for the plans that the reorder makes
    const sph_dev_params &P = Pp[BS[blk]];
    const unsigned i = blk * kTPB + threadIdx.x;
    if (i >= P.poff + (unsigned)P.n)
        return;
    const unsigned k = key[i];
    const unsigned pos = start[k] + slot[i];
    perm_src[pos] = (int)i;
    perm_id[pos] = id_src[i];
    key_dst[pos] = k; // every position of a cell holds its key, whatever the order inside
}

// Rank each particle by id inside its cell and gather its fields to
// (cell, id) order.  The slot order within a cell is arbitrary (atomics);
// ranking restores the reference's bucket order (ascending id).  The rank
// also feeds the occupancy counters: a particle of rank 100 means its cell
// holds more than the reference's 100 bucket slots (src/fluid.c:174).
constexpr unsigned kRankBatch = 8;
constexpr unsigned kRankHalo = 64; // staged ids either side of a workgroup's positions
// The launch's first `planners` workgroups make the tile plans of the sorted
// positions for the gathers that follow, beside the others, which rank and
// move the particles.  (Made by the ranking workgroups themselves, by some of
// their lanes or by a fifth wave, the plans lengthened the 10.6 us of a
// reorder of 1M particles to 11.2 - 13.0.)
template <int NF>
__global__ void __launch_bounds__(kTPB)
k_reorder(const sph_dev_params *__restrict__ Pp, const int *__restrict__ BS,
          const unsigned *__restrict__ start, const int *__restrict__ perm_src,
          const int *__restrict__ perm_id, const unsigned *__restrict__ skey,
          sph_reorder_fields<NF> f, int *__restrict__ id_dst, unsigned planners,
          sph_tile_plans plans, sph_dev_counters *__restrict__ C)
{
    __shared__ int wid[kTPB + 2 * kRankHalo];
    if (blockIdx.x < planners) {
        make_plan(blockIdx.x * kPlansPerGroup + threadIdx.x / 8u, gridDim.x - planners, Pp, BS,
                  skey, start, plans);
        return;
    }
    const unsigned blk = xcd_block(planners);
    const sph_dev_params &P = Pp[BS[blk]];
    const unsigned s0 = blk * kTPB;
    const unsigned end = P.poff + (unsigned)P.n;
    if (s0 >= end)
        return; // a padding workgroup
    const unsigned k = s0 + threadIdx.x;
    const bool live = k < end;
    // the ids of sorted positions [w0, w1): this workgroup's and up to
    // kRankHalo either side, inside the scene, staged for the ranking
    static_assert(2 * kRankHalo <= kTPB, "two staged ids per thread");
    const unsigned w0 = s0 >= P.poff + kRankHalo ? s0 - kRankHalo : P.poff;
    const unsigned w1 = min(s0 + kTPB + kRankHalo, end);
    const unsigned g0 = w0 + threadIdx.x, g1 = g0 + kTPB;
    const int id0 = g0 < w1 ? perm_id[g0] : 0;
    const int id1 = g1 < w1 ? perm_id[g1] : 0;
    // the lane's own record, its fields and its cell's range, all in flight
    // with the staging loads, before the barrier
    int i = 0, myid = 0;
    unsigned b = 0, e = 0;
    float2 v[NF];
#pragma unroll
    for (int q = 0; q < NF; q++)
        v[q] = make_float2(0.0f, 0.0f);
    if (live) {
        i = perm_src[k];
        myid = perm_id[k];
        const unsigned c = skey[k]; // the sorted keys, written by the scatter
#pragma unroll
        for (int q = 0; q < NF; q++)
            v[q] = f.src[q][i];
        b = start[c];
        e = start[c + 1];
    }
    if (g0 < w1)
        wid[g0 - w0] = id0;
    if (g1 < w1)
        wid[g1 - w0] = id1;
    __syncthreads();
    unsigned occupancy = 0;
    if (live) {
        // rank = members of the cell with a smaller id, kRankBatch at a time
        // (indices clamped into the cell, so every read is in bounds and none
        // is predicated): from the staged ids when the cell lies inside them
        unsigned rank = 0;
        if (b >= w0 && e <= w1) {
            for (unsigned m = b; m < e; m += kRankBatch) {
                int idv[kRankBatch];
#pragma unroll
                for (int t = 0; t < kRankBatch; t++)
                    idv[t] = wid[min(m + t, e - 1u) - w0];
#pragma unroll
                for (int t = 0; t < kRankBatch; t++)
                    rank += (m + t < e && idv[t] < myid) ? 1u : 0u;
            }
        } else {
            for (unsigned m = b; m < e; m += kRankBatch) {
                int idv[kRankBatch];
#pragma unroll
                for (int t = 0; t < kRankBatch; t++)
                    idv[t] = perm_id[min(m + t, e - 1u)];
#pragma unroll
                for (int t = 0; t < kRankBatch; t++)
                    rank += (m + t < e && idv[t] < myid) ? 1u : 0u;
            }
        }
        const unsigned d = b + rank;
#pragma unroll
        for (int q = 0; q < NF; q++)
            f.dst[q][d] = v[q];
        id_dst[d] = myid;
        if (rank == SPH_REF_MAX_BUCKET)
            atomicAdd(&C->bucket_overflow, 1ull);
        occupancy = rank + 1;
    }
    const unsigned m = wave_max_u32(occupancy);
    if (lane0())
        raise_max(&C->max_cell_count, m);
}

// The whole sort of a small context in one launch.  Every workgroup makes all
// cell starts for itself, in LDS, from the counts (at most kSmallCounts; they
// come from L2), and then places its own 256 source particles: the rank in the
// cell from the cell's member list, the fields straight to their sorted
// position.  The starts in memory are written, and the other counts cleared,
// by all workgroups together.  Two count arrays take turns (the counts read
// here are cleared by the next sort), because no workgroup may clear what
// another still reads.  The members of a cell that its list's row does not
// hold are searched for among the scene's keys, by the whole workgroup, one
// such cell after the other.
//
// us a step with this sort, against scan + scatter + reorder, steps 21-84 /
// 251-314: 1.5k 24 / 31 against 31 / 39, 4k 24 / 39 against 30 / 48, 16k 32 /
// 51 against 39 / 58, 25k 38 / 55 against 44 / 62.
// TPB threads, of which the first 256 own a particle each; thread t sums the
// counts [SEG t, SEG t + SEG) of the LDS copy (four spare words a segment keep
// the threads' 16-byte reads on different banks).
constexpr unsigned kSmallCounts = 32768;

template <int SEG, int TPB>
__global__ void __launch_bounds__(TPB)
k_sort_small(const sph_dev_params *__restrict__ Pp, const int *__restrict__ BS,
             const unsigned *__restrict__ key, const uint4 *__restrict__ cnt,
             uint4 *__restrict__ cnt_next, unsigned mp, uint4 *__restrict__ start,
             sph_buckets lists, sph_reorder_fields<2> f, int *__restrict__ id_dst,
             unsigned *__restrict__ key_dst, sph_dev_counters *__restrict__ C)
{
    constexpr unsigned kStride = SEG + 4;
    __shared__ __align__(16) unsigned sc[TPB * kStride];
    __shared__ unsigned wsum[TPB / kWave];
    auto at = [](unsigned c) { return c / SEG * kStride + c % SEG; };
    const unsigned blk = blockIdx.x, t = threadIdx.x;
    const bool owner = TPB == kTPB || t < (unsigned)kTPB;
    const unsigned i = blk * kTPB + (owner ? t : 0u);
    // the own particle, on its way while the starts are made
    const unsigned k0 = key[i];
    const int myid = lists.ids[i];
    const float2 v0 = f.src[0][i], v1 = f.src[1][i];
    const sph_dev_params &P = Pp[BS[blk]];
    const unsigned end = P.poff + (unsigned)P.n;
    const bool live = owner && i < end;
    const unsigned c = live ? k0 : 0u;
    // the start of the cell's list, as well
    constexpr unsigned kFirst = 16;
    int4 row[kFirst / 4];
    const int4 *list = reinterpret_cast<const int4 *>(lists.rows + (size_t)c * kBucketRow);
#pragma unroll
    for (unsigned u = 0; u < kFirst / 4; u++)
        row[u] = list[u];
    // counts into LDS, then exclusive sums in place
    for (unsigned u = t; u < mp / 4u; u += TPB)
        *(uint4 *)&sc[at(4u * u)] = cnt[u];
    __syncthreads();
    const unsigned segs = mp / SEG; // mp: a multiple of 2,048, at most TPB segments
    unsigned *seg = &sc[t * kStride];
    unsigned tot = 0;
    if (t < segs)
        for (unsigned u = 0; u < SEG; u += 4)
            tot += sum4(*(const uint4 *)&seg[u]);
    unsigned inc = tot;
    const unsigned lane = t & (kWave - 1u);
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
        const unsigned y = (unsigned)__shfl_up((int)inc, o, kWave);
        inc += lane >= (unsigned)o ? y : 0u;
    }
    if (lane == kWave - 1u)
        wsum[t / kWave] = inc;
    __syncthreads();
    unsigned run = inc - tot;
    for (unsigned w = 0; w < t / kWave; w++)
        run += wsum[w];
    if (t < segs)
        for (unsigned u = 0; u < SEG; u += 4) {
            const uint4 n = *(const uint4 *)&seg[u];
            *(uint4 *)&seg[u] = make_uint4(run, run + n.x, run + n.x + n.y, run + n.x + n.y + n.z);
            run += sum4(n);
        }
    __syncthreads();
    // every workgroup's share of the starts and of the cleared counts
    for (unsigned u = blk * TPB + t; u < mp / 4u; u += gridDim.x * TPB) {
        start[u] = *(const uint4 *)&sc[at(4u * u)];
        cnt_next[u] = make_uint4(0u, 0u, 0u, 0u);
    }
    const unsigned b = sc[at(c)], n = sc[at(c + 1u)] - b; // c + 1 <= cells < mp
    unsigned rank = 0;
    if (live && n <= kBucketRow) {
        auto count4 = [&](int4 q, unsigned m) {
            rank += (m < n && q.x < myid ? 1u : 0u) + (m + 1u < n && q.y < myid ? 1u : 0u) +
                    (m + 2u < n && q.z < myid ? 1u : 0u) + (m + 3u < n && q.w < myid ? 1u : 0u);
        };
#pragma unroll
        for (unsigned u = 0; u < kFirst / 4; u++)
            count4(row[u], 4u * u);
        for (unsigned m = kFirst; m < n; m += 16u) {
            int4 q[4];
#pragma unroll
            for (unsigned u = 0; u < 4; u++)
                q[u] = list[min(m / 4u + u, kBucketRow / 4u - 1u)];
#pragma unroll
            for (unsigned u = 0; u < 4; u++)
                count4(q[u], m + 4u * u);
        }
    }
    bool over = live && n > kBucketRow;
    if (__syncthreads_or(over)) {
        __shared__ unsigned pick, nfound;
        __shared__ int found[TPB];
        for (;;) {
            if (t == 0) {
                pick = ~0u;
                nfound = 0;
            }
            __syncthreads();
            if (over)
                atomicMin(&pick, c);
            __syncthreads();
            const unsigned cell = pick;
            if (cell == ~0u)
                break; // every thread at once
            const bool mine = over && c == cell;
            for (unsigned m0 = P.poff; m0 < end; m0 += TPB) {
                if (m0 + t < end && key[m0 + t] == cell)
                    found[atomicAdd(&nfound, 1u)] = lists.ids[m0 + t];
                __syncthreads();
                const unsigned nf = nfound;
                if (mine)
                    for (unsigned u = 0; u < nf; u++)
                        rank += found[u] < myid ? 1u : 0u;
                __syncthreads();
                if (t == 0)
                    nfound = 0;
                __syncthreads();
            }
            over = over && !mine;
        }
    }
    unsigned occupancy = 0;
    if (live) {
        const unsigned d = b + rank;
        f.dst[0][d] = v0;
        f.dst[1][d] = v1;
        id_dst[d] = myid;
        key_dst[d] = c;
        if (rank == SPH_REF_MAX_BUCKET)
            atomicAdd(&C->bucket_overflow, 1ull);
        occupancy = rank + 1;
    }
    const unsigned m = wave_max_u32(occupancy);
    if (lane0())
        raise_max(&C->max_cell_count, m);
}

// The tile plans alone (sph_launch_plan).
__global__ void __launch_bounds__(kTPB)
k_plan(const sph_dev_params *__restrict__ Pp, const int *__restrict__ BS, unsigned tiles,
       const unsigned *__restrict__ start, const unsigned *__restrict__ skey,
       sph_tile_plans plans)
{
    make_plan(blockIdx.x * kPlansPerGroup + threadIdx.x / 8u, tiles, Pp, BS, skey, start, plans);
}

// ---------------------------------------------------------------------------
// Density (src/hash.c:190-194, 225-229 with src/fluid.c:527-539) in gather
// form: each particle sums (1-r/h)^2 and (1-r/h)^3 over its neighbours.
template <bool CAP, int LP = 1, bool LISTED = false>
__device__ __forceinline__ void
density_tile(const sph_dev_params *__restrict__ Pp, const int *__restrict__ BS,
             const sph_tile_plan *__restrict__ plans, const float2 *__restrict__ POS,
             const unsigned *__restrict__ K, const unsigned *__restrict__ start,
             float2 *__restrict__ RHO, uint4 *__restrict__ masks,
             sph_dev_counters *__restrict__ C, float2 *tile, unsigned blk)
{
    constexpr unsigned kPer = kTPB / LP; // particles per workgroup
    const unsigned s0 = blk * kPer;
    const unsigned s = s0 + threadIdx.x / LP;
    // the lane's own particle and the tile's plan, before the scene
    // parameters (every slot of the grid is inside the arrays)
    const float2 a = POS[s];
    const unsigned ks = K[s];
    const sph_tile_plan T = LP != 16 ? plans[blk] : sph_tile_plan{};
    const sph_dev_params P = Pp[BS[blk / LP]];
    const unsigned s1 = min(s0 + kPer, P.poff + (unsigned)P.n);
    const bool lead = threadIdx.x % LP == 0; // the lane that stores the particle's results
    if (s0 >= s1 || P.frozen || (LISTED && (T.wide & kCrowded)))
        return; // a padding workgroup, a frozen scene, or a tile that four lanes walk
    // the candidate rows, before the staging
    const bool live = s < s1;
    const unsigned key = live ? ks : P.cell_base; // pad lanes: any valid cell
    const unsigned j = cell_row<LP == 16>(T, live, s, key, P);
    const sph_rows R = sph_row_bounds(key, j, P, start);
    float rho = 0.0f, rhon = 0.0f;
    auto load = [&](unsigned g) { return POS[g]; };
    auto test = [&](float2 b) {
        const float dx = a.x - b.x, ddy = a.y - b.y;
        return dx * dx + ddy * ddy;
    };
    const float h_recip = sph_vgpr(P.h_recip);
    // the pair's (1 - r/h)^2 and ^3, or zero outside h (rho + 0 == rho, as
    // rho >= +0)
    auto weights = [&](float r2) {
        const float OmR = 1.0f - sph_sqrt_common(r2) * h_recip;
        const float OmR2 = OmR * OmR;
        float2 t = make_float2(OmR2, OmR2 * OmR);
        if (__builtin_expect(__ballot(sph_uncommon_pair(r2, kPairLoRoot, P)) != 0ull, 0)) {
            const float ratio = sph_sqrt(r2) * h_recip;
            const float w = (1.0f - ratio) * (1.0f - ratio);
            const bool in = ratio < 1.0f;
            t = make_float2(in ? w : 0.0f, in ? w * (1.0f - ratio) : 0.0f);
        }
        return t;
    };
    auto pair = [&](float2 b) { return weights(test(b)); };
    sph_masks_record mk;
    uint2 fh;
    if constexpr (LP == 1) {
        auto body = [&](unsigned, float2 b, auto &&) {
            const float2 t = pair(b);
            rho = rho + t.x;
            rhon = rhon + t.y;
        };
        fh = walk_group<CAP, 2 * kTileCap>(T, tile, load, live, s, R, key, j, P, start, test, body,
                                           mk);
    } else if constexpr (LP == 16) {
        auto wide = [&](float2 b, bool cand, auto &&, bool &accepted, bool &) {
            const float r2 = test(b);
            accepted = cand && !(r2 > P.h2);
            const float2 t = weights(accepted ? r2 : 0.5f * P.h2);
            return sph_pair_term{accepted ? t.x : 0.0f, accepted ? t.y : 0.0f};
        };
        auto apply = [&](const sph_pair_term &t) {
            rho = rho + t.a;
            rhon = rhon + t.b;
        };
        fh = sph_walk_wide<CAP>(s, live, R, P.bucket_cap, load, wide, apply, [](bool) {});
        fh.x = sph_row_sum(fh.x);
        fh.y = sph_row_sum(fh.y);
    } else {
        auto term = [&](unsigned, float2 b, auto &&, bool &) {
            const float2 t = pair(b);
            return sph_pair_term{t.x, t.y};
        };
        auto apply = [&](const sph_pair_term &t) {
            rho = rho + t.a;
            rhon = rhon + t.b;
        };
        auto never = [](bool) {};
        sph_split_body<decltype(term), decltype(apply), decltype(never)> sb{term, apply, never};
        fh = walk_group<CAP, 2 * kTileCap, LP>(T, tile, load, live, s, R, key, j, P, start, test,
                                               sb, mk);
    }
    if (live && lead) {
        RHO[s] = make_float2(rho, rhon);
        if (LP != 16)
            masks[s] = mk.m; // for the relaxation of the same step
    }
    const unsigned full = fh.x, half = lead ? fh.y : 0u;
    report_neighbors(full, half, C);
}

// Its tiles hold positions only: twice the candidates of the other gathers'
// float4 tiles in the same LDS bytes, so denser rows stay in LDS at no cost in
// occupancy (registers allow 7 workgroups per CU either way).
template <bool CAP>
__global__ void __launch_bounds__(kTPB, kGatherMinBlocks)
k_density(const sph_dev_params *__restrict__ Pp, const int *__restrict__ BS,
          const sph_tile_plan *__restrict__ plans, const float2 *__restrict__ POS,
          const unsigned *__restrict__ K, const unsigned *__restrict__ start,
          float2 *__restrict__ RHO, uint4 *__restrict__ masks, sph_dev_counters *__restrict__ C)
{
    __shared__ float2 tile[2 * kTileCap + kSphWalkPad];
    density_tile<CAP, 1>(Pp, BS, plans, POS, K, start, RHO, masks, C, tile, xcd_block());
}

// The fused step's variant with one lane per particle, and four in crowded
// tiles.
template <bool CAP>
__global__ void __launch_bounds__(kTPB, kMixedMinBlocks)
k_density_mixed(const sph_dev_params *__restrict__ Pp, const int *__restrict__ BS,
                sph_tile_plans plans, const float2 *__restrict__ POS,
                const unsigned *__restrict__ K, const unsigned *__restrict__ start,
                float2 *__restrict__ RHO, uint4 *__restrict__ masks,
                sph_dev_counters *__restrict__ C)
{
    __shared__ float2 tile[2 * kTileCap + kSphWalkPad];
    const unsigned listed = plans.crowded_max * 4u;
    if (blockIdx.x < listed) {
        const unsigned k = blockIdx.x / 4u;
        if (k < *plans.crowded_n)
            density_tile<CAP, 4>(Pp, BS, plans.t64, POS, K, start, RHO, masks, C, tile,
                                 plans.crowded[k] * 4u + blockIdx.x % 4u);
        return;
    }
    density_tile<CAP, 1, true>(Pp, BS, plans.t256, POS, K, start, RHO, masks, C, tile,
                               xcd_block(listed));
}

// With four lanes per particle (sph_gather_lanes).
template <bool CAP>
__global__ void __launch_bounds__(kTPB, 1)
k_density_quad(const sph_dev_params *__restrict__ Pp, const int *__restrict__ BS,
               const sph_tile_plan *__restrict__ plans, const float2 *__restrict__ POS,
               const unsigned *__restrict__ K, const unsigned *__restrict__ start,
               float2 *__restrict__ RHO, uint4 *__restrict__ masks,
               sph_dev_counters *__restrict__ C)
{
    __shared__ float2 tile[2 * kTileCap + kSphWalkPad];
    density_tile<CAP, 4>(Pp, BS, plans, POS, K, start, RHO, masks, C, tile, xcd_block());
}

// Sixteen lanes per particle.
template <bool CAP>
__global__ void __launch_bounds__(kTPB, 1)
k_density_row(const sph_dev_params *__restrict__ Pp, const int *__restrict__ BS,
              const float2 *__restrict__ POS, const unsigned *__restrict__ K,
              const unsigned *__restrict__ start, float2 *__restrict__ RHO,
              uint4 *__restrict__ masks, sph_dev_counters *__restrict__ C)
{
    density_tile<CAP, 16>(Pp, BS, nullptr, POS, K, start, RHO, masks, C, nullptr, xcd_block());
}

// Double-density relaxation (src/fluid.c:541-611) in gather form.
// FUSED adds the velocity update (src/fluid.c:642-653): boundary, then
// v = (x - x_prev)/dt clamped, and the histogram of the next sort; without
// FUSED only the relaxed positions are written.
template <bool FUSED, bool CAP, int LP = 1, bool LISTED = false>
__device__ __forceinline__ void
relax_tile(const sph_dev_params *__restrict__ Pp, const int *__restrict__ BS,
           const sph_tile_plan *__restrict__ plans, const float2 *__restrict__ POS,
           const float2 *__restrict__ PREV, const float2 *__restrict__ RHO,
           const unsigned *__restrict__ K, const unsigned *__restrict__ start,
           float2 *__restrict__ out_pos,
           float2 *__restrict__ out_vel, unsigned *__restrict__ out_key,
           unsigned *__restrict__ out_slot, unsigned *__restrict__ cnt,
           const uint4 *__restrict__ masks, sph_dev_counters *__restrict__ C,
           unsigned long long *__restrict__ clock, float4 *tile, unsigned blk,
           const sph_buckets &lists = {})
{
    constexpr unsigned kPer = kTPB / LP; // particles per workgroup
    const unsigned s0 = blk * kPer;
    const unsigned s = s0 + threadIdx.x / LP;
    // the lane's own key and the tile's plan, before the scene
    // parameters (every slot of the grid is inside the arrays)
    const unsigned ks = K[s];
    const int id = lists.rows ? lists.ids[s] : 0;
    const sph_tile_plan T = LP != 16 ? plans[blk] : sph_tile_plan{};
    const sph_dev_params P = Pp[BS[blk / LP]];
    const unsigned s1 = min(s0 + kPer, P.poff + (unsigned)P.n);
    const bool lead = threadIdx.x % LP == 0; // the lane that stores the particle's results
    if (LISTED && s0 < s1 && (T.wide & kCrowded))
        return; // four lanes per particle walk it (a tile of no particle has no plan)
    if (FUSED) {
        add_pad(P, s0, cnt);
        if (s0 == 0 && threadIdx.x == 0)
            atomicAdd(clock, 1ull); // one step of simulated time
    }
    if (s0 >= s1)
        return; // a padding workgroup
    if (FUSED && P.frozen) {
        // frozen scene: keep the position; out_vel already holds the
        // velocity parked by the prediction kernel at this same slot
        if (s < s1 && lead) {
            const float2 a = POS[s];
            out_pos[s] = a;
            const unsigned nk = sph_cell_key(a.x, a.y, P, &C->key_out_of_range);
            out_key[s] = nk;
            claim_slot(s, nk, id, cnt, out_slot, lists);
        }
        return;
    }
    // the lane's own particle and candidate rows, loaded before the staging
    const float2 a = POS[s];
    const float2 ar = RHO[s];
    const bool live = s < s1;
    const unsigned key = live ? ks : P.cell_base; // pad lanes: any valid cell
    const unsigned j = cell_row<LP == 16>(T, live, s, key, P);
    const sph_rows R = sph_row_bounds(key, j, P, start);
    // a neighbour's record carries its pressure and near-pressure
    // (src/fluid.c:563-564), evaluated once per record rather than per pair
    auto load = [&](unsigned g) {
        const float2 p = POS[g], r = RHO[g];
        return make_float4(p.x, p.y, P.k * (r.x - P.rest_density), P.k_near * r.y);
    };
    const float aP = P.k * (ar.x - P.rest_density);
    const float aPn = P.k_near * ar.y;
    float nx = a.x, ny = a.y;
    auto test = [&](float4 b) {
        const float dx = a.x - b.x, ddy = a.y - b.y;
        return dx * dx + ddy * ddy;
    };
    const float h_recip = sph_vgpr(P.h_recip), h = sph_vgpr(P.h), k_spring = sph_vgpr(P.k_spring);
    const double dt2 = (double)(P.dt * P.dt);
    // the pair's displacement (zero when not pushed: n - 0 == n); on_nudge
    // hears whether an uncommon pair takes the 1e-6 nudge, before it
    auto push = [&](float4 b, float dx, float ddy, float r2, auto &&own, auto &&on_nudge) {
        // b - a = -(a - b) exactly in IEEE arithmetic
        const sph_root q = sph_root_common(r2);
        const float D = sph_relax_D(dt2, aP + b.z, aPn + b.w, 1.0f - q.r * h_recip, k_spring, h,
                                    q.r);
        sph_pair_term t{D * -dx * q.rinv, D * -ddy * q.rinv};
        if (__builtin_expect(__ballot(sph_uncommon_pair(r2, kPairLoNudge, P)) != 0ull, 0)) {
            const float rr = sph_sqrt(r2);
            const float r_recip = sph_rcp(rr); // 1.0f / rr
            const float ratio = rr * h_recip;
            const bool moves = ratio < 1.0f && rr > 0.0f;
            const float E = sph_relax_D(dt2, aP + b.z, aPn + b.w, 1.0f - ratio, k_spring, h, rr);
            t.a = moves ? E * -dx * r_recip : 0.0f;
            t.b = moves ? E * -ddy * r_recip : 0.0f;
            on_nudge(rr <= 0.000001f && own());
        }
        return t;
    };
    auto pair = [&](float4 b, auto &&own, auto &&on_nudge) {
        const float dx = a.x - b.x, ddy = a.y - b.y;
        return push(b, dx, ddy, dx * dx + ddy * ddy, own, on_nudge);
    };
    auto nudge = [&](bool yes) {
        nx = yes ? nx + 0.000001f : nx;
        ny = yes ? ny + 0.000001f : ny;
    };
    auto apply = [&](const sph_pair_term &t) {
        nx = nx - t.a;
        ny = ny - t.b;
    };
    if constexpr (LP == 1) {
        auto body = [&](unsigned, float4 b, auto &&own) { apply(pair(b, own, nudge)); };
        if (FUSED) { // the density pass of this step walked the same neighbour set
            sph_masks_replay mk{live ? masks[s] : make_uint4(0u, 0u, 0u, 0u)};
            walk_group<CAP, kTileCap>(T, tile, load, live, s, R, key, j, P, start, test, body, mk);
        } else {
            sph_masks_none mk;
            walk_group<CAP, kTileCap>(T, tile, load, live, s, R, key, j, P, start, test, body, mk);
        }
    } else if constexpr (LP == 16) {
        auto wide = [&](float4 b, bool cand, auto &&own, bool &accepted, bool &nudged) {
            const float dx = a.x - b.x, ddy = a.y - b.y;
            const float r2 = dx * dx + ddy * ddy;
            accepted = cand && !(r2 > P.h2);
            const sph_pair_term t = push(b, dx, ddy, accepted ? r2 : 0.5f * P.h2, own,
                                         [&](bool yes) { nudged = yes; });
            nudged = nudged && accepted;
            return sph_pair_term{accepted ? t.a : 0.0f, accepted ? t.b : 0.0f};
        };
        sph_walk_wide<CAP>(s, live, R, P.bucket_cap, load, wide, apply, nudge);
    } else {
        auto term = [&](unsigned, float4 b, auto &&own, bool &nudged) {
            return pair(b, own, [&](bool yes) { nudged = yes; });
        };
        sph_split_body<decltype(term), decltype(apply), decltype(nudge)> sb{term, apply, nudge};
        if (FUSED) {
            sph_masks_replay mk{live ? masks[s] : make_uint4(0u, 0u, 0u, 0u)};
            walk_group<CAP, kTileCap, LP>(T, tile, load, live, s, R, key, j, P, start, test, sb,
                                          mk);
        } else {
            sph_masks_none mk;
            walk_group<CAP, kTileCap, LP>(T, tile, load, live, s, R, key, j, P, start, test, sb,
                                          mk);
        }
    }
    if (!live || !lead)
        return;
    if (FUSED) {
        sph_boundary(nx, ny, P);
        const float2 q = PREV[s];
        float vx = (nx - q.x) / P.dt;
        float vy = (ny - q.y) / P.dt;
        sph_check_velocity(vx, vy);
        out_vel[s] = make_float2(vx, vy);
        if (!(isfinite(nx) && isfinite(ny)))
            atomicAdd(&C->nonfinite, 1ull);
        const unsigned nk = sph_cell_key(nx, ny, P, &C->key_out_of_range);
        out_key[s] = nk;
        claim_slot(s, nk, id, cnt, out_slot, lists);
    }
    out_pos[s] = make_float2(nx, ny);
}

template <bool FUSED, bool CAP>
__global__ void __launch_bounds__(kTPB, CAP ? kGatherMinBlocks - 1 : kGatherMinBlocks)
k_relax(const sph_dev_params *__restrict__ Pp, const int *__restrict__ BS,
        const sph_tile_plan *__restrict__ plans, const float2 *__restrict__ POS,
        const float2 *__restrict__ PREV, const float2 *__restrict__ RHO,
        const unsigned *__restrict__ K, const unsigned *__restrict__ start,
        float2 *__restrict__ out_pos,
        float2 *__restrict__ out_vel, unsigned *__restrict__ out_key,
        unsigned *__restrict__ out_slot, unsigned *__restrict__ cnt,
        const uint4 *__restrict__ masks, sph_dev_counters *__restrict__ C,
        unsigned long long *__restrict__ clock)
{
    __shared__ float4 tile[kTileCap + kSphWalkPad];
    relax_tile<FUSED, CAP, 1>(Pp, BS, plans, POS, PREV, RHO, K, start, out_pos, out_vel, out_key,
                              out_slot, cnt, masks, C, clock, tile, xcd_block());
}

// The fused step's variant with one lane per particle, and four in crowded
// tiles.
template <bool CAP>
__global__ void __launch_bounds__(kTPB, CAP ? kMixedMinBlocks - 1 : kMixedMinBlocks)
k_relax_mixed(const sph_dev_params *__restrict__ Pp, const int *__restrict__ BS,
              sph_tile_plans plans, const float2 *__restrict__ POS,
              const float2 *__restrict__ PREV, const float2 *__restrict__ RHO,
              const unsigned *__restrict__ K, const unsigned *__restrict__ start,
              float2 *__restrict__ out_pos, float2 *__restrict__ out_vel,
              unsigned *__restrict__ out_key, unsigned *__restrict__ out_slot,
              unsigned *__restrict__ cnt, const uint4 *__restrict__ masks,
              sph_dev_counters *__restrict__ C, unsigned long long *__restrict__ clock)
{
    __shared__ float4 tile[kTileCap + kSphWalkPad];
    const unsigned listed = plans.crowded_max * 4u;
    if (blockIdx.x < listed) {
        const unsigned k = blockIdx.x / 4u;
        if (k < *plans.crowded_n)
            relax_tile<true, CAP, 4>(Pp, BS, plans.t64, POS, PREV, RHO, K, start, out_pos,
                                     out_vel, out_key, out_slot, cnt, masks, C, clock, tile,
                                     plans.crowded[k] * 4u + blockIdx.x % 4u);
        return;
    }
    relax_tile<true, CAP, 1, true>(Pp, BS, plans.t256, POS, PREV, RHO, K, start, out_pos, out_vel,
                                   out_key, out_slot, cnt, masks, C, clock, tile,
                                   xcd_block(listed));
}

// With four lanes per particle (sph_gather_lanes).
template <bool CAP>
__global__ void __launch_bounds__(kTPB, 1)
k_relax_quad(const sph_dev_params *__restrict__ Pp, const int *__restrict__ BS,
             const sph_tile_plan *__restrict__ plans, const float2 *__restrict__ POS,
             const float2 *__restrict__ PREV, const float2 *__restrict__ RHO,
             const unsigned *__restrict__ K, const unsigned *__restrict__ start,
             float2 *__restrict__ out_pos, float2 *__restrict__ out_vel,
             unsigned *__restrict__ out_key, unsigned *__restrict__ out_slot,
             unsigned *__restrict__ cnt, const uint4 *__restrict__ masks,
             sph_dev_counters *__restrict__ C, unsigned long long *__restrict__ clock)
{
    __shared__ float4 tile[kTileCap + kSphWalkPad];
    relax_tile<true, CAP, 4>(Pp, BS, plans, POS, PREV, RHO, K, start, out_pos, out_vel, out_key,
                             out_slot, cnt, masks, C, clock, tile, xcd_block());
}

// Sixteen lanes per particle.
template <bool CAP>
__global__ void __launch_bounds__(kTPB, 1)
k_relax_row(const sph_dev_params *__restrict__ Pp, const int *__restrict__ BS,
            const float2 *__restrict__ POS, const float2 *__restrict__ PREV,
            const float2 *__restrict__ RHO, const unsigned *__restrict__ K,
            const unsigned *__restrict__ start, float2 *__restrict__ out_pos,
            float2 *__restrict__ out_vel, unsigned *__restrict__ out_key,
            unsigned *__restrict__ out_slot, unsigned *__restrict__ cnt,
            const uint4 *__restrict__ masks, sph_dev_counters *__restrict__ C,
            unsigned long long *__restrict__ clock, sph_buckets lists)
{
    relax_tile<true, CAP, 16>(Pp, BS, nullptr, POS, PREV, RHO, K, start, out_pos, out_vel, out_key,
                              out_slot, cnt, masks, C, clock, nullptr, xcd_block(), lists);
}

// One piece of a result to pinned host memory and, when the host can read it,
// the piece's flag: the host copies a piece on while the next ones cross the
// link, which bounds this kernel (23 us a MB).
__global__ void __launch_bounds__(kTPB)
k_to_host(const uint4 *__restrict__ src, uint4 *__restrict__ dst, size_t bytes,
          unsigned *__restrict__ flags, unsigned mark)
{
    constexpr unsigned kWords = kHostPiece / sizeof(uint4), kEach = kWords / kTPB;
    const size_t w0 = (size_t)blockIdx.x * kWords, words = bytes / sizeof(uint4);
    const unsigned t = threadIdx.x;
    uint4 v[kEach];
#pragma unroll
    for (unsigned u = 0; u < kEach; u++)
        if (w0 + u * kTPB + t < words)
            v[u] = src[w0 + u * kTPB + t];
#pragma unroll
    for (unsigned u = 0; u < kEach; u++)
        if (w0 + u * kTPB + t < words)
            dst[w0 + u * kTPB + t] = v[u];
    const unsigned rest = (unsigned)(bytes % sizeof(uint4)) / 4u;
    if (blockIdx.x == gridDim.x - 1 && t < rest)
        reinterpret_cast<unsigned *>(dst + words)[t] =
            reinterpret_cast<const unsigned *>(src + words)[t];
    __threadfence_system();
    __syncthreads();
    if (t == 0)
        __hip_atomic_store(&flags[blockIdx.x], mark, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// Reference coordinate packing (src/fluid.c:356-363), written by id.
__global__ void __launch_bounds__(kTPB)
k_pack_coords(const sph_dev_params *__restrict__ Pp, const int *__restrict__ BS,
              const float2 *__restrict__ POS, const int *__restrict__ ID,
              short *__restrict__ out)
{
    const unsigned blk = xcd_block();
    const sph_dev_params &P = Pp[BS[blk]];
    const unsigned s = blk * kTPB + threadIdx.x;
    if (s >= P.poff + (unsigned)P.n)
        return;
    const size_t id = P.uoff + (unsigned)ID[s];
    const float2 p = POS[s];
    out[2 * id] = (short)((2.0f * p.x / P.max_x - 1.0f) * 32767.0f);
    out[2 * id + 1] = (short)((2.0f * p.y / P.max_y - 1.0f) * 32767.0f);
}

// Neighbour sets of the current hash, written by id (small-N read-back for
// tests): full set in canonical order, and the half-list length the
// reference would hold for each particle.
__global__ void __launch_bounds__(kTPB)
k_neighbor_lists(const sph_dev_params *__restrict__ Pp, const int *__restrict__ BS,
                 const float2 *__restrict__ POS, const unsigned *__restrict__ K,
                 const int *__restrict__ ID, const unsigned *__restrict__ start, int stride,
                 int *__restrict__ full_by_id, int *__restrict__ half_by_id,
                 int *__restrict__ ids_by_id)
{
    const unsigned blk = xcd_block();
    const sph_dev_params P = Pp[BS[blk]];
    const unsigned s = blk * kTPB + threadIdx.x;
    if (s >= P.poff + (unsigned)P.n)
        return;
    const int me = (int)P.uoff + ID[s];
    const float2 a = POS[s];
    int full = 0, half = 0;
    // the bucket cap: rank in the cell = sorted position - the cell's start
    auto dropped = [&](unsigned k) { return P.bucket_cap && k - start[K[k]] >= P.bucket_cap; };
    if (!dropped(s))
        sph_walk(s, K[s], P, start, global_src<float2>([&](unsigned g) { return POS[g]; }),
                 [&](unsigned k, int dy, unsigned b1, unsigned b2, float2 b) {
                     const float dx = a.x - b.x, ddy = a.y - b.y;
                     if (k == s || dx * dx + ddy * ddy > P.h2 || dropped(k))
                         return;
                     if (full < stride)
                         ids_by_id[(size_t)me * stride + full] = ID[k];
                     full++;
                     half += sph_owns(k, s, dy, b1, b2);
                 });
    full_by_id[me] = full;
    half_by_id[me] = half;
}

// dst[pos_of_id[id_src[k]]] = src[k]: re-canonicalise auxiliary fields.
__global__ void __launch_bounds__(kTPB)
k_pos_of_id(const sph_dev_params *__restrict__ Pp, const int *__restrict__ BS,
            const int *__restrict__ ID, int *__restrict__ pos_of_id)
{
    const unsigned blk = xcd_block();
    const sph_dev_params &P = Pp[BS[blk]];
    const unsigned s = blk * kTPB + threadIdx.x;
    if (s < P.poff + (unsigned)P.n)
        pos_of_id[P.uoff + (unsigned)ID[s]] = (int)s;
}

__global__ void __launch_bounds__(kTPB)
k_permute_by_id(const sph_dev_params *__restrict__ Pp, const int *__restrict__ BS,
                const int *__restrict__ id_src, const int *__restrict__ pos_of_id,
                sph_reorder_fields<2> f)
{
    const unsigned blk = xcd_block();
    const sph_dev_params &P = Pp[BS[blk]];
    const unsigned k = blk * kTPB + threadIdx.x;
    if (k >= P.poff + (unsigned)P.n)
        return;
    const int d = pos_of_id[P.uoff + (unsigned)id_src[k]];
#pragma unroll
    for (int q = 0; q < 2; q++)
        f.dst[q][d] = f.src[q][k];
}

// ---------------------------------------------------------------------------
// Host-side launchers.  `slots` is the padded slot count of all scenes
// (a multiple of kTPB); BS maps each logical workgroup to its scene.

#define GRID(slots) dim3((unsigned)((slots) / kTPB))

namespace {

// Start/stop events for the next launch (sph_set_next_launch_events).
thread_local hipEvent_t g_next_start = nullptr, g_next_stop = nullptr;

// Launch on `st`; when timing events are pending, through
// hipExtLaunchKernelGGL, whose events carry the kernel's own start and end
// times (no dispatch latency).
template <class F, class... Args>
void launch(F kernel, dim3 grid, dim3 block, hipStream_t st, Args... args)
{
    if (g_next_start) {
        hipEvent_t a = g_next_start, b = g_next_stop;
        g_next_start = g_next_stop = nullptr;
        hipExtLaunchKernelGGL(kernel, grid, block, 0, st, a, b, 0, args...);
    } else {
        hipLaunchKernelGGL(kernel, grid, block, 0, st, args...);
    }
}

} // namespace

// Exhaustive checks of sph_sqrt (FN 0) against sqrtf and sph_rcp (FN 1)
// against IEEE division, and of sph_root_common's root (FN 0) and reciprocal
// root (FN 1): every float with bit pattern in [lo, hi) (grid-stride; the
// last three over their domains), bit for bit (any NaN equals any NaN).
__device__ __attribute__((noinline)) float ieee_sqrt(float x) { return sqrtf(x); }
__device__ __attribute__((noinline)) float ieee_rcp(float x) { return 1.0f / x; }

template <int FN>
__global__ void __launch_bounds__(256)
k_selftest_math(unsigned lo, unsigned hi, unsigned long long *__restrict__ bad)
{
    unsigned long long nbad = 0;
    const unsigned long long stride = (unsigned long long)gridDim.x * blockDim.x;
    for (unsigned long long b = lo + (unsigned long long)blockIdx.x * blockDim.x + threadIdx.x;
         b < hi; b += stride) {
        const float x = __uint_as_float((unsigned)b);
        auto differ = [](float got, float want) {
            return __float_as_uint(got) != __float_as_uint(want) && !(got != got && want != want);
        };
        bool bad_x = false;
        if (FN == 0)
            bad_x = differ(sph_sqrt(x), ieee_sqrt(x));
        else if (sph_rcp_domain(x))
            bad_x = differ(sph_rcp(x), ieee_rcp(x));
        if (x >= 0x1p-96f && x <= 0x1p120f) {
            const sph_root q = sph_root_common(x);
            const float r = ieee_sqrt(x);
            bad_x = bad_x || differ(FN == 0 ? q.r : q.rinv, FN == 0 ? r : ieee_rcp(r));
        }
        nbad += bad_x ? 1u : 0u;
    }
    for (int o = 32; o > 0; o >>= 1)
        nbad += __shfl_xor(nbad, o, 64);
    if ((threadIdx.x & 63u) == 0 && nbad)
        atomicAdd(bad, nbad);
}

void sph_launch_selftest_math(hipStream_t st, int fn, unsigned lo, unsigned hi,
                              unsigned long long *bad)
{
    if (fn == 0)
        launch(k_selftest_math<0>, dim3(4096), dim3(256), st, lo, hi, bad);
    else
        launch(k_selftest_math<1>, dim3(4096), dim3(256), st, lo, hi, bad);
}

void sph_set_next_launch_events(hipEvent_t start, hipEvent_t stop)
{
    g_next_start = start;
    g_next_stop = stop;
}

__global__ void __launch_bounds__(kTPB)
k_restore(const sph_dev_params *__restrict__ Pp, const int *__restrict__ BS,
          const int *__restrict__ flags, sph_restore_args a)
{
    const unsigned blk = blockIdx.x;
    const int scene = BS[blk];
    if (!flags[scene])
        return;
    const sph_dev_params &P = Pp[scene];
    const unsigned s = blk * kTPB + threadIdx.x;
#pragma unroll
    for (int q = 0; q < 4; q++)
        a.dst[q][s] = a.src[q][s];
    a.id_dst[s] = a.id_src[s];
    a.key_dst[s] = a.key_src[s];
    // the scene's cell starts, shared by all of its workgroups: one workgroup
    // copying them alone is a chain of ncells / 256 dependent rounds (920 us
    // for the 960,000 cells of the 1M dam break, against 17 us shared)
    const unsigned wg = blk - P.poff / kTPB, nwg = ((unsigned)P.n + P.pad) / kTPB;
    for (unsigned long long c = wg * kTPB + threadIdx.x; c <= P.ncells; c += nwg * kTPB)
        a.start_dst[P.cell_base + c] = a.start_src[P.cell_base + c];
}

// Workgroup b copies 1,024 16-byte units of the array that its place in the
// launch falls into.  (As one memcpy each, the eight arrays of a snapshot of
// 1M particles were eight launches of 3 - 4 us and, the host not keeping up
// with them, gaps of 7 us between; one launch takes 21 us.)
constexpr unsigned kCopyUnits = 4 * kTPB;
__device__ __host__ __forceinline__ unsigned copy_groups(unsigned n16)
{
    return (n16 + kCopyUnits - 1) / kCopyUnits;
}

__global__ void __launch_bounds__(kTPB)
k_copy(sph_copy_set c)
{
    unsigned b = blockIdx.x;
    if (b == 0 && threadIdx.x == 0 && c.word_src)
        *c.word_dst = *c.word_src;
#pragma unroll
    for (int i = 0; i < kCopyArrays; i++) {
        const unsigned g = i < c.count ? copy_groups(c.n16[i]) : 0u;
        if (b < g) {
            const uint4 *src = static_cast<const uint4 *>(c.src[i]) + b * (size_t)kCopyUnits;
            uint4 *dst = static_cast<uint4 *>(c.dst[i]) + b * (size_t)kCopyUnits;
            const unsigned n = min(c.n16[i] - b * kCopyUnits, kCopyUnits);
            uint4 v[4];
#pragma unroll
            for (unsigned u = 0; u < 4; u++)
                if (threadIdx.x + u * kTPB < n)
                    v[u] = src[threadIdx.x + u * kTPB];
#pragma unroll
            for (unsigned u = 0; u < 4; u++)
                if (threadIdx.x + u * kTPB < n)
                    dst[threadIdx.x + u * kTPB] = v[u];
            return;
        }
        b -= g;
    }
}

__global__ void __launch_bounds__(kTPB)
k_gather_state(const sph_dev_params *__restrict__ Pp, const int *__restrict__ BS,
               const float2 *__restrict__ POS, const float2 *__restrict__ VEL,
               const int *__restrict__ ID, float4 *__restrict__ out)
{
    const unsigned blk = xcd_block();
    const sph_dev_params &P = Pp[BS[blk]];
    const unsigned s = blk * kTPB + threadIdx.x;
    if (s >= P.poff + (unsigned)P.n)
        return;
    const float2 p = POS[s], v = VEL[s];
    out[P.uoff + (unsigned)ID[s]] = make_float4(p.x, p.y, v.x, v.y);
}

// The reference's particle records (fluid_particle, 13 words) by caller
// index: position, velocity, a and id from the canonical order (ID0); x_prev,
// density and the pressures (src/fluid.c:563-564) from the auxiliary fields'
// order (IDA: ID0, or ID1 after fused steps).
__global__ void __launch_bounds__(kTPB)
k_gather_aos(const sph_dev_params *__restrict__ Pp, const int *__restrict__ BS,
             const float2 *__restrict__ POS, const float2 *__restrict__ VEL,
             const int *__restrict__ ID0, const float2 *__restrict__ PREV,
             const float2 *__restrict__ RHO, const int *__restrict__ IDA,
             const float2 *__restrict__ ACC, float *__restrict__ out)
{
    const unsigned blk = xcd_block();
    const sph_dev_params &P = Pp[BS[blk]];
    const unsigned s = blk * kTPB + threadIdx.x;
    if (s >= P.poff + (unsigned)P.n)
        return;
    const int id = ID0[s];
    const size_t g = P.uoff + (unsigned)id;
    const float2 p = POS[s], v = VEL[s], a = ACC[g];
    float *r = out + 13 * g;
    r[2] = p.x;
    r[3] = p.y;
    r[4] = v.x;
    r[5] = v.y;
    r[6] = a.x;
    r[7] = a.y;
    r[12] = __int_as_float(id);
    const float2 q = PREV[s], rho = RHO[s];
    float *r2 = out + 13 * ((size_t)P.uoff + (unsigned)IDA[s]);
    r2[0] = q.x;
    r2[1] = q.y;
    r2[8] = rho.x;
    r2[9] = rho.y;
    r2[10] = P.k * (rho.x - P.rest_density);
    r2[11] = P.k_near * rho.y;
}

// Positions by caller index (scene offset + id), for position-only read-back.
__global__ void __launch_bounds__(kTPB)
k_gather_xy(const sph_dev_params *__restrict__ Pp, const int *__restrict__ BS,
            const float2 *__restrict__ POS, const int *__restrict__ ID, float2 *__restrict__ out)
{
    const unsigned blk = xcd_block();
    const sph_dev_params &P = Pp[BS[blk]];
    const unsigned s = blk * kTPB + threadIdx.x;
    if (s >= P.poff + (unsigned)P.n)
        return;
    out[P.uoff + (unsigned)ID[s]] = POS[s];
}

__global__ void __launch_bounds__(kTPB)
k_load_state(const sph_dev_params *__restrict__ Pp, const int *__restrict__ BS,
             const float4 *__restrict__ in, float2 *__restrict__ POS, float2 *__restrict__ VEL,
             float2 *__restrict__ PREV, float2 *__restrict__ RHO, int *__restrict__ ID)
{
    const unsigned blk = xcd_block();
    const sph_dev_params &P = Pp[BS[blk]];
    const unsigned s = blk * kTPB + threadIdx.x;
    if (s >= P.poff + (unsigned)P.n)
        return;
    const unsigned id = s - P.poff;
    const float4 q = in[P.uoff + id];
    POS[s] = make_float2(q.x, q.y);
    PREV[s] = make_float2(q.x, q.y);
    VEL[s] = make_float2(q.z, q.w);
    RHO[s] = make_float2(0.0f, 0.0f);
    ID[s] = (int)id;
}

// Several lanes per particle in small contexts.  There the gather launches are
// short of work, and a launch's time is set by its slowest workgroups: the
// dense bottom rows of a settling column, whose walks the lanes share.  Sixteen
// when there is at most half a 256-slot tile per CU (32,768 particles on 256
// CUs), four up to two (131,072), one beyond, where the lanes' repeated
// per-particle work costs more than the shorter walks gain.  Measured on dam
// breaks, us a step over steps 21-84 / 251-314 (one lane, four, sixteen):
//   1.5k   56 / 90     39 / 57     24 / 31
//   4k     54 / 133    40 / 77     24 / 39
//   16k    57 / 139    43 / 80     32 / 51
//   33k    56 / 133    43 / 79     44 / 60
//   66k    56 / 134    48 / 81     63 / 83
//   131k   60 / 135    68 / 85     96 / 118
//   262k   67 / 141    97 / 119   154 / 185
// (sixteen lanes with k_sort_small up to 33k; 39 / 58 at 16k without).
// SPH_SMALL_SCENE_LANES=1 turns the several-lane paths off.
#ifndef SPH_SMALL_SCENE_LANES
#define SPH_SMALL_SCENE_LANES 16
#endif
static unsigned device_cus()
{
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) {
        (void)hipGetLastError();
        return 0;
    }
    return cus > 0 ? (unsigned)cus : 0u;
}

int sph_gather_lanes(unsigned slots)
{
    const unsigned long long tiles = slots / kTPB, n = device_cus();
    if (!n)
        return 1;
    const int lanes = 2ull * tiles <= n ? 16 : tiles <= 2ull * n ? 4 : 1;
    return lanes <= SPH_SMALL_SCENE_LANES ? lanes : SPH_SMALL_SCENE_LANES;
}

// Up to four tiles per CU (262,144 particles on 256 CUs) all workgroups are
// resident at once; beyond, the mixed kernels' five a CU, where the one-lane
// kernels have seven, cost more while the fluid is evenly spread than the lists
// gain (320k particles: 79 against 74 us a step over steps 21-84, 89 against 100
// over 101-164), and from 1M on the chip is busy with the sum of the work (1M,
// steps 501-600: 290 against 247).
bool sph_lists_crowded(unsigned slots, int lanes)
{
    return lanes == 1 && slots / kTPB <= 4u * device_cus();
}

// The mixed kernels' workgroups: a quarter of a listed tile each, then the tiles.
static dim3 mixed_grid(unsigned slots, const sph_tile_plans &plans)
{
    return dim3(slots / kTPB + 4u * plans.crowded_max);
}

void sph_launch_visc_predict(hipStream_t st, unsigned slots, bool grav, bool visc, bool pred,
                             bool cap, const sph_dev_params *P, const int *BS,
                             const sph_tile_plans &plans, const float2 *POS, const float2 *VEL,
                             const unsigned *K, const unsigned *start, float2 *opos,
                             unsigned *okey, unsigned *oslot, unsigned *cnt,
                             sph_dev_counters *C, const unsigned long long *clock,
                             float2 *held_vel, int lanes, const sph_buckets &lists)
{
#define VP(G, V, R, CAP)                                                                         \
    launch(k_visc_predict<G, V, R, CAP>, GRID(slots), kTPB, st, P, BS, plans.t256, POS, VEL, K,  \
           start, opos, okey, oslot, cnt, C, clock, held_vel)
#define VPM(CAP)                                                                                 \
    launch(k_visc_predict_mixed<CAP>, mixed_grid(slots, plans), kTPB, st, P, BS, plans, POS,     \
           VEL, K, start, opos, okey, oslot, cnt, C, clock, held_vel)
#define VP4(CAP)                                                                                 \
    launch(k_visc_predict_quad<CAP>, GRID(4 * (slots)), kTPB, st, P, BS, plans.t64, POS, VEL, K, \
           start, opos, okey, oslot, cnt, C, clock, held_vel)
#define VP16(CAP)                                                                                \
    launch(k_visc_predict_row<CAP>, GRID(16 * (slots)), kTPB, st, P, BS, POS, VEL, K, start,     \
           opos, okey, oslot, cnt, C, clock, held_vel, lists)
#define VPC(G, V, R)                                                                             \
    do {                                                                                         \
        if (cap)                                                                                 \
            VP(G, V, R, true);                                                                   \
        else                                                                                     \
            VP(G, V, R, false);                                                                  \
    } while (0)
    // without viscosity the walk does not run: no capped variant; several lanes
    // per particle for the fused step's variant only
    if (grav && visc && pred && lanes == 16) {
        if (cap)
            VP16(true);
        else
            VP16(false);
    } else if (grav && visc && pred && lanes == 4) {
        if (cap)
            VP4(true);
        else
            VP4(false);
    } else if (grav && visc && pred && plans.crowded) {
        if (cap)
            VPM(true);
        else
            VPM(false);
    } else if (grav && visc && pred)
        VPC(true, true, true);
    else if (grav && !visc && pred)
        VP(true, false, true, false);
    else if (!grav && visc && !pred)
        VPC(false, true, false);
    else if (!grav && visc && pred)
        VPC(false, true, true);
    else if (!grav && !visc && pred)
        VP(false, false, true, false);
    else
        VPC(true, true, false);
#undef VP16
#undef VP4
#undef VPM
#undef VPC
#undef VP
}

void sph_launch_gravity(hipStream_t st, unsigned slots, const sph_dev_params *P, const int *BS,
                        float2 *VEL, float2 *RHO)
{
    launch(k_gravity, GRID(slots), kTPB, st, P, BS, VEL, RHO);
}

void sph_launch_predict(hipStream_t st, unsigned slots, const sph_dev_params *P, const int *BS,
                        float2 *POS, const float2 *VEL, float2 *PREV)
{
    launch(k_predict, GRID(slots), kTPB, st, P, BS, POS, VEL, PREV);
}

void sph_launch_update_velocities(hipStream_t st, unsigned slots, const sph_dev_params *P,
                                  const int *BS, float2 *POS, float2 *VEL, const float2 *PREV)
{
    launch(k_update_velocities, GRID(slots), kTPB, st, P, BS, POS, VEL, PREV);
}

void sph_launch_key_hist(hipStream_t st, unsigned slots, const sph_dev_params *P, const int *BS,
                         const float2 *POS, unsigned *okey, unsigned *oslot, unsigned *cnt,
                         sph_dev_counters *C)
{
    launch(k_key_hist, GRID(slots), kTPB, st, P, BS, POS, okey, oslot, cnt, C);
}

unsigned sph_scan_blocks(unsigned m)
{
    return (unsigned)(((unsigned long long)m + kScanTile - 1) / kScanTile); // m near 2^32: no wrap
}

size_t sph_scan_padded(unsigned m) { return (size_t)sph_scan_blocks(m) * kScanTile; }

void sph_launch_scan_reduce(hipStream_t st, const unsigned *cnt, unsigned m, unsigned *bsum)
{
    launch(k_scan_reduce, dim3(sph_scan_blocks(m)), kScanThreads, st,
           reinterpret_cast<const uint4 *>(cnt), bsum);
}

void sph_launch_scan_apply(hipStream_t st, unsigned *cnt, unsigned m, const unsigned *bsum,
                           unsigned *start)
{
    launch(k_scan_apply, dim3(sph_scan_blocks(m)), kScanThreads, st,
           reinterpret_cast<uint4 *>(cnt), bsum, reinterpret_cast<uint4 *>(start));
}

#ifndef SPH_SCAN_SINGLE
#define SPH_SCAN_SINGLE 1
#endif
bool sph_scan_single_fits(unsigned m)
{
    return SPH_SCAN_SINGLE && sph_scan_padded(m) <= kScanSingle;
}

void sph_launch_scan_single(hipStream_t st, unsigned *cnt, unsigned m, unsigned *start)
{
    launch(k_scan_single, dim3(1), kScanSingleThreads, st, reinterpret_cast<uint4 *>(cnt),
           (unsigned)sph_scan_padded(m), reinterpret_cast<uint4 *>(start));
}

void sph_launch_scatter(hipStream_t st, unsigned slots, const sph_dev_params *P, const int *BS,
                        const unsigned *key, const unsigned *slot, const unsigned *start,
                        const int *id_src, int *perm_src, int *perm_id, unsigned *key_dst,
                        const sph_tile_plans &plans)
{
    launch(k_scatter, GRID(slots), kTPB, st, P, BS, key, slot, start, id_src, perm_src, perm_id,
           key_dst, plans.crowded_n);
}

void sph_launch_reorder2(hipStream_t st, unsigned slots, const sph_dev_params *P, const int *BS,
                         const unsigned *start, const int *perm_src, const int *perm_id,
                         const unsigned *skey, sph_reorder_fields<2> f, int *id_dst,
                         const sph_tile_plans &plans, sph_dev_counters *C)
{
    const unsigned planners = plan_groups(slots, plans);
    launch(k_reorder<2>, dim3(planners + slots / kTPB), kTPB, st, P, BS, start, perm_src, perm_id,
           skey, f, id_dst, planners, plans, C);
}

void sph_launch_reorder4(hipStream_t st, unsigned slots, const sph_dev_params *P, const int *BS,
                         const unsigned *start, const int *perm_src, const int *perm_id,
                         const unsigned *skey, sph_reorder_fields<4> f, int *id_dst,
                         const sph_tile_plans &plans, sph_dev_counters *C)
{
    const unsigned planners = plan_groups(slots, plans);
    launch(k_reorder<4>, dim3(planners + slots / kTPB), kTPB, st, P, BS, start, perm_src, perm_id,
           skey, f, id_dst, planners, plans, C);
}

bool sph_sort_small_fits(unsigned m, int lanes)
{
    return lanes == 16 && sph_scan_padded(m) <= kSmallCounts;
}

void sph_launch_sort_small(hipStream_t st, unsigned slots, const sph_dev_params *P, const int *BS,
                           const unsigned *key, const unsigned *cnt, unsigned *cnt_next,
                           unsigned m, unsigned *start, const sph_buckets &lists,
                           sph_reorder_fields<2> f, int *id_dst, unsigned *key_dst,
                           sph_dev_counters *C)
{
    const unsigned mp = (unsigned)sph_scan_padded(m);
#define SORT(SEG, TPB)                                                                           \
    launch(k_sort_small<SEG, TPB>, GRID(slots), TPB, st, P, BS, key,                             \
           reinterpret_cast<const uint4 *>(cnt), reinterpret_cast<uint4 *>(cnt_next), mp,        \
           reinterpret_cast<uint4 *>(start), lists, f, id_dst, key_dst, C)
    if (mp <= 2048u)
        SORT(8, 256);
    else if (mp <= 4096u)
        SORT(16, 256);
    else if (mp <= 8192u)
        SORT(16, 512);
    else if (mp <= 16384u)
        SORT(16, 1024);
    else
        SORT(32, 1024);
#undef SORT
}

void sph_launch_plan(hipStream_t st, unsigned slots, const sph_dev_params *P, const int *BS,
                     const unsigned *start, const unsigned *skey, const sph_tile_plans &plans)
{
    launch(k_plan, dim3(plan_groups(slots, plans)), kTPB, st, P, BS, slots / kTPB, start, skey,
           plans);
}

void sph_launch_density(hipStream_t st, unsigned slots, bool cap, const sph_dev_params *P,
                        const int *BS, const sph_tile_plans &plans, const float2 *POS,
                        const unsigned *K, const unsigned *start, float2 *RHO, uint4 *masks,
                        sph_dev_counters *C, int lanes)
{
    if (lanes == 16 && cap)
        launch(k_density_row<true>, GRID(16 * slots), kTPB, st, P, BS, POS, K, start, RHO, masks,
               C);
    else if (lanes == 16)
        launch(k_density_row<false>, GRID(16 * slots), kTPB, st, P, BS, POS, K, start, RHO, masks,
               C);
    else if (lanes == 4 && cap)
        launch(k_density_quad<true>, GRID(4 * (slots)), kTPB, st, P, BS, plans.t64, POS, K, start,
               RHO, masks, C);
    else if (lanes == 4)
        launch(k_density_quad<false>, GRID(4 * (slots)), kTPB, st, P, BS, plans.t64, POS, K,
               start, RHO, masks, C);
    else if (plans.crowded && cap)
        launch(k_density_mixed<true>, mixed_grid(slots, plans), kTPB, st, P, BS, plans, POS, K,
               start, RHO, masks, C);
    else if (plans.crowded)
        launch(k_density_mixed<false>, mixed_grid(slots, plans), kTPB, st, P, BS, plans, POS, K,
               start, RHO, masks, C);
    else if (cap)
        launch(k_density<true>, GRID(slots), kTPB, st, P, BS, plans.t256, POS, K, start, RHO,
               masks, C);
    else
        launch(k_density<false>, GRID(slots), kTPB, st, P, BS, plans.t256, POS, K, start, RHO,
               masks, C);
}

void sph_launch_relax(hipStream_t st, unsigned slots, bool fused, bool cap,
                      const sph_dev_params *P, const int *BS, const sph_tile_plans &plans,
                      const float2 *POS, const float2 *PREV, const float2 *RHO, const unsigned *K,
                      const unsigned *start, float2 *opos, float2 *ovel, unsigned *okey,
                      unsigned *oslot, unsigned *cnt, const uint4 *masks, sph_dev_counters *C,
                      unsigned long long *clock, int lanes, const sph_buckets &lists)
{
#define RL(F, CAP)                                                                               \
    launch(k_relax<F, CAP>, GRID(slots), kTPB, st, P, BS, plans.t256, POS, PREV, RHO, K, start,  \
           opos, ovel, okey, oslot, cnt, masks, C, clock)
#define RLM(CAP)                                                                                 \
    launch(k_relax_mixed<CAP>, mixed_grid(slots, plans), kTPB, st, P, BS, plans, POS, PREV, RHO, \
           K, start, opos, ovel, okey, oslot, cnt, masks, C, clock)
#define RL4(CAP)                                                                                 \
    launch(k_relax_quad<CAP>, GRID(4 * (slots)), kTPB, st, P, BS, plans.t64, POS, PREV, RHO, K,  \
           start, opos, ovel, okey, oslot, cnt, masks, C, clock)
#define RL16(CAP)                                                                                \
    launch(k_relax_row<CAP>, GRID(16 * (slots)), kTPB, st, P, BS, POS, PREV, RHO, K, start,      \
           opos, ovel, okey, oslot, cnt, masks, C, clock, lists)
    // several lanes per particle for the fused step's variant only
    if (fused && lanes == 16 && cap)
        RL16(true);
    else if (fused && lanes == 16)
        RL16(false);
    else if (fused && lanes == 4 && cap)
        RL4(true);
    else if (fused && lanes == 4)
        RL4(false);
    else if (fused && plans.crowded && cap)
        RLM(true);
    else if (fused && plans.crowded)
        RLM(false);
    else if (fused && cap)
        RL(true, true);
    else if (fused)
        RL(true, false);
    else if (cap)
        RL(false, true);
    else
        RL(false, false);
#undef RL16
#undef RL4
#undef RLM
#undef RL
}

void sph_launch_to_host(hipStream_t st, const void *src, void *dst, size_t bytes,
                        unsigned *flags, unsigned mark)
{
    launch(k_to_host, dim3((unsigned)((bytes + kHostPiece - 1) / kHostPiece)), kTPB, st,
           (const uint4 *)src, (uint4 *)dst, bytes, flags, mark);
}

void sph_launch_pack_coords(hipStream_t st, unsigned slots, const sph_dev_params *P,
                            const int *BS, const float2 *POS, const int *ID, short *out)
{
    launch(k_pack_coords, GRID(slots), kTPB, st, P, BS, POS, ID, out);
}

void sph_launch_neighbor_lists(hipStream_t st, unsigned slots, const sph_dev_params *P,
                               const int *BS, const float2 *POS, const unsigned *K, const int *ID,
                               const unsigned *start, int stride, int *full_by_id,
                               int *half_by_id, int *ids_by_id)
{
    launch(k_neighbor_lists, GRID(slots), kTPB, st, P, BS, POS, K, ID, start, stride, full_by_id,
                                                   half_by_id, ids_by_id);
}

void sph_launch_pos_of_id(hipStream_t st, unsigned slots, const sph_dev_params *P, const int *BS,
                          const int *ID, int *pos_of_id)
{
    launch(k_pos_of_id, GRID(slots), kTPB, st, P, BS, ID, pos_of_id);
}

void sph_launch_permute_by_id(hipStream_t st, unsigned slots, const sph_dev_params *P,
                              const int *BS, const int *id_src, const int *pos_of_id,
                              sph_reorder_fields<2> f)
{
    launch(k_permute_by_id, GRID(slots), kTPB, st, P, BS, id_src, pos_of_id, f);
}

void sph_launch_restore(hipStream_t st, unsigned slots, const sph_dev_params *P, const int *BS,
                        const int *flags, sph_restore_args a)
{
    launch(k_restore, dim3(slots / kTPB), kTPB, st, P, BS, flags, a);
}

void sph_launch_copy(hipStream_t st, const sph_copy_set &c)
{
    unsigned g = 0;
    for (int i = 0; i < c.count; i++)
        g += copy_groups(c.n16[i]);
    launch(k_copy, dim3(g ? g : 1), kTPB, st, c);
}

void sph_launch_gather_state(hipStream_t st, unsigned slots, const sph_dev_params *P,
                             const int *BS, const float2 *POS, const float2 *VEL, const int *ID,
                             float4 *out)
{
    launch(k_gather_state, GRID(slots), kTPB, st, P, BS, POS, VEL, ID, out);
}

void sph_launch_gather_aos(hipStream_t st, unsigned slots, const sph_dev_params *P, const int *BS,
                           const float2 *POS, const float2 *VEL, const int *ID0,
                           const float2 *PREV, const float2 *RHO, const int *IDA,
                           const float2 *ACC, float *out)
{
    launch(k_gather_aos, GRID(slots), kTPB, st, P, BS, POS, VEL, ID0, PREV, RHO, IDA, ACC, out);
}

void sph_launch_gather_xy(hipStream_t st, unsigned slots, const sph_dev_params *P, const int *BS,
                          const float2 *POS, const int *ID, float2 *out)
{
    launch(k_gather_xy, GRID(slots), kTPB, st, P, BS, POS, ID, out);
}

void sph_launch_load_state(hipStream_t st, unsigned slots, const sph_dev_params *P, const int *BS,
                           const float4 *in, float2 *POS, float2 *VEL, float2 *PREV, float2 *RHO,
                           int *ID)
{
    launch(k_load_state, GRID(slots), kTPB, st, P, BS, in, POS, VEL, PREV, RHO, ID);
}
