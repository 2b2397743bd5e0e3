// sph_kernels.h - launchers of the gfx950 kernels (sph_kernels.hip).
#pragma once

#include "sph_device.h"

// Source/destination pairs of interleaved (float2) fields for one reorder
// or permutation pass.
template <int NF>
struct sph_reorder_fields {
    const float2 *src[NF];
    float2 *dst[NF];
};

// The tile plans of the current sort: of 256 sorted particles each, and of 64
// (the four-lane gathers' tiles; null unless the context uses those).
struct sph_tile_plans {
    sph_tile_plan *t256 = nullptr, *t64 = nullptr;
    // The crowded ones among the tiles of 256, which four lanes per particle
    // walk (null: no list): *crowded_n of them, the first crowded_max listed.
    unsigned *crowded = nullptr, *crowded_n = nullptr, crowded_max = 0;
};

// The per-cell member lists of a small context's sort (sph_launch_sort_small):
// row `cell` of kBucketRow ints holds the ids of the particles that claimed
// its first kBucketRow slots.  rows null: no lists; ids: the producing
// kernel's particles' ids.
constexpr unsigned kBucketRow = 128;
struct sph_buckets {
    int *rows = nullptr;
    const int *ids = nullptr;
};

// Workgroup size of every particle kernel; scenes are padded to multiples.
constexpr unsigned kSphTPB = 256;

// Lanes per particle (1, 4 or 16) of the gathers of a context with `slots`
// padded slots, on the current device.
int sph_gather_lanes(unsigned slots);
// Whether a context with these lanes lists its crowded tiles.
bool sph_lists_crowded(unsigned slots, int lanes);

// cap: the reference's bucket cap is on (sph_dev_params::bucket_cap != 0).
// lanes: lanes per particle of the gathers, 1, 4 or 16 (sph_gather_lanes);
// more than one applies to the fused step's variants (grav, visc and pred; fused relax).
void sph_launch_visc_predict(hipStream_t st, unsigned slots, bool grav, bool visc, bool pred,
                             bool cap, const sph_dev_params *P, const int *BS,
                             const sph_tile_plans &plans, const float2 *POS, const float2 *VEL,
                             const unsigned *K, const unsigned *start, float2 *opos,
                             unsigned *okey, unsigned *oslot, unsigned *cnt,
                             sph_dev_counters *C, const unsigned long long *clock,
                             float2 *held_vel, int lanes, const sph_buckets &lists);
void sph_launch_gravity(hipStream_t st, unsigned slots, const sph_dev_params *P, const int *BS,
                        float2 *VEL, float2 *RHO);
void sph_launch_predict(hipStream_t st, unsigned slots, const sph_dev_params *P, const int *BS,
                        float2 *POS, const float2 *VEL, float2 *PREV);
void sph_launch_update_velocities(hipStream_t st, unsigned slots, const sph_dev_params *P,
                                  const int *BS, float2 *POS, float2 *VEL, const float2 *PREV);
void sph_launch_key_hist(hipStream_t st, unsigned slots, const sph_dev_params *P, const int *BS,
                         const float2 *POS, unsigned *okey, unsigned *oslot, unsigned *cnt,
                         sph_dev_counters *C);
// The scan over m counts reads and writes whole tiles: cnt and start must hold
// sph_scan_padded(m) entries (16-byte aligned), cnt's beyond m zero.
unsigned sph_scan_blocks(unsigned m);
size_t sph_scan_padded(unsigned m);
void sph_launch_scan_reduce(hipStream_t st, const unsigned *cnt, unsigned m, unsigned *bsum);
// Small count arrays (sph_scan_single_fits(m)): the same scan in one launch.
bool sph_scan_single_fits(unsigned m);
void sph_launch_scan_single(hipStream_t st, unsigned *cnt, unsigned m, unsigned *start);
void sph_launch_scan_apply(hipStream_t st, unsigned *cnt, unsigned m, const unsigned *bsum,
                           unsigned *start);
void sph_launch_scatter(hipStream_t st, unsigned slots, const sph_dev_params *P, const int *BS,
                        const unsigned *key, const unsigned *slot, const unsigned *start,
                        const int *id_src, int *perm_src, int *perm_id, unsigned *key_dst,
                        const sph_tile_plans &plans);
// skey: the sorted keys the scatter wrote (its key_dst)
void sph_launch_reorder2(hipStream_t st, unsigned slots, const sph_dev_params *P, const int *BS,
                         const unsigned *start, const int *perm_src, const int *perm_id,
                         const unsigned *skey, sph_reorder_fields<2> f, int *id_dst,
                         const sph_tile_plans &plans, sph_dev_counters *C);
void sph_launch_reorder4(hipStream_t st, unsigned slots, const sph_dev_params *P, const int *BS,
                         const unsigned *start, const int *perm_src, const int *perm_id,
                         const unsigned *skey, sph_reorder_fields<4> f, int *id_dst,
                         const sph_tile_plans &plans, sph_dev_counters *C);
// The whole sort of a small context (sph_sort_small_fits), whose producing
// kernel left its members' ids in `lists`: starts, sorted keys, ids and fields
// in one launch, and cnt_next cleared.
bool sph_sort_small_fits(unsigned m, int lanes);
void sph_launch_sort_small(hipStream_t st, unsigned slots, const sph_dev_params *P, const int *BS,
                           const unsigned *key, const unsigned *cnt, unsigned *cnt_next,
                           unsigned m, unsigned *start, const sph_buckets &lists,
                           sph_reorder_fields<2> f, int *id_dst, unsigned *key_dst,
                           sph_dev_counters *C);
// The tile plans alone, of sorted keys that no reorder has just placed.
void sph_launch_plan(hipStream_t st, unsigned slots, const sph_dev_params *P, const int *BS,
                     const unsigned *start, const unsigned *skey, const sph_tile_plans &plans);
// Copy src to pinned host memory, and set the flag of every kHostPiece bytes to
// `mark` once they are there.
constexpr size_t kHostPiece = 32u << 10;
void sph_launch_to_host(hipStream_t st, const void *src, void *dst, size_t bytes,
                        unsigned *flags, unsigned mark);
void sph_launch_density(hipStream_t st, unsigned slots, bool cap, const sph_dev_params *P,
                        const int *BS, const sph_tile_plans &plans, const float2 *POS,
                        const unsigned *K, const unsigned *start, float2 *RHO, uint4 *masks,
                        sph_dev_counters *C, int lanes);
void sph_launch_relax(hipStream_t st, unsigned slots, bool fused, bool cap,
                      const sph_dev_params *P, const int *BS, const sph_tile_plans &plans,
                      const float2 *POS, const float2 *PREV, const float2 *RHO, const unsigned *K,
                      const unsigned *start, float2 *opos, float2 *ovel, unsigned *okey,
                      unsigned *oslot, unsigned *cnt, const uint4 *masks, sph_dev_counters *C,
                      unsigned long long *clock, int lanes, const sph_buckets &lists);
void sph_launch_pack_coords(hipStream_t st, unsigned slots, const sph_dev_params *P,
                            const int *BS, const float2 *POS, const int *ID, short *out);
void sph_launch_neighbor_lists(hipStream_t st, unsigned slots, const sph_dev_params *P,
                               const int *BS, const float2 *POS, const unsigned *K, const int *ID,
                               const unsigned *start, int stride, int *full_by_id,
                               int *half_by_id, int *ids_by_id);
void sph_launch_pos_of_id(hipStream_t st, unsigned slots, const sph_dev_params *P, const int *BS,
                          const int *ID, int *pos_of_id);
void sph_launch_permute_by_id(hipStream_t st, unsigned slots, const sph_dev_params *P,
                              const int *BS, const int *id_src, const int *pos_of_id,
                              sph_reorder_fields<2> f);

// Per-scene copy of a state snapshot back into the live arrays: the slot
// range of every scene whose flag is set, and its cell starts (incl. the
// scene's padding cell).  F[0..3] = POS, VEL, PREV, RHO.
struct sph_restore_args {
    const float2 *src[4];
    float2 *dst[4];
    const int *id_src;
    int *id_dst;
    const unsigned *key_src, *start_src;
    unsigned *key_dst, *start_dst;
};
void sph_launch_restore(hipStream_t st, unsigned slots, const sph_dev_params *P, const int *BS,
                        const int *flags, sph_restore_args a);

// Device-to-device copies of several arrays in one launch: n16[i] 16-byte
// units each, sources and destinations 16-byte aligned; and one 64-bit word
// (word_src null: none).
constexpr int kCopyArrays = 8;
struct sph_copy_set {
    const void *src[kCopyArrays];
    void *dst[kCopyArrays];
    unsigned n16[kCopyArrays];
    int count = 0;
    const unsigned long long *word_src = nullptr;
    unsigned long long *word_dst = nullptr;
    void add(void *d, const void *s, size_t bytes) // bytes: rounded up to 16
    {
        src[count] = s;
        dst[count] = d;
        n16[count++] = (unsigned)((bytes + 15) / 16);
    }
};
void sph_launch_copy(hipStream_t st, const sph_copy_set &c);

// Caller-order state exchange with device buffers of float4 (x, y, v_x, v_y)
// per particle at uoff + id.  Load sets ids to the slot order (id = slot -
// poff), PREV = POS and RHO = 0.
void sph_launch_gather_state(hipStream_t st, unsigned slots, const sph_dev_params *P,
                             const int *BS, const float2 *POS, const float2 *VEL, const int *ID,
                             float4 *out);
void sph_launch_load_state(hipStream_t st, unsigned slots, const sph_dev_params *P, const int *BS,
                           const float4 *in, float2 *POS, float2 *VEL, float2 *PREV, float2 *RHO,
                           int *ID);
// fluid_particle records (13 words) by caller index uoff + id; IDA orders
// PREV and RHO, ACC holds (a_x, a_y) by caller index.
void sph_launch_gather_aos(hipStream_t st, unsigned slots, const sph_dev_params *P, const int *BS,
                           const float2 *POS, const float2 *VEL, const int *ID0,
                           const float2 *PREV, const float2 *RHO, const int *IDA,
                           const float2 *ACC, float *out);
// Positions (x, y) by caller index uoff + id.
void sph_launch_gather_xy(hipStream_t st, unsigned slots, const sph_dev_params *P, const int *BS,
                          const float2 *POS, const int *ID, float2 *out);

// Time the next kernel launch of this thread with a start/stop event pair
// (recorded by the launch itself: the kernel's own duration).
void sph_set_next_launch_events(hipEvent_t start, hipEvent_t stop);

// Exhaustive bit-for-bit check of sph_sqrt against sqrtf over float bit
// patterns [lo, hi).
void sph_launch_selftest_math(hipStream_t st, int fn, unsigned lo, unsigned hi,
                              unsigned long long *bad);
