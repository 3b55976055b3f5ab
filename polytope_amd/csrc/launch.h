// Host-side declarations of the kernel launchers (defined in the .hip files).
#pragma once

#include <hip/hip_runtime_api.h>
#include <hip/hip_vector_types.h>

#include <algorithm>

#include "ptx_internal.h"

namespace ptx {
// Blocks per CU that a launch of few ids is spread over (deal_ids): 1 / 2 / 4
// took 119 / 107 / 115 us for 50,021 rays on 81,920 faces, 342 / 300 / 330 us
// for a 64x48 thumbnail of 4 samples (82 to 130 and 407 us packed).
constexpr uint32_t kSpreadBlocks = 2;
constexpr uint32_t kDealBatch = 64;
}  // namespace ptx

namespace ptx {

// Grid and batches of a persistent launch over n ids: `full` blocks
// (what fits the device) and batches of 64, three quarters of them dealt out
// statically, when the ids fill it; else every wave gets one batch of its
// share, from as many blocks as hold the ids at one a lane, or as two waves
// per SIMD while that leaves a wave at least one id.  A wave of few rays runs
// fewer phases for lanes other than its own.
inline uint32_t deal_ids(uint32_t full, uint32_t num_cus, uint64_t n, Deal &d) {
   const uint64_t packed = (n + 255) / 256, spread = std::min<uint64_t>((n + 3) / 4, kSpreadBlocks * (uint64_t)num_cus);
   const uint32_t grid = (uint32_t)std::max<uint64_t>(1, std::min<uint64_t>(full, std::max(packed, spread)));
   d.n = (uint32_t)n;
   d.batch = (uint32_t)std::min<uint64_t>(kDealBatch, std::max<uint64_t>(1, (n + 4ull * grid - 1) / (4ull * grid)));
   d.batches = (uint32_t)((n + d.batch - 1) / d.batch);
   d.static_batches = d.batches <= 4 * grid ? d.batches : d.batches - d.batches / 4;
   return grid;
}

// Whether a launch hands out batches by its counter, which must then start at
// zero: where every batch is dealt out no kernel has to clear it first (5 us of
// the smallest query's 53, 10 of the smallest batch's 300).
inline bool counted(const Deal &d) { return d.static_batches < d.batches; }

// windows: the scene's window records (launch_build_windows), or null to step
// over sc.nodes; root_axis: the root's split axis (used with windows).
int launch_closest_hit(const DevScene &sc, const float *d_rays, const Deal &deal, ptx_hit *d_hits,
                       ptx_ray_counters *d_counters, ptx_hit_frame *d_frames, uint32_t *d_work, uint4 *d_spill,
                       uint32_t grid, uint32_t lds_depth, uint32_t refill_min, uint32_t leaf_min,
                       const Node64 *windows, uint32_t root_axis, hipStream_t stream);
// The same over the scene's four-wide form w (w.faces non-null), hits and
// frames; d_spill: (w.stack - lds_depth) 8-byte entries per resident lane.
int launch_closest_hit_wide(const DevScene &sc, const WideScene &w, const float *d_rays, const Deal &deal, ptx_hit *d_hits,
                            ptx_hit_frame *d_frames, uint32_t *d_work, void *d_spill, uint32_t grid,
                            uint32_t lds_depth, uint32_t refill_min, uint32_t leaf_min, hipStream_t stream);
int closest_hit_wide_blocks_per_cu(uint32_t lds_depth, bool frames);
// Resident blocks per CU of the closest-hit kernel; extra = counters or frames
// requested, windows = the form that steps over window records.
int closest_hit_blocks_per_cu(uint32_t lds_depth, bool extra, bool windows);
// Window records of the closest-hit kernel: win (4 * n_int Node64, 128-byte
// aligned) from the scene's n_int interior records.
int launch_build_windows(const Node64 *nodes, uint32_t n_int, Node64 *win, hipStream_t stream);

// Face records of the four-wide form from the scene's np leaf-ordered triangles
// and ids and their flat words (or null for none).
int launch_build_wide_faces(const float *tris, const uint32_t *pairs, const uint8_t *flat, uint32_t np, WideFace *out,
                            hipStream_t stream);

// Size of the per-device static scratch of the no-allocation closest-hit entry
// point: 256 bytes of work counters, then the deferred-stack spill.
constexpr size_t kNoAllocScratchBytes = size_t(64) << 20;
// Device address of that scratch on device `ordinal`, which must be current.
// Looked up once per device (hipGetSymbolAddress); 0 on success.
int noalloc_scratch_address(int ordinal, void **ptr);

}  // namespace ptx

namespace ptx {

uint32_t render_lds_depth();
// 0 extend, 1 primary, 2 plain megakernel, 3 plain with next-event estimation, 4 shadow connection;
// over the four-wide form 5 primary, 6 plain, 7 plain with next-event estimation
int render_blocks_per_cu(int which);
// W / wides: the scenes' four-wide forms, which the kernel then steps over
// (every scene of the launch has one whose stack fits the spill); null = the
// binary records.
// deal: of the four-wide kernels (deal_ids).
void launch_primary(const DevScene &S, const WideScene *W, const JobDev &J, const Deal &deal, uint32_t *work,
                    uint4 *spill, uint32_t leaf_min, uint32_t grid, hipStream_t st);
// Primary records of every job of a batch in one launch: jobs / scenes are the
// device tables, offsets (njobs + 1 entries, device) the first pixel id of
// each job and the total; max_stack bounds every scene's deferred stack.
void launch_primaries(const JobDev *jobs, const DevScene *scenes, const WideScene *wides, const uint32_t *offsets,
                      uint32_t njobs, const Deal &deal, uint32_t *work, uint4 *spill, uint32_t leaf_min, uint32_t max_stack, uint32_t grid,
                      hipStream_t st);
// Shadow connection of the wavefront form (rounds with next-event jobs):
// the vertex queue (48 B per entry, one entry per path slot at most), its
// count, the per-slot next-event sums (3 floats) and the connect grid.  q null:
// no next-event job in the round.
struct ShadowArgs {
   float4 *q = nullptr;
   uint32_t *count = nullptr;
   float *direct = nullptr;
   uint32_t grid = 0;
};
void launch_round_start(const Chunk *chunks, uint32_t nchunks, uint32_t nslots, const JobDev *jobs,
                        const DevScene *scenes, float *res, float *q_out, uint32_t *count_out, uint32_t *bounce,
                        const ShadowArgs &sh, uint4 *spill, uint32_t max_stack, uint32_t grid, hipStream_t st);
void launch_bounce(const float *q_in, const uint32_t *count_in, float *q_out, uint32_t *count_out, float *hits,
                   const JobDev *jobs, const DevScene *scenes, float *res, uint32_t *work, uint4 *spill,
                   uint32_t max_stack, uint32_t leaf_min, uint32_t *bounce, const ShadowArgs &sh, uint32_t ext_grid,
                   uint32_t shade_grid, hipStream_t st);
// direct: the per-slot next-event sums of a wavefront round, added to the
// samples of next-event jobs; null for path-regeneration rounds.
void launch_accumulate(const Chunk *chunks, uint32_t nchunks, const JobDev *jobs, const float *res,
                       const float *direct, uint32_t grid, hipStream_t st);
void launch_finalize(float *film, uint32_t npix, uint32_t spp, hipStream_t st);
void launch_zero_floats(float *a, size_t n, hipStream_t st);
// dst[i] = src[i], n words, 16-byte aligned; src may be pinned host memory.
void launch_copy_words(uint32_t *dst, const uint32_t *src, size_t n, hipStream_t st);
int paths_blocks_per_cu();
// Path-regeneration mode: one launch per round; rounds limited to
// paths_max_chunks() chunks and paths_max_scenes() scenes.  nee_scratch (48
// bytes per resident lane, grid * 256 lanes) selects the kernel variant with
// next-event estimation for the jobs that ask for it; null = without.
uint32_t paths_max_chunks();
uint32_t paths_max_scenes();
void launch_paths(const Chunk *chunks, uint32_t nchunks, uint32_t nslots, const JobDev *jobs, const DevScene *scenes,
                  const WideScene *wides, uint32_t nscenes, float *res, const Deal &deal, uint32_t *work, uint4 *spill,
                  uint32_t max_stack, uint32_t shade_min, uint32_t leaf_min, float4 *nee_scratch, bool glossy,
                  bool textured, uint32_t grid, hipStream_t st);
// textured: the scene has textured meshes; cached: start every path from the
// pixel's primary record in J.primary (written by launch_primary).
void launch_mega(const DevScene &S, const WideScene *W, const JobDev &J, uint32_t sample, uint4 *spill, bool textured,
                 bool cached, uint32_t grid, hipStream_t st);

}  // namespace ptx
