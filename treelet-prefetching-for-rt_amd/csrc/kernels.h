// kernels.h — launch parameters shared by the host runtime and the kernels.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "rtx.h"

namespace rtxk {

// Error bits raised by kernels (mapped to rtx_status on the host).
enum : uint32_t {
  kErrStack = 1u,      // per-lane traversal stack overflow
  kErrType = 2u,       // malformed node type
  kErrRange = 4u,      // node outside the arena
  kErrRecords = 8u,    // record buffer overflow
  kErrInstSlot = 16u,  // treelet order: an instance leaf 128 MiB or more away from the TLAS header
  kErrSteps = 32u,     // per-ray step limit (cyclic or corrupt BVH)
  kErrBudget = 64u,    // treelet node larger than the budget
  kErrQueue = 128u     // partitioner work buffer overflow
};

// Record output of a trace kernel.
enum : int {
  kRecNone = 0,  // hits only
  kRecCsr = 1,   // records at record_offsets[ray]
  kRecSlab = 2,   // a ray's first record_slab records as slab entries
  kRecSlab4 = 3   // the same in 4-byte entries
};

constexpr uint32_t kBlock = 256;        // threads per block (4 waves of 64)
constexpr uint32_t kSlotWords = 64;     // control slot: [0] ray counter, [1] error, [2] overflow count, stats (u64) from word 16
constexpr uint32_t kMaxStepsPerRay = 1u << 24;
constexpr uint32_t kMaxBatchJobs = 1024;

// One entry of a multi-scene batch: a ray range of one scene (64 bytes).
struct alignas(64) BatchJob {
  const uint8_t* arena;
  uint64_t arena_bytes;
  uint64_t tlas;
  const rtx_ray* rays;
  rtx_hit* hits;
  const uint32_t* owner;
  uint32_t first_treelet;
  uint32_t n;
  uint32_t ray_base;  // rays of all earlier jobs
  uint32_t pad[3];
};

struct TraceParams {
  const uint8_t* arena;
  uint64_t arena_bytes;
  uint64_t tlas;
  const rtx_ray* rays;
  uint32_t n;
  uint32_t refill;  // refill the wave when at least this many lanes are idle
  rtx_hit* hits;
  rtx_record* records;
  uint64_t record_capacity;
  const uint64_t* record_offsets;
  // slab records: ray r's first record_slab records as slab entries of 8 bytes (4
  // with kRecSlab4), at slab_place() of the two arrays (`records` unused)
  uint64_t* slabs;
  uint64_t* slabs_rest;
  uint32_t record_slab;
  uint32_t rec_level_shift;  // kRecSlab4: the entries' slot bits
  uint32_t* rec_counts;    // slab records: ray r's record count at rec_counts[r]
  // level pass: per lane a tree_level_map of lm_cap u64 entries (zero between
  // rays) at lm_table + lane * lm_cap, and lm_cap / 2 positions at lm_list
  uint64_t* lm_table;
  uint32_t* lm_list;
  uint32_t lm_cap;
  const uint64_t* layout_remap;  // nullable: records carry these layout offsets (arena slot -> offset)
  uint32_t claim_start;    // rays are claimed from this index on, wrapping to 0
  const uint32_t* ray_list;  // nullable: claim k traces ray ray_list[k] (n = list length)
  uint32_t n_rays;           // rays in the ray / hit arrays (ray_list entries must lie below)
  const uint32_t* owner;  // node slot -> dense treelet index (nullable in plain mode)
  uint32_t first_treelet; // dense index of the treelet rooted at the TLAS header
  uint64_t* spill;        // global stack spill, spill_cap entries per stack per lane
  uint32_t spill_cap;
  uint32_t* ray_counter;
  uint32_t* error;
  unsigned long long* stats;  // rtx_prefetch_stats counters
  // a mapped host word set to 1 when any ray reports an error
  uint32_t* host_err;
  // treelet staging
  uint32_t prefetch;                 // RTX_PREFETCH_*
  float threshold;
  const uint32_t* image_slots;       // node slot held by each 64-byte unit of `images`
  const uint64_t* image_offset;      // dense treelet -> byte offset of its image in `images`
  const uint32_t* image_bytes;       // dense treelet -> image size
  const uint8_t* images;             // treelet-contiguous copies of the arena
  uint32_t slot_units;               // staging slot size in 64-byte units (0: one slot)
  float min_score;                   // learned policy: summed lane probability to stage a prediction
  float pred_fraction;               // learned policy: share of a predicted image staged (root first)
  const uint4* pred_table;           // learned policy: [pred_treelets * 8] rows of 4 packed predictions
  uint32_t pred_treelets;
  // multi-scene batch (batch kernels only): rays are numbered across jobs
  const BatchJob* jobs;
  uint32_t n_jobs;
  // every child box of the scene(s) has lower bound bytes <= upper ones, and no
  // node a NaN origin or a scale above 2^103, so a finite ray may pick each
  // axis's near and far bound by its direction sign
  uint32_t ordered_boxes;
  // every node of the scene(s) has its children packed from slot 0 on, an
  // instance leaf in two slots and any other child in one, all in the arena
  uint32_t regular_nodes;
};

// Most treelets resident at once in a wave's staging area.
constexpr uint32_t kMaxStageSlots = 16;

// Device scratch of rtx_trace_static (static_scratch.hip): 256 bytes of
// control words, then the per-lane global stack spill.
constexpr size_t kStaticScratchBytes = 128ull << 20;
constexpr size_t kStaticControlBytes = 256;
constexpr uint32_t kStaticMinSpill = 24;  // spill entries per lane and list it keeps at least
// Address of the calling thread's current device's copy of the scratch array
// (looked up once per device; `device` must be current).
hipError_t static_scratch_init(int device, void** out);

// Launchers (defined in the .hip files).
uint32_t trace_block_size(uint32_t stage_bytes);
hipError_t launch_trace(const TraceParams& p, uint32_t mode, int records, uint32_t lds_stack, uint32_t stage_bytes,
                        uint32_t grid, hipStream_t s);
hipError_t launch_trace_batch(const TraceParams& p, uint32_t mode, uint32_t lds_stack, uint32_t grid,
                              hipStream_t s);
// Workgroups of a trace kernel that fit on one CU at once (registers and LDS);
// 0 when the configuration has no kernel.
uint32_t trace_blocks_per_cu(uint32_t mode, int records, uint32_t lds_stack, uint32_t stage_bytes);
uint32_t trace_batch_blocks_per_cu(uint32_t mode, uint32_t lds_stack);
// Cooperative kernel for small batches (eight lanes per ray, no staging), plain or
// treelet order, with slab records or hits only: `cap` entries per list and ray
// (at most 144), 256-lane blocks, `groups` rays at a time in a wave (at most 8).
constexpr uint32_t kWideRayLanes = 8;
hipError_t launch_trace_wide(const TraceParams& p, uint32_t mode, bool records, uint32_t cap, uint32_t grid,
                             uint32_t groups, hipStream_t s);
uint32_t trace_wide_blocks_per_cu(uint32_t mode, bool records, uint32_t groups);
// Batches that take that kernel by default, in rays per CU: a batch that leaves most
// of the GPU idle is bound by the step latency of its longest rays, and a group
// tests a node's six children at once.  Up to the lines every ray has a group of
// its own, so waves claim without a counter (16,384 rays of the 1M-triangle scene
// in plain order 149 -> 116 us); treelet order's two stacks let only half as many
// be resident, and records make the second round cost more.  Eight lanes per ray
// against one, camera rays of the 16,384-triangle sphere / the 1M-triangle scene, us:
//   plain            32,768 rays 220 : 278 / 120 : 154, 40,960 rays 266 : 259 / 203 : 162
//   plain, records   32,768 rays 326 : 345 / 183 : 204, 40,960 rays 362 : 328 / 267 : 216
//   treelet          32,768 rays 235 : 253 / 212 : 217, 40,960 rays 189 : 186 / 226 : 217
//   treelet, records 16,384 rays 260 : 293 / 214 : 251, 24,576 rays 238 : 227 / 277 : 270
inline uint32_t wide_rays_per_cu(uint32_t mode, bool records) {
  return mode == RTX_MODE_TREELET && records ? 64u : 128u;
}
// Rays at a time in a wave of that kernel: the fewest with which all are resident
// (16 waves on a CU), since the rays of a wave wait for each other's passes.  Camera
// rays of the 16,384-triangle sphere in plain order, one / two / four / eight a wave, us:
//    4,096 rays 152 / 188 / 198 / 213,  8,192 rays 235 / 178 / 208 / 230,
//   16,384 rays 345 / 273 / 210 / 223
inline uint32_t wide_groups(uint64_t n, uint32_t n_cus) {
  uint32_t groups = 1;
  while (groups < 8 && n > 16ull * n_cus * groups) groups *= 2;
  return groups;
}
// The level pass over p.n rays (p.ray_list / claim order as in launch_trace):
// each hit's max_level becomes the maximum of the reference's final
// tree_level_map.  p.lm_table must hold grid * 256 zeroed maps of p.lm_cap
// (a power of two) entries.
hipError_t launch_level_pass(const TraceParams& p, uint32_t mode, uint32_t grid, hipStream_t s);
// Bytes of level-pass memory per lane: the map and its position list.
constexpr uint64_t level_pass_lane_bytes(uint32_t lm_cap) { return (uint64_t)lm_cap * 8 + (uint64_t)lm_cap / 2 * 4; }
constexpr uint32_t kLevelMapCap = 4096;  // map entries per lane: at most 2,048 nodes assigned per ray
// Clears `words` 32-bit words with a kernel (usable inside graph capture).
hipError_t launch_fill_zero(uint32_t* dst, uint32_t words, hipStream_t s);
// host[2..3] = *total (host: mapped host memory), so that the caller reads it
// after a stream synchronisation without a copy.
hipError_t launch_report_total(const uint64_t* total, uint32_t* host, hipStream_t s);
// CSR offsets[0..n] of the rays' record counts (hits[i].n_records).
hipError_t launch_scan_records(const rtx_hit* hits, uint32_t n, uint64_t* offsets, uint64_t* block_tmp, hipStream_t s);
// Statistics of a traced batch: acc[0..6] records per type, [7] hits, [8] any
// hits, [9] nodes, [10] max nodes, [11] max level, [12] fetch bytes, [13]
// accessed bytes (acc must start at 0; records may be null).
hipError_t launch_trace_stats(const rtx_hit* hits, uint32_t n, const rtx_record* records, uint64_t n_records,
                              unsigned long long* acc, hipStream_t s);
// The coherence engine's claim order of n rays (coherence.hip), queued on s.
// `scratch` holds coherence_scratch_bytes(n) bytes, 4-byte aligned.
size_t coherence_scratch_bytes(uint32_t n);
hipError_t coherence_order(const rtx_ray* rays, uint32_t n, const rtx_coherence_config& cfg, const float wmin[3],
                           const float wmax[3], uint32_t* order, uint32_t* hashes_out, void* scratch, hipStream_t s);
// Slab records: each lane holds its last 64 bytes of entries in LDS and writes
// them to the slab in aligned groups of 32 bytes (four entries, eight of four
// bytes), so slab rows are padded to a multiple of eight entries.
__host__ __device__ inline uint32_t slab_stride(uint32_t record_slab) { return (record_slab + 7u) & ~7u; }
// A row's first entries lie in one array and the rest in another, so that the
// entries of most rays (21 of them on average in the 1M-triangle diffuse batch)
// are dense in memory: rows of 512 entries would spread 110 MB of them over 2.7 GB.
constexpr uint32_t kSlabFront = 32;
__host__ __device__ inline uint32_t slab_front(uint32_t record_slab) {
  const uint32_t stride = slab_stride(record_slab);
  return stride < kSlabFront ? stride : kSlabFront;
}
// entry k of ray r's row, k a multiple of 4 (k < slab_stride)
template <typename E>
__host__ __device__ inline E* slab_place(uint64_t* slabs, uint64_t* rest, uint32_t record_slab, uint64_t r, uint32_t k) {
  const uint32_t front = slab_front(record_slab);
  return k < front ? reinterpret_cast<E*>(slabs) + r * front + k
                   : reinterpret_cast<E*>(rest) + r * (slab_stride(record_slab) - front) + (k - front);
}
// A slab entry: the node's arena slot (offset / 64) in the low word, the
// record type and level in the high word.  The size follows from the type;
// the treelet and the layout offset are looked up when the entry is expanded.
__host__ __device__ inline uint64_t slab_entry(uint32_t slot, uint32_t type, uint32_t level) {
  return (uint64_t)slot | ((uint64_t)(type | ((level > 255u ? 255u : level) << 8)) << 32);
}
// The 4-byte form: the slot in the low `shift` bits, the level above them, the
// type in the top three.  For scenes whose slots and levels fit 29 bits together
// (every node at one tree level, so the level is known beforehand to be at most
// the scene walk's).
constexpr uint32_t kSlab4TypeShift = 29;
__host__ __device__ inline uint32_t slab_entry4(uint32_t slot, uint32_t type, uint32_t level, uint32_t shift) {
  return slot | (level << shift) | (type << kSlab4TypeShift);
}
// The records of n rays out of their slabs: offsets[0..n] of the counts, each row's
// first `slab` entries as rtx_records at its offset (owner and layout_remap
// nullable, as in TraceParams), rays with more than `slab` records appended to
// overflow_list as ray_base + their index (count in overflow_count, which must
// start at 0 with a batch's first range).  With add_base the offsets go on from
// offsets[0], and the list and its count from the batch's earlier ranges.  No
// record is written when the total exceeds `capacity`.  host (nullable, mapped host
// memory): host[0] = the batch's overflowed rays so far, host[2..3] = offsets[n].
struct FinishParams {
  const uint32_t* counts;
  uint32_t n;
  uint32_t slab;
  uint64_t* slabs;
  uint64_t* slabs_rest;
  uint32_t shift;  // the 4-byte entries' rec_level_shift, 0 for 8-byte entries
  uint32_t add_base;
  const uint32_t* owner;
  const uint64_t* layout_remap;
  uint64_t slots;  // of the arena (owner and layout_remap entries)
  uint64_t* offsets;
  rtx_record* records;
  uint64_t capacity;
  uint32_t ray_base;
  uint32_t n_tiles;
  uint32_t* overflow_list;
  uint32_t* overflow_count;
  uint32_t* host;
  const uint64_t* tile_sums;  // set by launch_finish_records
};
// Batches of at most this many rays sum their counts in every workgroup (32 KiB
// of counts from L2) instead of in a launch of its own.
constexpr uint32_t kFinishAlone = 8192;
// Larger ones: up to this many tiles of 1,024 rays each workgroup sums them all, which
// costs the square of their number; more (ranges of short rows have up to 262,144) are
// scanned in a launch of their own.  1,024 / 4,096 / 8,192 / 32,768 tiles, us: summed
// 8.5 / 26 / 62 / 589, scanned 11 / 30 / 54 / 198.
constexpr uint32_t kTilesSummed = 4096;
// tile_sums: a word for each 1,024 rays begun, and one more
hipError_t launch_finish_records(FinishParams p, uint64_t* tile_sums, hipStream_t s);

}  // namespace rtxk
