// traverse.hip — per-ray BVH traversal kernels for gfx950.
//
// One ray per lane.  Waves are persistent: whenever at least `refill` lanes of
// a wave are idle, the wave takes that many ray indices from a global counter
// with one atomic, so uneven ray costs do not leave lanes idle.
//
// Both traversal orders of the reference are flattened into "pop one entry,
// process it" steps:
//  * PLAIN (traceRay, vulkan_ray_tracing.cc:2309-3076): the nested top/bottom
//    loops visit the first hit internal child immediately and push the other
//    hit children in slot order; that is the same sequence as pushing all hit
//    children in slot order with the first internal child pushed last.  Only
//    one instance is open at a time, so the instance context lives in
//    registers.  A node's hit children are pushed as one group (see Groups).
//  * TREELET (traceRayWithTreelets, :1522-2307): two LIFO lists.  A child goes
//    to the "current" list while the current treelet is still the one rooted
//    at the TLAS header and the child's owner is that treelet; after the
//    first move from the "other" list the reference compares against a host
//    address (:1752), so every later child goes to "other".  Which children
//    the first treelet owns is precomputed with the partition, one byte per
//    node slot, so a node costs one extra byte load, not one per child.
//    Entries carry the instance leaf that opened them (groups pushed after the
//    switch need none, see Groups); the object-space ray is recomputed from
//    that leaf when it differs from the cached one (same inputs, same floats).
//
// Stacks: a ring of K groups or entries per lane and list in LDS, spilling the
// oldest to a per-lane region in global memory (exact LIFO order).
//
// One wave iteration runs three passes, each only for the lanes that need it:
// instance leaves, triangle leaves, then internal nodes.  A lane that finishes
// a leaf pops its next entry at once and joins the internal-node pass if that
// entry is an internal node; an instance leaf hands over its BLAS root the
// same way when that root is the next entry to be popped.  Completed rays
// keep their state until the wave's next refill, which writes their hit
// records together.
//
// Small batches (wide_rays_per_cu) run trace_wide instead: eight lanes per ray,
// the six child boxes of a node tested at once (see the section before its
// definition).
//
// Treelet staging (STAGE > 0, one wave per workgroup): the wave keeps up to
// stage/slot treelet images in LDS slots, copied from the treelet-contiguous
// image buffer with coalesced 16-byte loads, and an LDS hash table from node
// slot to position in the staging area.  A node read first probes the table;
// hits read LDS, misses read global memory.  When most lanes miss, the wave
// gathers the owning treelet of each lane's next node and stages the most
// popular one into the least recently read slot, following the RT-unit policy
// of src/gpgpu-sim/shader.cc:3419-3559 (heuristic 0 always, 1 only above a
// popularity share, 2 a popularity-sized prefix).  The learned policy then
// also stages the treelets a prediction table names as the lanes' likely next
// ones.  Staging changes where node bytes are read from, never which nodes
// are visited.
#include <algorithm>
#include <type_traits>

#include "device_common.h"
#include "kernels.h"

using namespace rtxd;

namespace rtxk {
namespace {

constexpr uint32_t kFlTop = 1u, kFlLeaf = 2u;
constexpr uint32_t kNoSlot = 0xffffffffu;
constexpr uint32_t kNone = 0xffffffffu;

// An entry: node slot (32 bits), flags (2), tree level (8) and the
// instance leaf that opened the entry (22 bits, treelet order only).  The
// instance is stored as its slot's distance from the TLAS header slot, a
// signed 22-bit value, so instance leaves may lie anywhere within 128 MiB of
// the TLAS header whatever the arena's size.
constexpr int32_t kInstRelMax = 1 << 21;
__device__ __forceinline__ uint64_t make_entry(uint32_t slot, uint32_t flags, uint32_t level, uint32_t inst_rel) {
  uint32_t lv = level > 255u ? 255u : level;
  return (uint64_t)slot | ((uint64_t)(flags | (lv << 2) | ((inst_rel & 0x3fffffu) << 10)) << 32);
}
__device__ __forceinline__ uint32_t e_slot(uint64_t e) { return (uint32_t)e; }
__device__ __forceinline__ uint32_t e_flags(uint64_t e) { return (uint32_t)(e >> 32) & 3u; }
__device__ __forceinline__ uint32_t e_level(uint64_t e) { return ((uint32_t)(e >> 32) >> 2) & 255u; }
__device__ __forceinline__ uint32_t e_inst_rel(uint64_t e) { return (uint32_t)(e >> 42); }
// absolute instance-leaf slot of an entry, given the TLAS header slot
__device__ __forceinline__ uint32_t e_inst(uint64_t e, uint32_t tlas_slot) {
  return tlas_slot + (uint32_t)(((int32_t)(e_inst_rel(e) << 10)) >> 10);
}
// the relative field of instance-leaf slot `inst`, or false when it is out of range
__device__ __forceinline__ bool inst_rel_of(uint32_t inst, uint32_t tlas_slot, uint32_t& rel) {
  const int64_t d = (int64_t)inst - (int64_t)tlas_slot;
  rel = (uint32_t)d & 0x3fffffu;
  return d >= -kInstRelMax && d < kInstRelMax;
}

// LDS and global stack words are reached through pointers typed by address
// space, so a pop compiles to ds_read or global_load and never to a flat load
// (which would also wait for every outstanding store of the lane).
typedef __attribute__((address_space(3))) uint64_t lds_u64;
typedef __attribute__((address_space(1))) uint64_t glb_u64;

// ---- stacks of child groups ------------------------------------------------------
// A node's hit children left for later are one group: the slot of its first
// child and a word with the children still to visit (bits 16-21), which children
// are leaves (10-15), the tree level (2-9) and whether it is a TLAS node (1).
// The children are visited highest slot first, which is the order of popping
// them after pushing each in slot order.  The child visited next goes on as the
// lane's next entry: in plain order the first internal one, which is pushed last
// there, in treelet order the highest.  The newest group stays in registers,
// older ones are a ring of K per lane in LDS whose oldest spill to global memory.
// The depth counts the children outstanding, one each, and the ray reports a
// stack overflow at K + spill_cap of them.
// A group needs a regular node: children packed from slot 0 on, an instance leaf
// two slots and any other child one.  The scene walk checks that once for all
// nodes; other scenes push every child on its own.
// A push of up to six entries, each placed and stored under its own branch, was
// a third of the vector instructions of an internal node; a group takes 45
// instead of 155 and at most one LDS store, and the next child reaches the next
// iteration without LDS.  With the slab test on halves below, 1.34M camera and
// bounce rays on the 1M-triangle scene take 263 -> 228 M vector instructions and
// 594 -> 558 us in plain order; the registers it frees keep five waves there.  In
// treelet order 2.6M rays on the 21M-triangle scene take 2.33 -> 2.21 ms, and the
// diffuse batch with whole treelets staged 1.66 -> 1.44 ms.
//
// Treelet order has two lists.  The register group belongs to the list the next
// pop takes (the current one, and the other one after the switch); before the
// switch the other list is only pushed to.  An entry of a BLAS also names its
// instance, for which a group has no room: after the switch the lists are one
// stack, so whenever a group pushed since comes up, the ray's instance is again
// the one it was pushed in.  Before the switch, children in a BLAS are pushed
// one by one as entries (make_entry), told apart by bit 0 with bits 10 and up.
struct Groups {
  uint32_t base, word;  // the newest group; word < kGroupFirst: none left in it
  // its list: items in the ring and spilled (bits 0-7; position p of them is in
  // LDS unless p < bits 8-15), depth (16-23, at most 144); and the ray's opaque
  // and terminate flags (24, 25)
  uint32_t state;
};
constexpr uint32_t kGroupFirst = 1u << 16, kGroupLeaf = 10, kGroupTag = 1u, kGroupTop = 2u;
constexpr uint32_t kListItems = 0xffu, kListDepth = 1u << 16, kListDepthMask = 0xff0000u;
constexpr uint32_t kRayOpaque = 1u << 24, kRayTerminate = 1u << 25;
__device__ __forceinline__ uint32_t group_word(bool top, uint32_t level, uint32_t leaves, uint32_t mask) {
  return kGroupTag | (top ? kGroupTop : 0u) | ((level > 255u ? 255u : level) << 2) | (leaves << kGroupLeaf) | (mask << 16);
}
__device__ __forceinline__ bool is_group(uint64_t v) {
  const uint32_t w = (uint32_t)(v >> 32);
  return (w & kGroupTag) && (w >> kGroupLeaf);
}

// child i of a group as an entry (make_entry) without its instance
__device__ __forceinline__ uint64_t group_entry(uint32_t base, uint32_t word, uint32_t i) {
  const uint32_t leaves = __builtin_amdgcn_ubfe(word, kGroupLeaf, i);  // the leaves below child i
  const uint32_t two = (uint32_t)__builtin_amdgcn_sbfe((int)word, 1, 1) & leaves;
  const uint32_t leaf = (word >> (kGroupLeaf + i)) & 1u;
  return (uint64_t)(base + i + (uint32_t)__popc(two)) |
         ((uint64_t)((word & 0x3fcu) | __builtin_amdgcn_ubfe(word, 1, 1) | (leaf << 1)) << 32);
}

// One list's ring: `state` as in Groups, R its length, `lds` and spill() the
// lane's words.
template <int R, uint32_t BS, typename Spill>
__device__ __forceinline__ void ring_put(uint32_t& state, uint64_t v, lds_u64* lds, Spill&& spill) {
  const uint32_t cnt = state & kListItems, out = (state >> 8) & 0xffu;
  if (cnt - out == (uint32_t)R) {
    spill()[out] = lds[(out & (R - 1)) * BS];
    state += 0x100u;
  }
  lds[(cnt & (R - 1)) * BS] = v;
  state++;
}
template <int R, uint32_t BS, typename Spill>
__device__ __forceinline__ uint64_t ring_get(uint32_t& state, lds_u64* lds, Spill&& spill) {
  const uint32_t cnt = state & kListItems;
  state--;
  if (cnt <= ((state >> 8) & 0xffu)) {
    state -= 0x100u;
    return spill()[cnt - 1];
  }
  return lds[((cnt - 1) & (R - 1)) * BS];
}

// Masks of a node's six children from its size/type bytes (22-27), one bit a
// child: the bytes' flags times 1, 2, 4, ... summed by a four-byte dot product.
struct KidBytes {
  uint32_t lo, hi;  // children 0-3, 4-5
};
__device__ __forceinline__ uint32_t kid_mask(uint32_t lo, uint32_t hi) {
  return __builtin_amdgcn_udot4(lo & 0x01010101u, 0x08040201u, __builtin_amdgcn_udot4(hi & 0x0101u, 0x2010u, 0u, false),
                                false);
}
__device__ __forceinline__ uint32_t kids_present(KidBytes k) { return kid_mask(k.lo | (k.lo >> 1), k.hi | (k.hi >> 1)); }
__device__ __forceinline__ uint32_t kids_leaves(KidBytes k) {
  return kid_mask(((k.lo & 0x3c3c3c3cu) + 0x7c7c7c7cu) >> 7, ((k.hi & 0x3c3cu) + 0x7c7cu) >> 7);
}

// ---- slab tests by bounds ----------------------------------------------------------
// Six child boxes against a ray with one fused multiply-add per plane: a plane
// at q * 2^(e-8) + origin is met at t = q * S + C, S = 2^(e-8) * idir (exact) and
// C = (origin - o) * idir.  The reference rounds the plane, its distance from o
// and the product instead, so its t differs from this one, with u = 2^-24,
// P = origin - o and s = 2^(e-8), by at most
//   near planes  u |idir| (|origin| + 5 |P| + 1020 s)
//   far planes   u |idir| (|origin| + 6 |P| + 1020 s)     (C + W rounded too)
// (times 1 + 5u, and 2^-70 for denormal planes).  W is at least the sum of the
// two, over all axes.  The far planes and the far end of the ray's range are
// moved out by W: a child whose exit is then before its entry is missed by the
// reference too, and one whose exit is more than 2 W behind its entry is hit by
// it too, since min and max add no error.  Returns false when a child is in
// between, when W is not below 2^76 (infinite and NaN inputs, and all overflows
// of S, C and t), when the ray's range is NaN, or when the cull distance is
// -infinity: then the caller runs the reference's test.
//
// The near and far plane of an axis are picked by the direction's sign, which
// needs every box's lower bytes <= its upper ones: one v_perm takes two
// children's bytes out of two node words, each as the low byte of a half, which
// is q * 2^-24 exactly as a (denormal) half, and v_fma_mix takes halves.
// 150 vector instructions a node against 212 for the reference's roundings on the
// picked planes; 1.3 % of the node passes on the 1M-triangle scene and 4.4 % on the
// 21M-triangle one run the reference's test for one or two lanes.  Diffuse batch
// 557 -> 541 us (with records in treelet order 1146 -> 1104, staged 1423 -> 1382),
// 21M triangles in treelet order 2.18 -> 2.06 ms.
__device__ __forceinline__ bool bounded_children(const Words16& nd, F3 o, F3 idir, float tmin, float tmax, float cull,
                                                 uint32_t& hitmask) {
  const uint32_t ew = nd.w[4];  // exponents: bytes 18, 19 (word 4), 20 (word 5)
  const float sx = ldexpf(idir.x, (int)__builtin_amdgcn_sbfe((int)ew, 16, 8) + 16);  // S * 2^24
  const float sy = ldexpf(idir.y, ((int)ew >> 24) + 16);
  const float sz = ldexpf(idir.z, (int)__builtin_amdgcn_sbfe((int)nd.w[5], 0, 8) + 16);
  const float px = f_of(nd, 0) - o.x, py = f_of(nd, 1) - o.y, pz = f_of(nd, 2) - o.z;
  const float cx = px * idir.x, cy = py * idir.y, cz = pz * idir.z;
  auto fabs_ = [](float v) { return __builtin_fabsf(v); };
  const float ax = __builtin_fmaf(fabs_(px), 5.5f, fabs_(f_of(nd, 0))), ay = __builtin_fmaf(fabs_(py), 5.5f, fabs_(f_of(nd, 1))),
              az = __builtin_fmaf(fabs_(pz), 5.5f, fabs_(f_of(nd, 2)));
  const float a = __builtin_fmaf(ax, fabs_(idir.x), __builtin_fmaf(ay, fabs_(idir.y), az * fabs_(idir.z)));
  const float b = fabs_(sx) + fabs_(sy) + fabs_(sz);
  constexpr float k = 0x1.03p-23f;  // 1 % above 2 u
  const float w = __builtin_fmaf(a, k, __builtin_fmaf(b, k * 1020.0f * 0x1p-24f, 0x1p-60f));
  uint32_t nq[3][3], fq[3][3];
#pragma unroll
  for (int x = 0; x < 3; ++x) {
    const float d = x == 0 ? idir.x : x == 1 ? idir.y : idir.z;
    const uint32_t w0 = nd.w[7 + 3 * x], w1 = nd.w[8 + 3 * x], w2 = nd.w[9 + 3 * x];
    const uint32_t n0 = d < 0.0f ? 0x0c070c06u : 0x0c010c00u, f0 = n0 ^ 0x00060006u;
    const uint32_t n1 = n0 ^ 0x00020002u, f1 = f0 ^ 0x00020002u;
    nq[x][0] = __builtin_amdgcn_perm(w1, w0, n0);
    nq[x][1] = __builtin_amdgcn_perm(w2, w0, n1);
    nq[x][2] = __builtin_amdgcn_perm(w2, w1, n0);
    fq[x][0] = __builtin_amdgcn_perm(w1, w0, f0);
    fq[x][1] = __builtin_amdgcn_perm(w2, w0, f1);
    fq[x][2] = __builtin_amdgcn_perm(w2, w1, f0);
  }
  auto plane = [](uint32_t pair, int i, float s, float c) -> float {
    const uint16_t h = (uint16_t)((i & 1) ? pair >> 16 : pair & 0xffffu);
    return __builtin_fmaf((float)__builtin_bit_cast(_Float16, h), s, c);
  };
  // the cull test folded into the far end: for a non-NaN entry and a cull above
  // -inf, !(entry >= cull) is entry <= the largest float below cull; a NaN cull
  // culls nothing
  float far = tmax;
  if (!__builtin_isnan(cull)) {
    const uint32_t cu = __float_as_uint(cull);
    const uint32_t below = (int32_t)cu > 0 ? cu - 1u : ((cu << 1) == 0u ? 0x80000001u : cu + 1u);
    far = __builtin_fminf(tmax, __uint_as_float(below));
  }
  far += w;
  const float gx = cx + w, gy = cy + w, gz = cz + w;
  uint32_t missed = 0, least = 0xffffffffu;
#pragma unroll
  for (int i = 5; i >= 0; --i) {
    const float tn = __builtin_fmaxf(__builtin_fmaxf(__builtin_fmaxf(plane(nq[0][i >> 1], i, sx, cx), plane(nq[1][i >> 1], i, sy, cy)),
                                                     plane(nq[2][i >> 1], i, sz, cz)), tmin);
    const float tf = __builtin_fminf(__builtin_fminf(__builtin_fminf(plane(fq[0][i >> 1], i, sx, gx), plane(fq[1][i >> 1], i, sy, gy)),
                                                     plane(fq[2][i >> 1], i, sz, gz)), far);
    const uint32_t gap = __float_as_uint(tf - tn);
    missed = __builtin_amdgcn_alignbit(missed, gap, 31);  // its sign becomes bit 0
    least = min(least, gap);                              // negative gaps are the largest
  }
  hitmask = ~missed & 0x3fu;
  return w < 0x1p76f && !__builtin_isunordered(tmin, tmax) && cull != -__builtin_inff() && least > __float_as_uint(2.0f * w);
}

__device__ __forceinline__ uint32_t lanes_below(uint64_t mask) {
  return __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
}

__device__ __forceinline__ uint32_t slot_hash(uint32_t s) { return s * 2654435761u; }

// Ray traced by claim k of a single-scene launch: a listed ray, else rays in
// input order starting at claim_start and wrapping to 0.
__device__ __forceinline__ uint32_t claimed_ray(const TraceParams& p, uint32_t k) {
  if (p.ray_list) return p.ray_list[k];
  const uint32_t tail = p.n - p.claim_start;  // rays from claim_start to the end
  return k < tail ? k + p.claim_start : k - tail;
}

// The reference's accessedDataSize of one ray (vulkan_ray_tracing.cc:2260):
// every record size, the 8-byte leaf descriptors included.  It follows from
// the counters a ray keeps.  With a internal nodes, b instance leaves and c
// primitive leaves (the TLAS header record emitted):
//   fetch = 64 + 64a + 192b + 64c,  nodes = a + b + c,  records = 1 + a + 2b + 2c
// so b = (fetch/64 - 1 - nodes) / 2, c = records - 1 - nodes - b, and the
// descriptors add 8c bytes.
__device__ __forceinline__ uint32_t accessed_bytes_of(uint32_t n_rec, uint32_t n_nodes, uint32_t fetch) {
  if (n_rec == 0) return 0u;
  const uint32_t b = ((fetch >> 6) - 1u - n_nodes) >> 1;
  const uint32_t c = n_rec - 1u - n_nodes - b;
  return fetch + 8u * c;
}

__device__ __forceinline__ uint32_t wave_sum(uint32_t v) {
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

// Non-staged kernels are compiled for five waves per SIMD (at most 96 VGPRs);
// staged kernels are bounded by their LDS image instead.
// LM: the level pass.  The rays are traced again with the reference's
// tree_level_map kept per lane in global memory, and only each hit's max_level
// is written: the maximum over the final map (vulkan_ray_tracing.cc:2274-2279),
// where a node reassigned later keeps its last value.  Needed only for scenes
// in which a node is reachable at two levels; elsewhere every assignment of a
// node carries the same value and the traversal's running maximum is exact.
template <int MODE, int REC, int K, int STAGE, bool MULTI = false, bool LM = false>
__global__ __launch_bounds__(STAGE ? 64 : 256) __attribute__((amdgpu_waves_per_eu(STAGE ? 1 : (REC == kRecCsr || MODE == 1 || LM) ? 4 : 5)))
void trace_kernel(TraceParams p) {
  static_assert(!MULTI || (!REC && STAGE == 0), "batch kernels write hits only");
  static_assert(!LM || (!REC && STAGE == 0 && !MULTI), "the level pass writes max_level only");
  constexpr uint32_t BS = STAGE ? 64u : 256u;
  constexpr int NS = MODE == 1 ? 2 : 1;
  constexpr bool kSlab = REC == kRecSlab || REC == kRecSlab4;
  // ring length per list: treelet order keeps four groups where other LDS bounds
  // the waves on a CU (staging areas: two more waves; record rings: four blocks
  // instead of three, diffuse batch 1001 -> 946 us)
  constexpr int R = (STAGE || kSlab) && MODE == 1 ? 4 : K;
  constexpr uint32_t UNITS = STAGE / 64;
  constexpr uint32_t HSIZE = STAGE ? 2 * UNITS : 1;
  __shared__ uint64_t lds_stack[NS * R * BS];
  __shared__ uint4 stage_img[STAGE ? STAGE / 16 : 1];
  __shared__ uint32_t hkey[HSIZE];
  __shared__ uint16_t hpos[HSIZE];
  __shared__ uint8_t used[STAGE ? UNITS : 1];
  // slot table of the staging area: treelet, units held, iteration of the last
  // read served, staged on a prediction
  constexpr uint32_t MAXSLOTS = STAGE ? kMaxStageSlots : 1;
  __shared__ uint32_t sl_t[MAXSLOTS], sl_units[MAXSLOTS], sl_last[MAXSLOTS], sl_pred[MAXSLOTS], sl_first[MAXSLOTS];
  // prefetch effectiveness (src/gpgpu-sim/gpu-cache.cc:1960-2117): node slots
  // of staged units evicted unread (a later global read of one is TOO_EARLY)
  // and of recent global reads (staging one afterwards is TOO_LATE), each in a
  // direct-mapped table (a collision forgets the older slot)
  constexpr uint32_t EV = STAGE ? 128 : 1;
  __shared__ uint32_t ev_key[EV], dm_key[EV];
  // slab records: each lane's last RR slab entries (entry k at ring position
  // k % RR), written to the slab RG at a time
  typedef std::conditional_t<REC == kRecSlab4, uint32_t, uint64_t> rec_t;
  constexpr uint32_t RR = 64 / sizeof(rec_t), RG = 32 / sizeof(rec_t);
  __shared__ rec_t rec_ring[kSlab ? RR * BS : 1];

  // Staging-only parameters are read from the kernel-argument segment where
  // they are used (a scalar load each time; the empty asm keeps the compiler
  // from hoisting them) instead of living in scalar registers for the whole
  // launch: the staged kernels ran short of SGPRs and spilled 81 of them to
  // VGPR lanes, now 48 (plain+stage 1.347 -> 1.302 ms on the 1M-triangle batch).
  typedef const __attribute__((address_space(4))) TraceParams* kparams_ptr;
  auto kp = []() {
    kparams_ptr q = (kparams_ptr)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(q));
    return q;
  };
  const uint32_t tid = threadIdx.x;
  const uint32_t lane = tid & 63u;
  lds_u64* ldsA = (lds_u64*)(lds_stack + tid);
  typedef __attribute__((address_space(3))) rec_t lds_rec;
  lds_rec* ring = (lds_rec*)(rec_ring + (kSlab ? tid : 0u));
  const uint64_t lane_slot = (uint64_t)blockIdx.x * BS + tid;
  bool phase2 = false;  // treelet order: the current treelet was left (the lists are one stack from then on)
  // The lane's words of list l (0: the current one before the switch, 1: the
  // other), and of the list that the register group belongs to.  The spill area
  // is formed where it is used (rarely) instead of held in two registers.
  auto lds_of = [&](bool l) -> lds_u64* { return ldsA + (MODE == 1 && l ? (uint32_t)R * BS : 0u); };
  auto spill_of = [&](bool l) -> glb_u64* {
    uint32_t t = threadIdx.x;
    asm volatile("" : "+v"(t));
    const uint32_t per = p.spill_cap + (uint32_t)(K - R);
    return (glb_u64*)(p.spill + (((uint64_t)blockIdx.x * BS + t) * NS + (MODE == 1 && l ? 1u : 0u)) * per);
  };
  auto spill_cur = [&]() -> glb_u64* { return spill_of(phase2); };
  auto spill_other = [&]() -> glb_u64* { return spill_of(true); };
  // Scene of the lane's current ray (a batch kernel switches it per ray).
  const uint8_t* __restrict__ A = p.arena;
  uint64_t bytes = p.arena_bytes;
  uint64_t tlas = p.tlas;
  const uint32_t* owner = p.owner;
  uint32_t first_treelet = p.first_treelet;
  rtx_hit* hits_out = p.hits;
  const rtx_ray* rays_in = p.rays;
  uint32_t local_id = 0;
  __shared__ uint32_t job_base[MULTI ? kMaxBatchJobs + 1 : 1];
  if constexpr (MULTI) {
    for (uint32_t j = threadIdx.x; j <= p.n_jobs; j += BS) job_base[j] = j < p.n_jobs ? p.jobs[j].ray_base : p.n;
    __syncthreads();
  }

  Groups gs{0, 0, 0};
  uint32_t other = 0;  // treelet order before the switch: state of the other list
  bool active = false, exhausted = false;
  bool pending = false;  // the lane's completed ray still has to write its hit record
  uint32_t err = 0;

  F3 ro{}, rd{}, ridir{};
  float rtmin = 0.f, rtmax = 0.f;
  float min_thit = 0.f, min_thit_obj = 0.f;
  uint32_t closest_leaf = kNoSlot, closest_inst = kNoSlot;
  ObjRay cur{};
  uint32_t cur_inst = kNoSlot;
  uint32_t n_rec = 0, n_nodes = 0, fetch_bytes = 0, n_any = 0, max_level = 0;
  uint64_t rec_base = 0;
  uint32_t rec_flushed = 0;  // slab records: entries of the ray taken out of the ring

  // The entry a lane popped this iteration and processes below.
  bool has_e = false;
  uint64_t e = 0;

  // staging state (wave-uniform)
  uint32_t cooldown = 0, iter = 0, n_staged = 0;
  uint64_t st_treelets = 0, st_bytes = 0, st_wasted = 0, st_pred = 0, st_pred_hits = 0, st_fallback = 0;
  uint64_t st_timely = 0;
  uint32_t reads = 0, lds_hits = 0, too_early = 0, too_late = 0;
  uint32_t octant = 0;  // direction octant of the lane's ray (learned policy)
  // slots of `cap` units each (powers of two): nslots treelets stay resident
  uint32_t cap_shift = 0, nslots = 1;
  if constexpr (STAGE > 0) {
    uint32_t cap = UNITS;
    if (p.slot_units > 0 && p.slot_units < UNITS) cap = p.slot_units;
    while ((1u << cap_shift) < cap) cap_shift++;
    nslots = min(MAXSLOTS, UNITS >> cap_shift);
    for (uint32_t i = lane; i < HSIZE; i += 64) hkey[i] = 0;
    for (uint32_t i = lane; i < EV; i += 64) ev_key[i] = dm_key[i] = 0;
    for (uint32_t i = lane; i < MAXSLOTS; i += 64) {
      sl_t[i] = kNone;
      sl_units[i] = 0;
      sl_last[i] = 0;
      sl_pred[i] = 0;
      sl_first[i] = 0;
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }

  auto emit = [&](uint64_t off, uint32_t size, uint32_t type, uint32_t lvl) {
    if (type != RTX_TX_BVH_PRIMITIVE_LEAF_DESCRIPTOR) fetch_bytes += size;
    if constexpr (kSlab) {
      // a slab keeps the ray's first record_slab records, the rest are written
      // by a second pass over the rays that had more.  The entry holds what
      // the traversal knows; the owner and layout lookups wait for the
      // expansion, off the traversal's dependent chain.  It goes to the
      // lane's LDS ring first (flush_slab_group writes it out).
      const uint32_t slot = (uint32_t)(off >> 6);
      if constexpr (REC == kRecSlab4)
        ring[(n_rec & (RR - 1)) * BS] = slab_entry4(slot, type, lvl, p.rec_level_shift);
      else
        ring[(n_rec & (RR - 1)) * BS] = slab_entry(slot, type, lvl);
    } else if constexpr (REC == kRecCsr) {
      const uint64_t idx = rec_base + n_rec;
      if (idx < p.record_capacity) {
        uint32_t tl = owner ? owner[off >> 6] : RTX_NO_TREELET;
        const uint64_t roff = p.layout_remap ? p.layout_remap[off >> 6] : off;
        uint4 v;
        v.x = (uint32_t)roff;
        v.y = (uint32_t)(roff >> 32);
        v.z = tl;
        v.w = size | (type << 16) | ((lvl > 255u ? 255u : lvl) << 24);
        reinterpret_cast<uint4*>(p.records)[idx] = v;
      } else {
        err |= kErrRecords;
      }
    }
    n_rec++;
  };

  // Slab records: one group of the lane's ring, from entry rec_flushed on, to the
  // slab as two 16-byte stores that fill one aligned 32-byte sector (stores of
  // single entries scattered over the slabs cost partial-sector writes and fills).
  auto store_group = [&]() {
    if constexpr (kSlab) {
      uint4* dst = reinterpret_cast<uint4*>(slab_place<rec_t>(p.slabs, p.slabs_rest, p.record_slab, local_id, rec_flushed));
      uint4 v[2];
#pragma unroll
      for (uint32_t h = 0; h < 2; ++h) {
        uint32_t w[4];
#pragma unroll
        for (uint32_t k = 0; k < 16 / sizeof(rec_t); ++k) {
          const rec_t x = ring[((rec_flushed & (RR - 1)) + h * (16 / sizeof(rec_t)) + k) * BS];
          if constexpr (sizeof(rec_t) == 4) {
            w[k] = (uint32_t)x;
          } else {
            w[2 * k] = (uint32_t)x;
            w[2 * k + 1] = (uint32_t)((uint64_t)x >> 32);
          }
        }
        v[h] = make_uint4(w[0], w[1], w[2], w[3]);
      }
      dst[0] = v[0];
      dst[1] = v[1];
    }
  };
  // At the top of every iteration, which adds at most four entries (a refilled
  // ray's header and a visit's three): once some lane has no room for four
  // more, every lane with a whole group writes it.  Waiting for such a lane
  // keeps this out of most iterations.
  auto flush_slab_group = [&]() {
    if constexpr (kSlab) {
      if (__ballot(n_rec - rec_flushed > RR - 4u) == 0) return;
      if (n_rec - rec_flushed >= RG) {
        // entries past the slab are only counted
        if (rec_flushed < p.record_slab) store_group();
        rec_flushed += RG;
      }
    }
  };
  // The entries still in the ring when the ray's hit is written, as whole
  // groups too: the row is padded to whole groups, and the entries past the
  // ray's count (stale ring words) are never read.
  auto flush_slab_rest = [&]() {
    if constexpr (kSlab) {
      const uint32_t end = min(n_rec, p.record_slab);
      for (; rec_flushed < end; rec_flushed += RG) store_group();
      rec_flushed = n_rec;
    }
  };

  const uint32_t depth_limit = ((uint32_t)K + p.spill_cap) * kListDepth;
  auto save_group = [&]() {
    if (gs.word >= kGroupFirst)
      ring_put<R, BS>(gs.state, (uint64_t)gs.base | ((uint64_t)gs.word << 32), lds_of(phase2), spill_cur);
  };
  // Push one child, to the current list or the other one (after the switch
  // both are the list of the register group).
  auto push_entry = [&](uint64_t v, bool to_a) {
    if (MODE == 0 || to_a || phase2) {
      if ((gs.state & kListDepthMask) >= depth_limit) {
        err |= kErrStack;
        return;
      }
      save_group();
      gs.state += kListDepth;
      if constexpr (MODE == 0) {
        gs.base = e_slot(v);
        gs.word = group_word(e_flags(v) & kFlTop, e_level(v), (e_flags(v) >> 1) & 1u, 1u);
      } else {
        gs.word = 0;
        ring_put<R, BS>(gs.state, v, lds_of(phase2), spill_cur);
      }
    } else {
      if ((other & kListDepthMask) >= depth_limit) {
        err |= kErrStack;
        return;
      }
      other += kListDepth;
      ring_put<R, BS>(other, v, lds_of(true), spill_other);
    }
  };
  auto list_empty = [&]() -> bool { return gs.word < kGroupFirst && (gs.state & kListItems) == 0; };
  // current_treelet_root := host address of the moved node (:1748-1754)
  auto leave_treelet = [&]() {
    phase2 = true;
    gs.state |= other;  // the current list is empty: only the ray's flags are set
    other = 0;
  };

  // ---- the level pass's per-lane tree_level_map: open addressing over
  // lm_cap entries ((slot + 1) << 32 | level, 0 = empty), at most half full,
  // and the positions this ray wrote (for the final maximum and the clear)
  uint64_t* lm_t = nullptr;
  uint32_t* lm_l = nullptr;
  uint32_t lm_n = 0;
  if constexpr (LM) {
    lm_t = p.lm_table + lane_slot * (uint64_t)p.lm_cap;
    lm_l = p.lm_list + lane_slot * (uint64_t)(p.lm_cap / 2);
  }
  auto lm_pos = [&](uint32_t slot) -> uint32_t {
    uint32_t h = slot_hash(slot) & (p.lm_cap - 1);
    while (true) {
      const uint64_t v = lm_t[h];
      if (v == 0 || (uint32_t)(v >> 32) == slot + 1) return h;
      h = (h + 1) & (p.lm_cap - 1);
    }
  };
  auto lm_get = [&](uint32_t slot) -> uint32_t { return (uint32_t)lm_t[lm_pos(slot)]; };
  auto lm_set = [&](uint32_t slot, uint32_t level) {
    const uint32_t h = lm_pos(slot);
    if (lm_t[h] == 0) {
      if (lm_n >= p.lm_cap / 2) {  // the map is full: the ray reports a stack overflow
        err |= kErrStack;
        return;
      }
      lm_l[lm_n++] = h;
    }
    lm_t[h] = ((uint64_t)(slot + 1) << 32) | level;
  };

  // TLAS header slot of the lane's scene (instance leaves are stored relative to it)
  auto tlas_slot = [&]() -> uint32_t { return (uint32_t)(tlas >> 6); };
  // Treelet order: does `slot` belong to the current ("first") treelet?
  auto goes_current = [&](uint32_t slot) -> bool {
    if (MODE == 0) return true;
    if (phase2) return false;
    return owner[slot] == first_treelet;
  };
  // The first-treelet child bits of node slot `slot`: one byte per slot after
  // the owner words (bit i: child i of an internal node is owned by the first
  // treelet; bit 0 of an instance leaf: its BLAS root is).
  auto first_bits = [&](uint32_t slot) -> uint32_t {
    return reinterpret_cast<const uint8_t*>(owner + (bytes >> 6))[slot];
  };

  // Position of `slot` in the staged image, or kNone.
  auto staged_pos = [&](uint32_t slot) -> uint32_t {
    if constexpr (STAGE > 0) {
      if (n_staged == 0) return kNone;
      uint32_t h = slot_hash(slot) & (HSIZE - 1);
      for (uint32_t probe = 0; probe < HSIZE; ++probe) {
        const uint32_t k = hkey[h];
        if (k == slot + 1) return hpos[h];
        if (k == 0) return kNone;
        h = (h + 1) & (HSIZE - 1);
      }
    }
    return kNone;
  };

  // Read `count` 16-byte words of a node starting at byte `first` (a multiple
  // of 16): from the staged image when `pos` is its staged position, else
  // from global memory.  Explicit LDS and global paths keep both loads typed.
  auto read_words = [&](uint64_t off, uint32_t pos, uint32_t first, uint4* w, int count) {
    if constexpr (STAGE > 0) {
      reads++;
      if (pos != kNone) {
        lds_hits++;
        used[pos] = 1;
        sl_last[pos >> cap_shift] = iter;
        const uint4* q = stage_img + pos * 4 + first / 16;
        for (int k = 0; k < count; ++k) w[k] = q[k];
        return;
      }
      // a demand read from global memory: TOO_EARLY when the node's unit
      // was staged and evicted unread; remembered for TOO_LATE
      const uint32_t s = (uint32_t)(off >> 6), h = slot_hash(s) & (EV - 1);
      if (ev_key[h] == s + 1 && atomicCAS(&ev_key[h], s + 1, 0u) == s + 1) too_early++;
      dm_key[h] = s + 1;
    }
    const uint4* q = reinterpret_cast<const uint4*>(A + off + first);
    for (int k = 0; k < count; ++k) w[k] = q[k];
  };
  auto read_node = [&](uint64_t off, uint32_t pos) -> Words16 {
    uint4 w[4];
    read_words(off, pos, 0, w, 4);
    Words16 r;
    for (int k = 0; k < 4; ++k) {
      r.w[4 * k] = w[k].x;
      r.w[4 * k + 1] = w[k].y;
      r.w[4 * k + 2] = w[k].z;
      r.w[4 * k + 3] = w[k].w;
    }
    return r;
  };

  auto load_instance = [&](uint32_t inst) {
    const uint64_t ioff = (uint64_t)inst << 6;
    if (ioff + 128 > bytes) {
      err |= kErrRange;
      return;
    }
    const uint4* q = reinterpret_cast<const uint4*>(A + ioff + 16);
    uint4 a = q[0], b = q[1], c = q[2];
    float m[12] = {__uint_as_float(a.x), __uint_as_float(a.y), __uint_as_float(a.z), __uint_as_float(a.w),
                   __uint_as_float(b.x), __uint_as_float(b.y), __uint_as_float(b.z), __uint_as_float(b.w),
                   __uint_as_float(c.x), __uint_as_float(c.y), __uint_as_float(c.z), __uint_as_float(c.w)};
    cur = transform_ray(m, ro, rd, rtmin, rtmax);
    cur_inst = inst;
  };

  auto wave_sync = [&]() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  };

  // Account slot j's unused units, then empty it (wave-uniform).
  auto evict_slot = [&](uint32_t j) {
    if constexpr (STAGE > 0) {
      const uint32_t units = sl_units[j];
      if (sl_t[j] == kNone) return;
      const uint32_t base = j << cap_shift;
      uint32_t u = 0;
      for (uint32_t i = lane; i < units; i += 64) u += used[base + i] ? 1u : 0u;
      u = wave_sum(u);
      st_wasted += (uint64_t)(units - u) * 64;
      st_timely += (uint64_t)u * 64;
      if (sl_pred[j] && u > 0) st_pred_hits++;
      const uint64_t img = kp()->image_offset[sl_t[j]] / 64 + sl_first[j];
      for (uint32_t i = lane; i < units; i += 64) {
        if (used[base + i]) continue;
        const uint32_t s = kp()->image_slots[img + i];
        if (s != kNone) ev_key[slot_hash(s) & (EV - 1)] = s + 1;
      }
      wave_sync();
      if (lane == 0) {
        sl_t[j] = kNone;
        sl_units[j] = 0;
        sl_pred[j] = 0;
      }
      wave_sync();
      n_staged--;
    }
  };
  auto evict_all = [&]() {
    if constexpr (STAGE > 0)
      for (uint32_t j = 0; j < nslots; ++j) evict_slot(j);
  };

  // Copy treelet t (at most `max_units` 64-byte units of its image: the first
  // ones, or the last ones when `latter`) into a slot (wave-uniform): the slot
  // already holding it, else an empty one, else the least recently read one
  // that served no read in this iteration.  The hash table is rebuilt over
  // every resident slot.  Returns whether it copied.
  auto stage = [&](uint32_t t, uint32_t max_units, bool predicted, bool latter = false) -> bool {
    if constexpr (STAGE > 0) {
      const uint32_t tt = __builtin_amdgcn_readfirstlane(t);
      const uint32_t total = kp()->image_bytes[tt] / 64;
      uint32_t units = min(total, min(1u << cap_shift, max_units));
      units = __builtin_amdgcn_readfirstlane(units);
      if (units == 0) return false;
      const uint32_t first = latter ? total - units : 0u;
      // victim: the slot holding that part of t, else an empty slot, else the
      // least recently read slot that served no read in this iteration
      uint32_t victim = kNone, empty = kNone, lru = kNone, lru_it = 0;
      for (uint32_t j = 0; j < nslots; ++j) {
        const uint32_t sj = sl_t[j];
        if (sj == tt && sl_first[j] == first) victim = j;
        if (sj == kNone) {
          if (empty == kNone) empty = j;
        } else if (sl_last[j] < iter && (lru == kNone || sl_last[j] < lru_it)) {
          lru = j;
          lru_it = sl_last[j];
        }
      }
      if (victim != kNone) {
        if (sl_units[victim] >= units) {
          if (lane == 0) sl_last[victim] = iter;
          wave_sync();
          return false;
        }
      } else {
        victim = empty != kNone ? empty : lru;
        if (victim == kNone) return false;
      }
      victim = __builtin_amdgcn_readfirstlane(victim);
      evict_slot(victim);
      const uint32_t base = victim << cap_shift;
      const uint4* src = reinterpret_cast<const uint4*>(kp()->images + kp()->image_offset[tt]) + first * 4;
      for (uint32_t i = lane; i < units * 4; i += 64) stage_img[base * 4 + i] = src[i];
      for (uint32_t i = lane; i < units; i += 64) used[base + i] = 0;
      for (uint32_t i = lane; i < HSIZE; i += 64) hkey[i] = 0;
      wave_sync();
      if (lane == 0) {
        sl_t[victim] = tt;
        sl_units[victim] = units;
        sl_last[victim] = iter;
        sl_pred[victim] = predicted ? 1u : 0u;
        sl_first[victim] = first;
      }
      wave_sync();
      // insert every resident unit: unit i of the staging area is unit
      // i & (cap - 1) of slot i >> cap_shift
      for (uint32_t i = lane; i < (nslots << cap_shift); i += 64) {
        const uint32_t j = i >> cap_shift, u = i & ((1u << cap_shift) - 1);
        const uint32_t sj = sl_t[j];
        if (sj == kNone || u >= sl_units[j]) continue;
        const uint32_t s = kp()->image_slots[kp()->image_offset[sj] / 64 + sl_first[j] + u];
        if (s == kNone) continue;
        if (j == victim) {
          const uint32_t hd = slot_hash(s) & (EV - 1);
          if (dm_key[hd] == s + 1 && atomicCAS(&dm_key[hd], s + 1, 0u) == s + 1) too_late++;
        }
        uint32_t h = slot_hash(s) & (HSIZE - 1);
        for (uint32_t probe = 0; probe < HSIZE; ++probe) {
          if (atomicCAS(&hkey[h], 0u, s + 1) == 0u) {
            hpos[h] = (uint16_t)i;
            break;
          }
          h = (h + 1) & (HSIZE - 1);
        }
      }
      wave_sync();
      n_staged++;
      st_treelets++;
      st_bytes += (uint64_t)units * 64;
      if (predicted) st_pred++;
      return true;
    }
    return false;
  };

  // Pop the lane's next entry into `e`; false when its lists are empty.
  auto pop_next = [&]() -> bool {
    bool whole = false;
    if (gs.word < kGroupFirst) {
      if ((gs.state & kListItems) == 0) {
        if (MODE == 0 || (other & kListItems) == 0) return false;
        leave_treelet();
      }
      const uint64_t v = ring_get<R, BS>(gs.state, lds_of(phase2), spill_cur);
      if (MODE == 1 && !is_group(v)) {
        e = v;
        whole = true;
      } else {
        gs.base = (uint32_t)v;
        gs.word = (uint32_t)(v >> 32);
      }
    }
    if (!whole) {
      const uint32_t i = 15u - (uint32_t)__builtin_clz(gs.word);
      e = group_entry(gs.base, gs.word, i);
      if (MODE == 1 && !(gs.word & kGroupTop)) e |= (uint64_t)((cur_inst - (uint32_t)(tlas >> 6)) << 10) << 32;
      gs.word ^= kGroupFirst << i;
    }
    gs.state -= kListDepth;
    // every processed entry emits at least one record
    if (n_rec > kMaxStepsPerRay) err |= kErrSteps;
    return true;
  };

  // Write the hit record of the lane's completed ray (:2990-3038).  Deferred
  // to the wave's refill so the write path runs once per batch of completed
  // rays instead of in nearly every iteration.
  auto write_hit = [&]() {
    if constexpr (LM) {
      // the maximum over the final map; the entries are cleared for the next ray
      uint32_t mx = 0;
      for (uint32_t i = 0; i < lm_n; ++i) {
        const uint32_t h = lm_l[i];
        mx = max(mx, (uint32_t)lm_t[h]);
        lm_t[h] = 0;
      }
      lm_n = 0;
      hits_out[local_id].max_level = mx;
      if (err) {
        atomicOr(p.error, err);
        if (p.host_err) *reinterpret_cast<volatile uint32_t*>(p.host_err) = 1u;
      }
      return;
    }
    flush_slab_rest();
    uint4 o0 = make_uint4(0, 0, 0, 0), o1 = make_uint4(0, 0, 0, 0), o2 = make_uint4(0, 0, 0, 0);
    uint4 o4 = make_uint4(0xffffffffu, 0xffffffffu, 0, 0);
    if (err == 0 && min_thit < rtmax && closest_leaf != kNoSlot) {
      const Words16 q = load64B(A + ((uint64_t)closest_leaf << 6));
      const uint32_t inst_id = *reinterpret_cast<const uint32_t*>(A + ((uint64_t)closest_inst << 6) + 72);
      const F3 v0 = mk3(f_of(q, 4), f_of(q, 5), f_of(q, 6));
      const F3 v1 = mk3(f_of(q, 7), f_of(q, 8), f_of(q, 9));
      const F3 v2 = mk3(f_of(q, 10), f_of(q, 11), f_of(q, 12));
      const F3 ip = add3(ro, mk3(rd.x * min_thit, rd.y * min_thit, rd.z * min_thit));
      // the object-space ray of the closest hit's instance, recomputed from the
      // instance leaf (the same inputs as when the hit was accepted)
      const uint4* iq = reinterpret_cast<const uint4*>(A + ((uint64_t)closest_inst << 6) + 16);
      const uint4 ia = iq[0], ib = iq[1], ic = iq[2];
      const float im[12] = {__uint_as_float(ia.x), __uint_as_float(ia.y), __uint_as_float(ia.z), __uint_as_float(ia.w),
                            __uint_as_float(ib.x), __uint_as_float(ib.y), __uint_as_float(ib.z), __uint_as_float(ib.w),
                            __uint_as_float(ic.x), __uint_as_float(ic.y), __uint_as_float(ic.z), __uint_as_float(ic.w)};
      const ObjRay hr = transform_ray(im, ro, rd, rtmin, rtmax);
      const F3 op = add3(hr.o, mk3(hr.d.x * min_thit_obj, hr.d.y * min_thit_obj, hr.d.z * min_thit_obj));
      const F3 bc = barycentric(op, v0, v1, v2);
      o0 = make_uint4(1u, q.w[2], q.w[1] & 0x0fffffffu, inst_id);
      o1 = make_uint4(__float_as_uint(min_thit), __float_as_uint(ip.x), __float_as_uint(ip.y),
                      __float_as_uint(ip.z));
      o2 = make_uint4(__float_as_uint(bc.x), __float_as_uint(bc.y), __float_as_uint(bc.z), n_rec);
      o4.x = closest_inst << 6;
      o4.y = closest_inst >> 26;
    } else {
      o2.w = n_rec;
    }
    o4.z = accessed_bytes_of(n_rec, n_nodes, fetch_bytes);
    uint4* hq = reinterpret_cast<uint4*>(hits_out + local_id);
    hq[0] = o0;
    hq[1] = o1;
    hq[2] = o2;
    hq[3] = make_uint4(n_nodes, fetch_bytes, n_any, max_level);
    hq[4] = o4;
    if constexpr (kSlab) p.rec_counts[local_id] = n_rec;
    if (err) {
      atomicOr(p.error, err);
      if (p.host_err) *reinterpret_cast<volatile uint32_t*>(p.host_err) = 1u;
    }
  };

  // the TLAS header of a single-scene launch, read once
  uint4 tl_h0 = make_uint4(0, 0, 0, 0), tl_h1 = make_uint4(0, 0, 0, 0);
  if (!MULTI && tlas + 64 <= bytes) {
    const uint4* hq = reinterpret_cast<const uint4*>(A + tlas);
    tl_h0 = hq[0];
    tl_h1 = hq[1];
  }
  while (true) {
    flush_slab_group();
    // ---- refill idle lanes from the global ray counter (wave converged) ----
    const uint64_t idle = __ballot(!active);
    const uint32_t nidle = (uint32_t)__popcll(idle);
    if (!exhausted && nidle > 0 && (nidle == 64u || nidle >= p.refill)) {
      if (pending) {
        write_hit();
        pending = false;
      }
      const uint32_t leader = (uint32_t)__ffsll((long long)idle) - 1u;
      uint32_t base = 0;
      if (lane == leader) base = atomicAdd(p.ray_counter, nidle);
      base = (uint32_t)__builtin_amdgcn_readlane((int)base, (int)leader);
      if ((uint64_t)base + nidle >= p.n) exhausted = true;
      if (!active) {
        const uint32_t k = base + lanes_below(idle);
        const uint32_t r = k < p.n ? (MULTI ? k : claimed_ray(p, k)) : 0u;
        if (k < p.n && !MULTI && r >= p.n_rays) {
          // a listed ray outside the batch: reported, never read
          atomicOr(p.error, kErrRange);
          if (p.host_err) *reinterpret_cast<volatile uint32_t*>(p.host_err) = 1u;
        } else if (k < p.n) {
          active = true;
          local_id = r;
          if constexpr (MULTI) {
            // job holding ray r: job_base[j] <= r < job_base[j + 1]
            uint32_t lo = 0, hi = p.n_jobs;
            while (hi - lo > 1) {
              const uint32_t mid = (lo + hi) >> 1;
              if (job_base[mid] <= r)
                lo = mid;
              else
                hi = mid;
            }
            const BatchJob& jb = p.jobs[lo];
            A = jb.arena;
            bytes = jb.arena_bytes;
            tlas = jb.tlas;
            owner = jb.owner;
            first_treelet = jb.first_treelet;
            hits_out = jb.hits;
            rays_in = jb.rays;
            local_id = r - job_base[lo];
          }
          const uint4* rq = reinterpret_cast<const uint4*>(rays_in + local_id);
          uint4 r0 = rq[0], r1 = rq[1], r2 = rq[2];
          ro = mk3(__uint_as_float(r0.x), __uint_as_float(r0.y), __uint_as_float(r0.z));
          rtmin = __uint_as_float(r0.w);
          rd = mk3(__uint_as_float(r1.x), __uint_as_float(r1.y), __uint_as_float(r1.z));
          rtmax = __uint_as_float(r1.w);
          ridir = calc_idir(rd);
          octant = (rd.x < 0.f ? 1u : 0u) | (rd.y < 0.f ? 2u : 0u) | (rd.z < 0.f ? 4u : 0u);
          min_thit = rtmax;
          min_thit_obj = 0.f;
          closest_leaf = kNoSlot;
          closest_inst = kNoSlot;
          cur_inst = kNoSlot;
          n_rec = n_nodes = fetch_bytes = n_any = 0;
          rec_flushed = 0;
          max_level = 1;  // tree_level_map[topRootAddr] = 1
          if constexpr (REC == kRecCsr) rec_base = p.record_offsets[r];
          gs = Groups{0, 0, ((r2.x & RTX_RAY_FLAG_OPAQUE) ? kRayOpaque : 0u) |
                                ((r2.x & RTX_RAY_FLAG_TERMINATE_ON_FIRST_HIT) ? kRayTerminate : 0u)};
          other = 0;
          phase2 = false;
          err = 0;
          // TLAS header record and bounds test (vulkan_ray_tracing.cc:2444-2484)
          const uint64_t t = tlas;
          if (t + 64 > bytes) {
            err |= kErrRange;
          } else {
            emit(t, 64, RTX_TX_BVH_STRUCTURE, 0);
            uint4 h0, h1;
            if constexpr (MULTI) {
              const uint4* hq = reinterpret_cast<const uint4*>(A + t);
              h0 = hq[0];
              h1 = hq[1];
            } else {
              h0 = tl_h0;
              h1 = tl_h1;
            }
            const uint64_t root = t + ((uint64_t)h0.x | ((uint64_t)h0.y << 32));
            F3 lo = mk3(__uint_as_float(h0.z), __uint_as_float(h0.w), __uint_as_float(h1.x));
            F3 hi = mk3(__uint_as_float(h1.y), __uint_as_float(h1.z), __uint_as_float(h1.w));
            float th;
            // tree_level_map[topRootAddr] = 1, before the bounds test (:2470)
            if constexpr (LM) lm_set((uint32_t)(root >> 6), 1u);
            if (ray_box(lo, hi, ridir, ro, rtmin, rtmax, th)) {
              if ((root & 63) || root + 64 > bytes) {
                err |= kErrRange;
              } else {
                const uint32_t rs = (uint32_t)(root >> 6);
                push_entry(make_entry(rs, kFlTop, 1, 0), goes_current(rs));
              }
            }
          }
        }
      }
    }
    if (__ballot(active) == 0) {
      if (exhausted) break;
      continue;
    }

    // ---- pop the lane's next entry, or complete the ray ---------------------
    if (active && has_e && err != 0) has_e = false;
    if (active && !has_e) {
      if (err == 0 && pop_next()) {
        has_e = true;
      } else {
        // ray complete; its hit record is written at the wave's next refill
        pending = true;
        active = false;
      }
    }

    const uint32_t slot = e_slot(e);
    const uint32_t flags = e_flags(e);
    const uint32_t level = e_level(e);
    const uint64_t off = (uint64_t)slot << 6;

    const bool step = has_e && err == 0;

    // ---- staging decision (wave converged) -----------------------------------
    uint32_t pos = kNone;
    if constexpr (STAGE > 0) {
      iter++;
      const bool want = has_e && err == 0;
      if (want) pos = staged_pos(slot);
      if (kp()->prefetch != RTX_PREFETCH_NONE) {
        const uint32_t nact = (uint32_t)__popcll(__ballot(want));
        const uint32_t nmiss = (uint32_t)__popcll(__ballot(want && pos == kNone));
        if (cooldown > 0) {
          cooldown--;
        } else if (nact > 0 && 2 * nmiss > nact) {
          // The RT unit's vote (src/gpgpu-sim/shader.cc:3424-3446): the
          // treelet of every lane's next node is counted, and the most
          // popular one wins, ties going to the lowest root offset (the
          // ordered map's first maximum; dense treelet indices follow root
          // offsets).  Each round takes one distinct treelet, and the loop ends
          // when fewer lanes remain than the best count.  The candidate is read
          // by lane number (one v_readlane; a shuffle goes through LDS).
          const uint32_t own = (want && off + 64 <= bytes) ? owner[slot] : kNone;
          uint64_t rem = __ballot(own != kNone);
          const uint32_t voters = (uint32_t)__popcll(rem);
          uint32_t best = kNone, bestc = 0;
          while (rem && (uint32_t)__popcll(rem) >= bestc) {
            const uint32_t lead = (uint32_t)__ffsll((long long)rem) - 1u;
            const uint32_t cand = (uint32_t)__builtin_amdgcn_readlane((int)own, (int)lead);
            const uint64_t m = __ballot(own == cand);
            const uint32_t cnt = (uint32_t)__popcll(m);
            if (cnt > bestc || (cnt == bestc && cand < best)) {
              best = cand;
              bestc = cnt;
            }
            rem &= ~m;
          }
          // heuristics 0-3 (:3437-3559): always; share >= threshold; the
          // first round(n * share) units; the last round(n * share) units
          const float share = voters ? (float)bestc / (float)voters : 0.f;
          bool ok = best != kNone;
          if (kp()->prefetch == RTX_PREFETCH_POPULARITY && share < kp()->threshold) ok = false;
          bool staged = false;
          if (ok) {
            uint32_t maxu = UNITS;
            const bool part = kp()->prefetch == RTX_PREFETCH_PARTIAL || kp()->prefetch == RTX_PREFETCH_LATTER;
            if (part) maxu = (uint32_t)((float)(kp()->image_bytes[best] / 64) * share + 0.5f);
            // a treelet already resident is not staged again (the "same root as
            // the last prefetch" check of :3564)
            staged = stage(best, maxu, false, kp()->prefetch == RTX_PREFETCH_LATTER);
          }
          if (!staged) cooldown = 8;
          if (kp()->prefetch == RTX_PREFETCH_LEARNED) {
            // Each lane's predicted next treelets for (its treelet, its
            // octant).  A predicted treelet (its first pred_fraction of units)
            // is staged when the lanes' summed probability reaches min_score,
            // at most two per decision.
            uint4 row = make_uint4(0, 0, 0, 0);
            if (own != kNone && kp()->pred_table && own < kp()->pred_treelets)
              row = kp()->pred_table[(size_t)own * RTX_OCTANTS + octant];
            uint32_t ent[4] = {row.x, row.y, row.z, row.w};
            if (__ballot(row.x != 0) == 0) st_fallback++;
            uint32_t n_new = 0;
            for (int round = 0; round < 8 && n_new < 2; ++round) {
              uint32_t mine = 0;
              for (int k = 3; k >= 0; --k)
                if (ent[k] != 0) mine = ent[k];
              const uint64_t has = __ballot(mine != 0);
              if (has == 0) break;
              const uint32_t lead = (uint32_t)__ffsll((long long)has) - 1u;
              const uint32_t cand = (uint32_t)__builtin_amdgcn_readlane((int)mine, (int)lead) & 0xffffffu;
              float sc = 0.f;
              for (int k = 0; k < 4; ++k)
                if (ent[k] != 0 && (ent[k] & 0xffffffu) == cand) {
                  sc += (float)(ent[k] >> 24) * (1.f / 255.f);
                  ent[k] = 0;
                }
              for (int o = 32; o > 0; o >>= 1) sc += __shfl_xor(sc, o, 64);
              const uint32_t ct = cand - 1u;
              if (sc >= kp()->min_score && ct < kp()->pred_treelets) {
                const uint32_t units = kp()->image_bytes[ct] / 64;
                const uint32_t part = max(1u, (uint32_t)((float)units * kp()->pred_fraction + 0.5f));
                n_new += stage(ct, part, true) ? 1u : 0u;
              }
            }
          }
          if (want) pos = staged_pos(slot);
        }
      }
    }

    // ---- process the entry ----------------------------------------------------
    if (step) {
      has_e = false;
      if (MODE == 1 && !(flags & kFlTop) && e_inst(e, tlas_slot()) != cur_inst) load_instance(e_inst(e, tlas_slot()));
      // lanes on internal nodes (their own entry, or one reached through a
      // leaf in this iteration) share one internal-node pass at the end
      bool inner = err == 0 && !(flags & kFlLeaf);
      if (err != 0 || !(flags & kFlLeaf)) {
        // internal node: below; an error completes the ray next iteration
      } else if (flags & kFlTop) {
        // ---- instance leaf (:2602-2668 / :1872-1955) ----------------------
        if (off + 128 > bytes) {
          err |= kErrRange;
        } else {
          // a 128-byte leaf is served from LDS only when both of its units are staged
          uint32_t ipos = kNone;
          if constexpr (STAGE > 0)
            if (pos != kNone && (pos & ((1u << cap_shift) - 1)) + 1 < sl_units[pos >> cap_shift]) ipos = pos;
          uint4 w4[4];
          read_words(off, ipos, 16, w4, 4);
          // bytes 16..79 span both units of the leaf
          if constexpr (STAGE > 0)
            if (ipos != kNone) used[ipos + 1] = 1;
          const uint4 a = w4[0], b = w4[1], c = w4[2], d = w4[3];
          float m[12] = {__uint_as_float(a.x), __uint_as_float(a.y), __uint_as_float(a.z), __uint_as_float(a.w),
                         __uint_as_float(b.x), __uint_as_float(b.y), __uint_as_float(b.z), __uint_as_float(b.w),
                         __uint_as_float(c.x), __uint_as_float(c.y), __uint_as_float(c.z), __uint_as_float(c.w)};
          const uint64_t bvh = (uint64_t)d.x | ((uint64_t)d.y << 32);
          emit(off, 128, RTX_TX_BVH_INSTANCE_LEAF, level);
          n_nodes++;
          const uint64_t blas = off + bvh;
          if ((blas & 63) || blas + 64 > bytes) {
            err |= kErrRange;
          } else {
            const uint2 ro2 = *reinterpret_cast<const uint2*>(A + blas);
            emit(blas, 64, RTX_TX_BVH_STRUCTURE, level);
            cur = transform_ray(m, ro, rd, rtmin, rtmax);
            cur_inst = slot;
            uint32_t irel = 0;
            if (MODE == 1 && !inst_rel_of(slot, tlas_slot(), irel)) err |= kErrInstSlot;
            const uint64_t root = blas + ((uint64_t)ro2.x | ((uint64_t)ro2.y << 32));
            if ((root & 63) || root + 64 > bytes) {
              err |= kErrRange;
            } else {
              const uint32_t rs = (uint32_t)(root >> 6);
              if (level > max_level) max_level = level;
              if constexpr (LM) lm_set(rs, lm_get(slot));  // :2668 / :1944
              const bool to_a = MODE == 0 || (!phase2 && (first_bits(slot) & 1u));
              // The BLAS root is popped next when it goes on top of the list
              // the next pop takes: always in plain order; in treelet order
              // when it joins the current list, or the other list while the
              // current one is empty (that pop starts phase 2).  Such a root is
              // tested in this iteration's internal-node pass instead.
              if (err == 0 && (MODE == 0 || to_a || phase2 || list_empty())) {
                if (MODE == 1 && !to_a && !phase2) leave_treelet();
                e = make_entry(rs, 0u, level, irel);
                inner = true;
              } else {
                push_entry(make_entry(rs, 0u, level, irel), to_a);
              }
            }
          }
        }
      } else {
        // ---- primitive leaf (:2789-2985 / :2073-2203) ---------------------
        if (off + 64 > bytes) {
          err |= kErrRange;
        } else {
          emit(off, 8, RTX_TX_BVH_PRIMITIVE_LEAF_DESCRIPTOR, level);
          const Words16 q = read_node(off, pos);
          if (((q.w[1] >> 29) & 1u) == 0u) {
            if ((q.w[3] & 0x1ffffu) != 0u) err |= kErrType;
            const F3 v0 = mk3(f_of(q, 4), f_of(q, 5), f_of(q, 6));
            const F3 v1 = mk3(f_of(q, 7), f_of(q, 8), f_of(q, 9));
            const F3 v2 = mk3(f_of(q, 10), f_of(q, 11), f_of(q, 12));
            float th = 0.f;
            const bool h = mt_test(v0, v1, v2, cur.o, cur.d, th);
            const float wt = th / cur.tmult;
            bool accept;
            if (MODE == 0) {
              accept = h && rtmin <= wt && wt <= rtmax;
              if (accept && (gs.state & kRayOpaque) && wt < min_thit) min_thit = th / cur.tmult;
            } else {
              accept = h && rtmin <= wt && wt <= rtmax && wt < min_thit;
              if (accept) min_thit = th / cur.tmult;
            }
            if (accept) {
              min_thit_obj = th;
              closest_leaf = slot;
              closest_inst = cur_inst;
              emit(off, 64, RTX_TX_BVH_QUAD_LEAF_HIT, level);
              n_nodes++;
              if (MODE == 0 && !(gs.state & kRayOpaque)) n_any++;
              if (gs.state & kRayTerminate) {
                gs = Groups{0, 0, gs.state & (kRayOpaque | kRayTerminate)};
                other = 0;
              }
            } else {
              emit(off, 64, RTX_TX_BVH_QUAD_LEAF, level);
              n_nodes++;
            }
          } else {
            emit(off, 64, RTX_TX_BVH_PROCEDURAL_LEAF, level);
            n_nodes++;
          }
        }
        // the lane pops its next entry now; an internal node is tested in this
        // iteration's internal-node pass (in staged kernels its read still
        // probes the staged treelets; it only misses the iteration's vote)
        if (err == 0 && pop_next()) {
          if (err == 0 && !(e_flags(e) & kFlLeaf))
            inner = true;
          else
            has_e = true;
        }
      }
      if (inner) {
        const uint32_t slot = e_slot(e);
        const uint32_t flags = e_flags(e);
        const uint32_t level = e_level(e);
        const uint64_t off = (uint64_t)slot << 6;
        if (MODE == 1 && !(flags & kFlTop) && e_inst(e, tlas_slot()) != cur_inst) load_instance(e_inst(e, tlas_slot()));
        if (err == 0) {
          // ---- internal node (top :2499-2599 / bottom :2686-2786) ----------
          if (off + 64 > bytes) {
            err |= kErrRange;
          } else {
            const Words16 nd = read_node(off, STAGE > 0 ? staged_pos(slot) : pos);
            // Treelet order before the first switch: which children the first
            // treelet owns (read beside the node, used after its tests)
            const uint32_t fbits = (MODE == 1 && !phase2) ? first_bits(slot) : 0u;
            emit(off, 64, RTX_TX_BVH_INTERNAL_NODE, level);
            n_nodes++;
            const bool top = (flags & kFlTop) != 0;
            F3 o, idir;
            float tmin, tmax, cull;
            if (top) {
              o = ro;
              idir = ridir;
            } else {
              o = cur.o;
              idir = cur.idir;
            }
            // the object-space range and cull distance scale with the direction
            // (x * 1 = x for the TLAS); formed per node, they hold no registers
            const float tscale = top ? 1.0f : cur.tmult;
            tmin = rtmin * tscale;
            tmax = rtmax * tscale;
            cull = min_thit * tscale;
            const uint64_t first_child = off + (uint64_t)((int64_t)(int32_t)nd.w[3] * 64);
            const KidBytes kids{__builtin_amdgcn_alignbyte(nd.w[6], nd.w[5], 2), nd.w[6] >> 16};
            uint32_t hitmask = 0;
            bool sure = false;
            if (p.ordered_boxes) sure = bounded_children(nd, o, idir, tmin, tmax, cull, hitmask);
            hitmask &= kids_present(kids);
            if (!sure) {
              // the reference's own test (read again: its words are not kept)
              uint64_t at = off;
              asm volatile("" : "+v"(at));
              const Words16 nw = load64B(A + at);
              const F3 sc = child_scales((int)(int8_t)byte_of(nw, 18), (int)(int8_t)byte_of(nw, 19), (int)(int8_t)byte_of(nw, 20));
              hitmask = 0;
#pragma unroll
              for (int i = 0; i < 6; ++i) {
                const uint32_t size = byte_of(nw, 22 + i) & 3u;
                if (size > 0) {
                  F3 lo, hi;
                  child_box(nw, i, sc, lo, hi);
                  float th;
                  bool h = ray_box(lo, hi, idir, o, tmin, tmax, th);
                  if (h && th >= cull) h = false;
                  if (h) hitmask |= 1u << i;
                }
              }
            }
            if (hitmask) {
              const uint32_t lvl = level + 1;
              if (lvl > max_level) max_level = lvl;
              // the node's map value when it is processed (:2569-2581, :2756-2767,
              // :1837-1858, :2034-2055)
              const uint32_t lm_child = LM ? lm_get(slot) + 1 : 0u;
              const uint32_t inst = top ? 0u : e_inst_rel(e);
              const uint32_t base_flags = top ? kFlTop : 0u;
              bool pushed = false;
              if constexpr (!LM) {
                // A scene of regular nodes: the hit children of a list are one
                // group, without the one that its next pop would take.  No child
                // needs a check here: the scene walk placed all of them in the
                // arena.
                if (p.regular_nodes) {
                  pushed = true;
                  const uint32_t mine = MODE == 0 || phase2 ? hitmask : hitmask & fbits;  // to the register group's list
                  const uint32_t theirs = hitmask & ~mine;
                  const uint32_t d_mine = (uint32_t)__popc(mine) * kListDepth, d_theirs = (uint32_t)__popc(theirs) * kListDepth;
                  if ((gs.state & kListDepthMask) + d_mine > depth_limit ||
                      (MODE == 1 && (other & kListDepthMask) + d_theirs > depth_limit)) {
                    err |= kErrStack;
                  } else {
                    const uint32_t leaves = kids_leaves(kids);
                    const uint32_t word = group_word(top, lvl, leaves, 0u);
                    const uint32_t first = slot + nd.w[3];
                    uint32_t next;  // one bit
                    if (MODE == 0) {
                      const uint32_t im = mine & ~leaves;
                      next = im & (0u - im);
                    } else {
                      next = mine ? 0x80000000u >> __builtin_clz(mine) : 0u;
                    }
                    if (MODE == 0 || phase2 || top) {
                      const uint32_t rest = mine & ~next;
                      if (rest) {
                        save_group();
                        gs.base = first;
                        gs.word = word | (rest << 16);
                      }
                      gs.state += d_mine;
                      if (MODE == 1 && theirs) {
                        ring_put<R, BS>(other, (uint64_t)first | ((uint64_t)(word | (theirs << 16)) << 32), lds_of(true),
                                        spill_other);
                        other += d_theirs;
                      }
                    } else {
                      for (uint32_t m = hitmask & ~next; m; m &= m - 1) {
                        const uint32_t i = (uint32_t)__builtin_ctz(m);
                        push_entry(group_entry(first, word, i) | ((uint64_t)inst << 42), (mine >> i) & 1u);
                      }
                      gs.state += next ? kListDepth : 0u;
                    }
                    if (next) {
                      e = group_entry(first, word, (uint32_t)__builtin_ctz(next)) | ((uint64_t)inst << 42);
                      has_e = true;
                      gs.state -= kListDepth;
                      if (n_rec > kMaxStepsPerRay) err |= kErrSteps;
                    }
                  }
                }
              }
              int deferred = -1;
              uint32_t deferred_cs = 0;
              const uint32_t cur_bits = fbits;
              uint64_t child = first_child;
#pragma unroll
              for (int i = 0; i < 6 && !pushed; ++i) {
                const uint32_t info = byte_of(nd, 22 + i) & 0x3fu;
                const uint64_t c = child;
                child += (uint64_t)(info & 3u) * 64;
                if (!(hitmask & (1u << i))) continue;
                const uint32_t ctype = info >> 2;
                const bool leaf = ctype != 0;
                if (top && leaf && ctype != 1u) err |= kErrType;
                if ((c & 63) || c + 64 > bytes) {
                  err |= kErrRange;
                  continue;
                }
                const uint32_t cs = (uint32_t)(c >> 6);
                if constexpr (LM) lm_set(cs, lm_child);
                if (MODE == 0 && !leaf && deferred < 0) {
                  deferred = i;
                  deferred_cs = cs;
                  continue;
                }
                push_entry(make_entry(cs, base_flags | (leaf ? kFlLeaf : 0u), lvl, inst), MODE == 0 || ((cur_bits >> i) & 1u));
              }
              if (MODE == 0 && deferred >= 0 && !pushed) {
                push_entry(make_entry(deferred_cs, base_flags, lvl, inst), true);
              }
            }
          }
        }
      }
    }
  }

  if (pending) write_hit();

  if constexpr (STAGE > 0) {
    evict_all();
    const uint32_t r = wave_sum(reads), hl = wave_sum(lds_hits);
    const uint32_t te = wave_sum(too_early), tl = wave_sum(too_late);
    if (lane == 0) {
      atomicAdd(&p.stats[8], (unsigned long long)st_timely);
      atomicAdd(&p.stats[9], (unsigned long long)te * 64ull);
      atomicAdd(&p.stats[10], (unsigned long long)tl * 64ull);
      atomicAdd(&p.stats[0], (unsigned long long)r);
      atomicAdd(&p.stats[1], (unsigned long long)hl);
      atomicAdd(&p.stats[2], (unsigned long long)st_treelets);
      atomicAdd(&p.stats[3], (unsigned long long)st_bytes);
      atomicAdd(&p.stats[4], (unsigned long long)st_wasted);
      atomicAdd(&p.stats[5], (unsigned long long)st_pred);
      atomicAdd(&p.stats[6], (unsigned long long)st_pred_hits);
      atomicAdd(&p.stats[7], (unsigned long long)st_fallback);
    }
  }
}

// ---- record offsets: exclusive scan of hits[i].n_records --------------------
constexpr uint32_t kScanBlock = 256;
constexpr uint32_t kScanItems = 4;
constexpr uint32_t kScanTile = kScanBlock * kScanItems;

__device__ __forceinline__ uint64_t block_exclusive_scan(uint64_t v, uint64_t* smem, uint64_t& total) {
  const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
  uint64_t x = v;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    uint64_t y = __shfl_up(x, d, 64);
    if (lane >= (uint32_t)d) x += y;
  }
  if (lane == 63) smem[wave] = x;
  __syncthreads();
  uint64_t wsum = 0;
  for (uint32_t w = 0; w < wave; ++w) wsum += smem[w];
  total = smem[0] + smem[1] + smem[2] + smem[3];
  __syncthreads();
  return wsum + x - v;
}

__global__ __launch_bounds__(kScanBlock) void scan_tiles(const rtx_hit* hits, uint32_t n, uint64_t* out,
                                                         uint64_t* tile_sums) {
  __shared__ uint64_t smem[4];
  const uint64_t base = (uint64_t)blockIdx.x * kScanTile + threadIdx.x * kScanItems;
  uint64_t v[kScanItems];
  uint64_t s = 0;
#pragma unroll
  for (uint32_t k = 0; k < kScanItems; ++k) {
    v[k] = base + k < n ? hits[base + k].n_records : 0;
    s += v[k];
  }
  uint64_t total;
  uint64_t ex = block_exclusive_scan(s, smem, total);
#pragma unroll
  for (uint32_t k = 0; k < kScanItems; ++k) {
    if (base + k < n) out[base + k] = ex;
    ex += v[k];
  }
  if (threadIdx.x == 0) tile_sums[blockIdx.x] = total;
}

__global__ __launch_bounds__(kScanBlock) void scan_sums(uint64_t* tile_sums, uint32_t n_tiles, uint64_t* out,
                                                        uint32_t n) {
  __shared__ uint64_t smem[4];
  uint64_t carry = 0;
  for (uint32_t b = 0; b < n_tiles; b += kScanBlock) {
    const uint32_t i = b + threadIdx.x;
    uint64_t v = i < n_tiles ? tile_sums[i] : 0;
    uint64_t total;
    uint64_t ex = block_exclusive_scan(v, smem, total);
    if (i < n_tiles) tile_sums[i] = carry + ex;
    carry += total;
  }
  if (threadIdx.x == 0) out[n] = carry;
}

__global__ __launch_bounds__(kScanBlock) void scan_add(uint64_t* out, uint32_t n, const uint64_t* tile_sums) {
  const uint64_t base = (uint64_t)blockIdx.x * kScanTile + threadIdx.x * kScanItems;
  const uint64_t add = tile_sums[blockIdx.x];
#pragma unroll
  for (uint32_t k = 0; k < kScanItems; ++k)
    if (base + k < n) out[base + k] += add;
}

// ---- cooperative traversal for small batches (both orders) -----------------
//
// One ray per group of kWideLanes lanes.  Every lane of a group holds the same
// ray state and takes the same branches; an internal node's six child boxes
// are tested by lanes 0-5 of the group at once, so a traversal step issues a
// fraction of the instructions of trace_kernel, whose lanes each test all six.
// A batch too small to fill the GPU is bound by the step latency of its
// longest rays, which this shortens.  Slab records go to their row directly (one
// store by the group's first lane): 256 rays of the 1M-triangle scene with records
// take 127 -> 94 us in plain order and 179 -> 121 us in treelet order, the 32-ray
// batch of the sphere 110 -> 79 us, of which the finishing launch is 10.  The per-ray sequence of popped entries,
// and so every hit record and counter, is that of trace_kernel<MODE, false, K,
// 0>: each list (one in plain order, two in treelet order) is an LDS array of
// `cap` = K + spill_cap entries per ray, and a push fails exactly when the
// per-lane kernel's LDS ring and spill area for that list are both full.
// Lane j pushes hit child j itself, at its place in that push sequence.
constexpr uint32_t kWideLanes = 8;
constexpr uint32_t kWideCap = 144;  // K + spill_cap for K <= 16
constexpr uint32_t kWideBlock = 256;

// Byte `base + j` (j in 0..5) of a node held in registers, for a lane-varying j:
// it lies in word base / 4 or the next one.
__device__ __forceinline__ uint32_t byte_at(const Words16& n, int base, uint32_t j) {
  const uint32_t b = (uint32_t)base + j;
  const uint32_t w = (b >> 2) == (uint32_t)(base >> 2) ? n.w[base >> 2] : n.w[(base >> 2) + 1];
  return (w >> ((b & 3u) * 8u)) & 0xffu;
}

template <int MODE, bool REC>
__global__ __launch_bounds__(kWideBlock) void trace_wide(TraceParams p, uint32_t cap, uint32_t groups) {
  constexpr uint32_t NS = MODE == 1 ? 2 : 1;
  extern __shared__ uint64_t wide_stk[];  // NS * kWideCap entries per ray (wide_lds_bytes)
  const uint32_t tid = threadIdx.x;
  const uint32_t lane = tid & 63u;
  const uint32_t j = tid & (kWideLanes - 1);
  const uint32_t gbase = lane & ~(kWideLanes - 1);  // the group's first lane in the wave
  // (groups past the launch's limit hold no ray)
  lds_u64* sta = (lds_u64*)wide_stk + ((tid >> 6) * groups + min(gbase / kWideLanes, groups - 1u)) * (NS * kWideCap);
  lds_u64* stb = sta + (NS - 1) * kWideCap;
  const uint8_t* __restrict__ A = p.arena;
  const uint64_t bytes = p.arena_bytes;
  const uint64_t tlas = p.tlas;
  const uint32_t* owner = p.owner;
  const uint32_t first_treelet = p.first_treelet;

  bool active = false, exhausted = false, pending = false;
  bool phase2 = false;
  // plain order: the groups of trace_kernel, their older ones (da of them) in LDS
  Groups gs{0, 0, 0};
  uint32_t depth = 0;
  // this lane's child in the byte arrays of a node's words (a zero-extended byte
  // by one v_perm from two words): lower bounds start a word, upper bounds and the
  // size/type bytes start in a word's third byte
  const uint32_t jj = min(j, 5u), sel_lo = 0x0c0c0c00u | jj, sel_hi = 0x0c0c0c00u | (jj + 2u);
  uint32_t da = 0, db = 0, err = 0, local_id = 0;
  F3 ro{}, rd{}, ridir{};
  float rtmin = 0.f, rtmax = 0.f;
  uint32_t rflags = 0;
  float min_thit = 0.f, min_thit_obj = 0.f;
  uint32_t closest_leaf = kNoSlot, closest_inst = kNoSlot;
  ObjRay cur{};
  uint32_t cur_inst = kNoSlot;
  bool ray_ok = false, cur_ok = false;
  uint32_t n_rec = 0, n_nodes = 0, fetch_bytes = 0, n_any = 0, max_level = 0;
  bool has_e = false;
  uint64_t e = 0;

  auto emit = [&](uint64_t off, uint32_t size, uint32_t type, uint32_t lvl) {
    if (type != RTX_TX_BVH_PRIMITIVE_LEAF_DESCRIPTOR) fetch_bytes += size;
    if constexpr (REC) {
      // straight to the ray's slab row
      if (j == 0 && n_rec < p.record_slab) {
        const uint32_t at = (uint32_t)(off >> 6), k = n_rec & ~7u;
        if (p.rec_level_shift)
          slab_place<uint32_t>(p.slabs, p.slabs_rest, p.record_slab, local_id, k)[n_rec & 7u] =
              slab_entry4(at, type, lvl, p.rec_level_shift);
        else
          slab_place<uint64_t>(p.slabs, p.slabs_rest, p.record_slab, local_id, k)[n_rec & 7u] = slab_entry(at, type, lvl);
      }
    }
    n_rec++;
  };
  // lane 0 of the group writes; the group's later pops read it back in order
  // (the list depths are updated through selects, not a reference to one of
  // them, which would put both in scratch memory)
  auto save_group = [&]() {
    if (gs.word < kGroupFirst) return;
    if (j == 0) sta[da] = (uint64_t)gs.base | ((uint64_t)gs.word << 32);
    da++;
  };
  auto push = [&](uint64_t v, bool to_a) {
    if constexpr (MODE == 0) {
      if (depth >= cap) {
        err |= kErrStack;
        return;
      }
      save_group();
      gs.base = e_slot(v);
      gs.word = group_word(e_flags(v) & kFlTop, e_level(v), (e_flags(v) >> 1) & 1u, 1u);
      depth++;
      return;
    }
    const bool a = to_a;
    const uint32_t d = a ? da : db;
    if (d >= cap) {
      err |= kErrStack;
      return;
    }
    if (j == 0) *(a ? sta + d : stb + d) = v;
    da = a ? d + 1 : da;
    db = a ? db : d + 1;
  };
  auto pop_next = [&]() -> bool {
    if constexpr (MODE == 0) {
      if (gs.word < kGroupFirst) {
        if (da == 0) return false;
        const uint64_t v = sta[--da];
        gs.base = (uint32_t)v;
        gs.word = (uint32_t)(v >> 32);
      }
      const uint32_t i = 15u - (uint32_t)__builtin_clz(gs.word);
      e = group_entry(gs.base, gs.word, i);
      gs.word ^= kGroupFirst << i;
      depth--;
      if (n_rec > kMaxStepsPerRay) err |= kErrSteps;
      return true;
    }
    if (da == 0 && db == 0) return false;
    const bool a = da > 0;
    // moving to the other list: current_treelet_root := host address of the moved node (:1748-1754)
    if (!a) phase2 = true;
    const uint32_t d = (a ? da : db) - 1;
    e = *(a ? sta + d : stb + d);
    da = a ? d : da;
    db = a ? db : d;
    if (n_rec > kMaxStepsPerRay) err |= kErrSteps;
    return true;
  };
  auto tlas_slot = [&]() -> uint32_t { return (uint32_t)(tlas >> 6); };
  auto goes_current = [&](uint32_t slot) -> bool {
    if (MODE == 0) return true;
    if (phase2) return false;
    return owner[slot] == first_treelet;
  };
  // first-treelet child bits of a node slot (one byte per slot after the owner words)
  auto first_bits = [&](uint32_t slot) -> uint32_t {
    return reinterpret_cast<const uint8_t*>(owner + (bytes >> 6))[slot];
  };
  auto load_instance = [&](uint32_t inst) {
    const uint64_t ioff = (uint64_t)inst << 6;
    if (ioff + 128 > bytes) {
      err |= kErrRange;
      return;
    }
    const uint4* q = reinterpret_cast<const uint4*>(A + ioff + 16);
    const uint4 a = q[0], b = q[1], c = q[2];
    const float m[12] = {__uint_as_float(a.x), __uint_as_float(a.y), __uint_as_float(a.z), __uint_as_float(a.w),
                         __uint_as_float(b.x), __uint_as_float(b.y), __uint_as_float(b.z), __uint_as_float(b.w),
                         __uint_as_float(c.x), __uint_as_float(c.y), __uint_as_float(c.z), __uint_as_float(c.w)};
    cur = transform_ray(m, ro, rd, rtmin, rtmax);
    cur_ok = slab_inputs_ok(cur.o, cur.d, cur.idir, cur.tmin, cur.tmax);
    cur_inst = inst;
  };
  // the hit record (as trace_kernel writes it): lanes 0-3 store one 16-byte word each
  auto write_hit = [&]() {
    uint4 o0 = make_uint4(0, 0, 0, 0), o1 = make_uint4(0, 0, 0, 0), o2 = make_uint4(0, 0, 0, 0);
    uint4 o4 = make_uint4(0xffffffffu, 0xffffffffu, 0, 0);
    if (err == 0 && min_thit < rtmax && closest_leaf != kNoSlot) {
      const Words16 q = load64B(A + ((uint64_t)closest_leaf << 6));
      const uint32_t inst_id = *reinterpret_cast<const uint32_t*>(A + ((uint64_t)closest_inst << 6) + 72);
      const F3 v0 = mk3(f_of(q, 4), f_of(q, 5), f_of(q, 6));
      const F3 v1 = mk3(f_of(q, 7), f_of(q, 8), f_of(q, 9));
      const F3 v2 = mk3(f_of(q, 10), f_of(q, 11), f_of(q, 12));
      const F3 ip = add3(ro, mk3(rd.x * min_thit, rd.y * min_thit, rd.z * min_thit));
      const uint4* iq = reinterpret_cast<const uint4*>(A + ((uint64_t)closest_inst << 6) + 16);
      const uint4 ia = iq[0], ib = iq[1], ic = iq[2];
      const float im[12] = {__uint_as_float(ia.x), __uint_as_float(ia.y), __uint_as_float(ia.z), __uint_as_float(ia.w),
                            __uint_as_float(ib.x), __uint_as_float(ib.y), __uint_as_float(ib.z), __uint_as_float(ib.w),
                            __uint_as_float(ic.x), __uint_as_float(ic.y), __uint_as_float(ic.z), __uint_as_float(ic.w)};
      const ObjRay hr = transform_ray(im, ro, rd, rtmin, rtmax);
      const F3 op = add3(hr.o, mk3(hr.d.x * min_thit_obj, hr.d.y * min_thit_obj, hr.d.z * min_thit_obj));
      const F3 bc = barycentric(op, v0, v1, v2);
      o0 = make_uint4(1u, q.w[2], q.w[1] & 0x0fffffffu, inst_id);
      o1 = make_uint4(__float_as_uint(min_thit), __float_as_uint(ip.x), __float_as_uint(ip.y),
                      __float_as_uint(ip.z));
      o2 = make_uint4(__float_as_uint(bc.x), __float_as_uint(bc.y), __float_as_uint(bc.z), n_rec);
      o4.x = closest_inst << 6;
      o4.y = closest_inst >> 26;
    } else {
      o2.w = n_rec;
    }
    o4.z = accessed_bytes_of(n_rec, n_nodes, fetch_bytes);
    uint4* hq = reinterpret_cast<uint4*>(p.hits + local_id);
    if (j == 0)
      hq[0] = o0;
    else if (j == 1)
      hq[1] = o1;
    else if (j == 2)
      hq[2] = o2;
    else if (j == 3)
      hq[3] = make_uint4(n_nodes, fetch_bytes, n_any, max_level);
    else if (j == 4)
      hq[4] = o4;
    if (REC && j == 0) p.rec_counts[local_id] = n_rec;
    if (err && j == 0) {
      atomicOr(p.error, err);
      if (p.host_err) *reinterpret_cast<volatile uint32_t*>(p.host_err) = 1u;
    }
  };

  uint4 tl_h0 = make_uint4(0, 0, 0, 0), tl_h1 = make_uint4(0, 0, 0, 0);
  if (tlas + 64 <= bytes) {
    const uint4* hq = reinterpret_cast<const uint4*>(A + tlas);
    tl_h0 = hq[0];
    tl_h1 = hq[1];
  }
  while (true) {
    // ---- refill idle groups from the global ray counter (wave converged) ----
    const uint64_t idle = __ballot(j == 0 && !active && gbase < groups * kWideLanes);
    const uint32_t nidle = (uint32_t)__popcll(idle);
    if (!exhausted && nidle > 0 && (nidle == groups || nidle * kWideLanes >= p.refill)) {
      if (pending) {
        write_hit();
        pending = false;
      }
      // a launch with a place for every ray takes them by wave: no counter
      uint32_t base = (blockIdx.x * (kWideBlock / 64) + (tid >> 6)) * groups;
      if ((uint64_t)gridDim.x * (kWideBlock / 64) * groups >= p.n) {
        exhausted = true;
      } else {
        const uint32_t leader = (uint32_t)__ffsll((long long)idle) - 1u;
        if (lane == leader) base = atomicAdd(p.ray_counter, nidle);
        base = (uint32_t)__builtin_amdgcn_readlane((int)base, (int)leader);
        if ((uint64_t)base + nidle >= p.n) exhausted = true;
      }
      if (!active && gbase < groups * kWideLanes) {
        const uint32_t k = base + (uint32_t)__popcll(idle & ((1ull << gbase) - 1ull));
        const uint32_t r = k < p.n ? claimed_ray(p, k) : 0u;
        if (k < p.n && r >= p.n_rays) {
          if (j == 0) {
            atomicOr(p.error, kErrRange);
            if (p.host_err) *reinterpret_cast<volatile uint32_t*>(p.host_err) = 1u;
          }
        } else if (k < p.n) {
          active = true;
          local_id = r;
          const uint4* rq = reinterpret_cast<const uint4*>(p.rays + r);
          const uint4 r0 = rq[0], r1 = rq[1], r2 = rq[2];
          ro = mk3(__uint_as_float(r0.x), __uint_as_float(r0.y), __uint_as_float(r0.z));
          rtmin = __uint_as_float(r0.w);
          rd = mk3(__uint_as_float(r1.x), __uint_as_float(r1.y), __uint_as_float(r1.z));
          rtmax = __uint_as_float(r1.w);
          rflags = r2.x;
          ridir = calc_idir(rd);
          ray_ok = slab_inputs_ok(ro, rd, ridir, rtmin, rtmax);
          min_thit = rtmax;
          min_thit_obj = 0.f;
          closest_leaf = kNoSlot;
          closest_inst = kNoSlot;
          cur_inst = kNoSlot;
          n_rec = n_nodes = fetch_bytes = n_any = 0;
          max_level = 1;
          da = db = 0;
          gs = Groups{0, 0, 0};
          depth = 0;
          phase2 = false;
          err = 0;
          has_e = false;
          if (tlas + 64 > bytes) {
            err |= kErrRange;
          } else {
            emit(tlas, 64, RTX_TX_BVH_STRUCTURE, 0);
            const uint64_t root = tlas + ((uint64_t)tl_h0.x | ((uint64_t)tl_h0.y << 32));
            const F3 lo = mk3(__uint_as_float(tl_h0.z), __uint_as_float(tl_h0.w), __uint_as_float(tl_h1.x));
            const F3 hi = mk3(__uint_as_float(tl_h1.y), __uint_as_float(tl_h1.z), __uint_as_float(tl_h1.w));
            float th;
            if (ray_box(lo, hi, ridir, ro, rtmin, rtmax, th)) {
              if ((root & 63) || root + 64 > bytes) {
                err |= kErrRange;
              } else {
                const uint32_t rs = (uint32_t)(root >> 6);
                push(make_entry(rs, kFlTop, 1, 0), goes_current(rs));
              }
            }
          }
        }
      }
    }
    if (__ballot(active) == 0) {
      if (exhausted) break;
      continue;
    }

    // ---- pop the group's next entry, or complete the ray ---------------------
    if (active && has_e && err != 0) has_e = false;
    if (active && !has_e) {
      if (err == 0 && pop_next()) {
        has_e = true;
      } else {
        pending = true;
        active = false;
      }
    }
    const bool step = has_e && err == 0;
    const uint32_t slot = e_slot(e);
    const uint32_t flags = e_flags(e);
    const uint32_t level = e_level(e);
    const uint64_t off = (uint64_t)slot << 6;
    bool inner = false;
    if (step) {
      has_e = false;
      if (MODE == 1 && !(flags & kFlTop) && e_inst(e, tlas_slot()) != cur_inst) load_instance(e_inst(e, tlas_slot()));
      if (err != 0) {
        // an instance reload out of the arena completes the ray next iteration
      } else if (!(flags & kFlLeaf)) {
        inner = true;
      } else if (flags & kFlTop) {
        // ---- instance leaf: the BLAS root is the group's next entry ----------
        if (off + 128 > bytes) {
          err |= kErrRange;
        } else {
          const uint4* q4 = reinterpret_cast<const uint4*>(A + off + 16);
          const uint4 a = q4[0], b = q4[1], c = q4[2], d = q4[3];
          const float m[12] = {__uint_as_float(a.x), __uint_as_float(a.y), __uint_as_float(a.z), __uint_as_float(a.w),
                               __uint_as_float(b.x), __uint_as_float(b.y), __uint_as_float(b.z), __uint_as_float(b.w),
                               __uint_as_float(c.x), __uint_as_float(c.y), __uint_as_float(c.z), __uint_as_float(c.w)};
          const uint64_t bvh = (uint64_t)d.x | ((uint64_t)d.y << 32);
          emit(off, 128, RTX_TX_BVH_INSTANCE_LEAF, level);
          n_nodes++;
          const uint64_t blas = off + bvh;
          if ((blas & 63) || blas + 64 > bytes) {
            err |= kErrRange;
          } else {
            const uint2 ro2 = *reinterpret_cast<const uint2*>(A + blas);
            emit(blas, 64, RTX_TX_BVH_STRUCTURE, level);
            cur = transform_ray(m, ro, rd, rtmin, rtmax);
            cur_ok = slab_inputs_ok(cur.o, cur.d, cur.idir, cur.tmin, cur.tmax);
            cur_inst = slot;
            uint32_t irel = 0;
            if (MODE == 1 && !inst_rel_of(slot, tlas_slot(), irel)) err |= kErrInstSlot;
            const uint64_t root = blas + ((uint64_t)ro2.x | ((uint64_t)ro2.y << 32));
            if ((root & 63) || root + 64 > bytes) {
              err |= kErrRange;
            } else {
              if (level > max_level) max_level = level;
              const bool to_a = MODE == 0 || (!phase2 && (first_bits(slot) & 1u));
              // the root is the next entry when it goes on top of the list the
              // next pop takes (see trace_kernel); otherwise it is pushed
              if (err == 0 && (MODE == 0 || to_a || da == 0)) {
                if (MODE == 1 && !to_a) phase2 = true;
                e = make_entry((uint32_t)(root >> 6), 0u, level, irel);
                has_e = true;
              } else {
                push(make_entry((uint32_t)(root >> 6), 0u, level, irel), to_a);
              }
            }
          }
        }
      } else {
        // ---- primitive leaf ------------------------------------------------
        if (off + 64 > bytes) {
          err |= kErrRange;
        } else {
          emit(off, 8, RTX_TX_BVH_PRIMITIVE_LEAF_DESCRIPTOR, level);
          const Words16 q = load64B(A + off);
          if (((q.w[1] >> 29) & 1u) == 0u) {
            if ((q.w[3] & 0x1ffffu) != 0u) err |= kErrType;
            const F3 v0 = mk3(f_of(q, 4), f_of(q, 5), f_of(q, 6));
            const F3 v1 = mk3(f_of(q, 7), f_of(q, 8), f_of(q, 9));
            const F3 v2 = mk3(f_of(q, 10), f_of(q, 11), f_of(q, 12));
            float th = 0.f;
            const bool h = mt_test(v0, v1, v2, cur.o, cur.d, th);
            const float wt = th / cur.tmult;
            bool accept;
            if (MODE == 0) {
              accept = h && rtmin <= wt && wt <= rtmax;
              if (accept && (rflags & RTX_RAY_FLAG_OPAQUE) && wt < min_thit) min_thit = th / cur.tmult;
            } else {
              accept = h && rtmin <= wt && wt <= rtmax && wt < min_thit;
              if (accept) min_thit = th / cur.tmult;
            }
            if (accept) {
              min_thit_obj = th;
              closest_leaf = slot;
              closest_inst = cur_inst;
              emit(off, 64, RTX_TX_BVH_QUAD_LEAF_HIT, level);
              n_nodes++;
              if (MODE == 0 && !(rflags & RTX_RAY_FLAG_OPAQUE)) n_any++;
              if (rflags & RTX_RAY_FLAG_TERMINATE_ON_FIRST_HIT) {
                da = db = 0;
                gs = Groups{0, 0, 0};
                depth = 0;
              }
            } else {
              emit(off, 64, RTX_TX_BVH_QUAD_LEAF, level);
              n_nodes++;
            }
          } else {
            emit(off, 64, RTX_TX_BVH_PROCEDURAL_LEAF, level);
            n_nodes++;
          }
        }
      }
    }
    if (inner) {
      // ---- internal node: lane j of the group tests child j ------------------
      if (off + 64 > bytes) {
        err |= kErrRange;
      } else {
        const Words16 nd = load64B(A + off);
        // treelet order before the first switch: which children the first treelet owns
        const uint32_t cur_bits = (MODE == 1 && !phase2) ? first_bits(slot) : 0u;
        emit(off, 64, RTX_TX_BVH_INTERNAL_NODE, level);
        n_nodes++;
        const bool top = (flags & kFlTop) != 0;
        const F3 sc = child_scales((int)(int8_t)byte_of(nd, 18), (int)(int8_t)byte_of(nd, 19), (int)(int8_t)byte_of(nd, 20));
        const F3 o = top ? ro : cur.o;
        const F3 idir = top ? ridir : cur.idir;
        const float tscale = top ? 1.0f : cur.tmult;
        const float tmin = rtmin * tscale, tmax = rtmax * tscale, cull = min_thit * tscale;
        const uint32_t info = __builtin_amdgcn_perm(nd.w[6], nd.w[5], sel_hi) & 0x3fu;  // size and type of child j
        const float ox = f_of(nd, 0), oy = f_of(nd, 1), oz = f_of(nd, 2);
        float th;
        bool h;
        if (__ballot(!((top ? ray_ok : cur_ok) && p.ordered_boxes)) == 0) {
          // a bound is a byte q times the scale: q as the low byte of a half is q *
          // 2^-24 exactly, and the FMA takes halves (see trace_kernel)
          auto bound = [](uint32_t q, float scale, float origin) -> float {
            return __builtin_fmaf((float)__builtin_bit_cast(_Float16, (uint16_t)q), scale * 0x1p24f, origin);
          };
          F3 lo, hi;
          lo.x = bound(__builtin_amdgcn_perm(nd.w[8], nd.w[7], sel_lo), sc.x, ox);
          lo.y = bound(__builtin_amdgcn_perm(nd.w[11], nd.w[10], sel_lo), sc.y, oy);
          lo.z = bound(__builtin_amdgcn_perm(nd.w[14], nd.w[13], sel_lo), sc.z, oz);
          hi.x = bound(__builtin_amdgcn_perm(nd.w[9], nd.w[8], sel_hi), sc.x, ox);
          hi.y = bound(__builtin_amdgcn_perm(nd.w[12], nd.w[11], sel_hi), sc.y, oy);
          hi.z = bound(__builtin_amdgcn_perm(nd.w[15], nd.w[14], sel_hi), sc.z, oz);
          h = ray_box_fast(lo, hi, idir, o, tmin, tmax, th);
        } else {
          F3 lo, hi;
          lo.x = __builtin_fmaf((float)byte_at(nd, 28, jj), sc.x, ox);
          lo.y = __builtin_fmaf((float)byte_at(nd, 40, jj), sc.y, oy);
          lo.z = __builtin_fmaf((float)byte_at(nd, 52, jj), sc.z, oz);
          hi.x = __builtin_fmaf((float)byte_at(nd, 34, jj), sc.x, ox);
          hi.y = __builtin_fmaf((float)byte_at(nd, 46, jj), sc.y, oy);
          hi.z = __builtin_fmaf((float)byte_at(nd, 58, jj), sc.z, oz);
          h = ray_box(lo, hi, idir, o, tmin, tmax, th);
        }
        h = h && !(th >= cull) && j < 6u && (info & 3u) != 0u;
        const uint32_t hitmask = (uint32_t)(__ballot(h) >> gbase) & 0x3fu;
        if (hitmask) {
          const uint32_t lvl = level + 1;
          if (lvl > max_level) max_level = lvl;
          const uint32_t inst = top ? 0u : e_inst_rel(e);
          const uint32_t base_flags = top ? kFlTop : 0u;
          if (MODE == 0 && p.regular_nodes) {
            // the hit children as one group, the first internal one the next entry
            const uint32_t n_push = (uint32_t)__popc(hitmask);
            if (depth + n_push > cap) {
              err |= kErrStack;
            } else {
              const uint32_t leaves = (uint32_t)(__ballot(j < 6u && (info >> 2) != 0u) >> gbase) & 0x3fu;
              const uint32_t word = group_word(top, lvl, leaves, 0u);
              const uint32_t first = slot + nd.w[3];
              const uint32_t im = hitmask & ~leaves;
              const uint32_t rest = hitmask & ~(im & (0u - im));
              depth += n_push;
              if (rest) {
                save_group();
                gs.base = first;
                gs.word = word | (rest << 16);
              }
              if (im) {
                e = group_entry(first, word, (uint32_t)__builtin_ctz(im));
                has_e = true;
                depth--;
                if (n_rec > kMaxStepsPerRay) err |= kErrSteps;
              }
            }
          } else {
          // Lane j pushes hit child j itself, at the position the per-lane
          // kernel's push sequence gives it: hit children in slot order (in
          // plain order the first internal one last), a list's pushes failing
          // from the one that would exceed its capacity on.
          uint64_t c = off + (uint64_t)((int64_t)(int32_t)nd.w[3] * 64);
#pragma unroll
          for (int i = 0; i < 5; ++i)
            if ((uint32_t)i < j) c += (uint64_t)(byte_of(nd, 22 + i) & 3u) * 64;
          const uint32_t ctype = j < 6u ? info >> 2 : 0u;
          const bool leaf = ctype != 0;
          const bool mine = j < 6u && ((hitmask >> j) & 1u);
          const bool pushed = mine && !(c & 63) && c + 64 <= bytes;
          const bool to_a = MODE == 0 || ((cur_bits >> j) & 1u);
          const uint32_t m_push = (uint32_t)(__ballot(pushed) >> gbase) & 0x3fu;
          if ((__ballot(mine && top && leaf && ctype != 1u) >> gbase) & 0x3fu) err |= kErrType;
          if (hitmask & ~m_push) err |= kErrRange;  // hit children outside the arena
          const uint32_t below = (1u << j) - 1u;
          uint32_t pos;
          if (MODE == 0) {
            const uint32_t m_int = (uint32_t)(__ballot(pushed && !leaf) >> gbase) & 0x3fu;
            const uint32_t n = (uint32_t)__popc(m_push);
            const uint32_t d = m_int ? (uint32_t)__builtin_ctz(m_int) : 8u;  // deferred child, 8 = none
            const uint32_t rest = m_push & ~(d < 8u ? 1u << d : 0u);
            // groups of one child, the newest group among the older ones first
            save_group();
            gs.word = 0;
            pos = j == d ? n - 1u : (uint32_t)__popc(rest & below);
            const uint32_t fit = min(n, cap - depth);
            if (pushed && pos < fit)
              sta[da + pos] = (uint64_t)(uint32_t)(c >> 6) |
                              ((uint64_t)group_word(top, lvl, leaf ? 1u : 0u, 1u) << 32);
            da += fit;
            depth += fit;
            if (fit < n) err |= kErrStack;
          } else {
            const uint32_t m_a = (uint32_t)(__ballot(pushed && to_a) >> gbase) & 0x3fu;
            const uint32_t m_b = m_push & ~m_a;
            pos = to_a ? da + (uint32_t)__popc(m_a & below) : db + (uint32_t)__popc(m_b & below);
            da = min(cap, da + (uint32_t)__popc(m_a));
            db = min(cap, db + (uint32_t)__popc(m_b));
          }
          const bool fits = MODE == 0 || pos < cap;
          if (MODE == 1 && pushed && fits)
            *(to_a ? sta + pos : stb + pos) =
                make_entry((uint32_t)(c >> 6), base_flags | (leaf ? kFlLeaf : 0u), lvl, inst);
          if ((__ballot(pushed && !fits) >> gbase) & 0x3fu) err |= kErrStack;
          }
        }
      }
    }
  }
  if (pending) write_hit();
}

using TraceFn = void (*)(TraceParams);

template <int MODE, int REC>
TraceFn pick_k(uint32_t lds_stack, uint32_t stage) {
  if (stage == 0) {
    switch (lds_stack) {
      case 4: return trace_kernel<MODE, REC, 4, 0>;
      case 8: return trace_kernel<MODE, REC, 8, 0>;
      case 16: return trace_kernel<MODE, REC, 16, 0>;
      default: return nullptr;
    }
  }
  if constexpr (REC == kRecSlab4) {  // staged kernels use 8-byte entries
    return nullptr;
  } else {
    switch (stage) {
      case 4096: return trace_kernel<MODE, REC, 8, 4096>;
      case 8192: return trace_kernel<MODE, REC, 8, 8192>;
      case 16384: return trace_kernel<MODE, REC, 8, 16384>;
      case 32768: return trace_kernel<MODE, REC, 8, 32768>;
      case 65536: return trace_kernel<MODE, REC, 8, 65536>;
      default: return nullptr;
    }
  }
}

template <int MODE>
TraceFn pick_rec(int records, uint32_t lds_stack, uint32_t stage) {
  switch (records) {
    case kRecNone: return pick_k<MODE, kRecNone>(lds_stack, stage);
    case kRecCsr: return pick_k<MODE, kRecCsr>(lds_stack, stage);
    case kRecSlab: return pick_k<MODE, kRecSlab>(lds_stack, stage);
    case kRecSlab4: return pick_k<MODE, kRecSlab4>(lds_stack, stage);
    default: return nullptr;
  }
}

TraceFn pick_trace(uint32_t mode, int records, uint32_t lds_stack, uint32_t stage) {
  return mode == RTX_MODE_PLAIN ? pick_rec<0>(records, lds_stack, stage) : pick_rec<1>(records, lds_stack, stage);
}

__global__ void report_total_kernel(const uint64_t* total, uint32_t* host) {
  if (threadIdx.x == 0) {
    volatile uint32_t* h = host;
    const uint64_t d = *total;
    h[2] = (uint32_t)d;
    h[3] = (uint32_t)(d >> 32);
  }
}

// ---- slab records -> CSR ----------------------------------------------------
// Three launches: record sums of tiles of kScanTile rays (with the list of rays whose
// records overflowed their slab), the rays' offsets (each workgroup summing the
// tiles before its own; a scan before it for many tiles), and the expansion.  A batch of at most kFinishAlone rays
// takes one launch, whose workgroups sum the counts themselves and expand their
// own 256 rays: six launches and 12 us less than scans, clear, compaction and
// report had for a 32-ray batch (122 -> 110 us).  It reports the overflows it has
// counted itself, for which its workgroups need not wait for each other; a later
// range of a batch, whose report is of all ranges, takes the three launches
// whatever its size.
//
// The expansion reads 128 MB and writes 468 MB for the 28M records of 1.34M rays
// (100 us at this card's rates) but is bound by the address units: each record
// costs a slab load, an owner gather and a 16-byte store whatever the lanes in
// use.  With one output record per lane all lanes are in use: 174 us; eight lanes
// per ray take 240 us, a search for each record's ray among 64 counts took 202 us
// and the separate scans 28 us more.
__global__ __launch_bounds__(kScanBlock) void sum_record_tiles(const uint32_t* counts, uint32_t n, uint32_t slab,
                                                               uint64_t* tile_sums, uint32_t ray_base,
                                                               uint32_t* overflow_list, uint32_t* overflow_count) {
  __shared__ uint64_t smem[4];
  uint64_t sum = 0;
#pragma unroll
  for (uint32_t k = 0; k < kScanItems; ++k) {
    const uint64_t r = (uint64_t)blockIdx.x * kScanTile + k * kScanBlock + threadIdx.x;
    const uint32_t c = r < n ? counts[r] : 0u;
    if (c > slab) overflow_list[atomicAdd(overflow_count, 1u)] = ray_base + (uint32_t)r;
    sum += c;
  }
  uint64_t total;
  block_exclusive_scan(sum, smem, total);
  if (threadIdx.x == 0) tile_sums[blockIdx.x] = total;
}

__device__ __forceinline__ void report_records(const FinishParams& p, uint32_t overflowed, uint64_t total) {
  if (!p.host) return;
  volatile uint32_t* h = p.host;
  h[0] = overflowed;
  h[2] = (uint32_t)total;
  h[3] = (uint32_t)(total >> 32);
}

// The rtx_record of a slab entry.
template <typename E>
__device__ __forceinline__ uint4 record_of(E v, uint32_t shift, uint64_t offset, uint32_t treelet) {
  const uint32_t lo = (uint32_t)v, hw = (uint32_t)((uint64_t)v >> 32);
  const uint32_t type = sizeof(E) == 4 ? lo >> kSlab4TypeShift : hw & 0xffu;
  const uint32_t level = sizeof(E) == 4 ? (lo & ((1u << kSlab4TypeShift) - 1u)) >> shift : hw >> 8;
  const uint32_t size = type == RTX_TX_BVH_INSTANCE_LEAF ? 128u : type == RTX_TX_BVH_PRIMITIVE_LEAF_DESCRIPTOR ? 8u : 64u;
  return make_uint4((uint32_t)offset, (uint32_t)(offset >> 32), treelet, size | (type << 16) | (level << 24));
}

// The first c records of a ray to `out`, by the eight lanes j = 0 .. 7.
template <typename E>
__device__ __forceinline__ void expand_row(const FinishParams& p, uint64_t ray, uint4* out, uint32_t c, uint32_t j) {
  constexpr uint32_t kUnroll = 4;
  static_assert(kSlabFront == 8 * kUnroll, "a pass reads from one of the two arrays");
  for (uint32_t pass = 0; pass < c; pass += kSlabFront) {
    const E* row = slab_place<E>(p.slabs, p.slabs_rest, p.slab, ray, pass) + j;
    E v[kUnroll];
    uint32_t slot[kUnroll], tl[kUnroll];
    uint64_t roff[kUnroll];
#pragma unroll
    for (uint32_t u = 0; u < kUnroll; ++u) v[u] = pass + 8 * u + j < c ? row[8 * u] : (E)0;
#pragma unroll
    for (uint32_t u = 0; u < kUnroll; ++u) {
      slot[u] = sizeof(E) == 4 ? (uint32_t)v[u] & ((1u << p.shift) - 1u) : (uint32_t)v[u];
      // (a ray that no claim listed keeps an older row: never looked up out of range)
      const bool ok = pass + 8 * u + j < c && slot[u] < p.slots;
      tl[u] = p.owner && ok ? p.owner[slot[u]] : RTX_NO_TREELET;
      roff[u] = p.layout_remap && ok ? p.layout_remap[slot[u]] : (uint64_t)slot[u] << 6;
    }
#pragma unroll
    for (uint32_t u = 0; u < kUnroll; ++u) {
      const uint32_t k = pass + 8 * u + j;
      if (k >= c) continue;
      out[k] = record_of(v[u], p.shift, roff[u], tl[u]);
    }
  }
}

// Offsets of a tile's rays.  The workgroups of up to kTilesSummed tiles sum all tiles
// each; more are scanned before (tile_sums then holds the sums before each tile, and
// all tiles' sum behind them).
__global__ __launch_bounds__(kScanBlock) void place_records(FinishParams p) {
  __shared__ uint64_t smem[4];
  const uint32_t tid = threadIdx.x;
  uint64_t n_all, n_before, n_mine;
  if (p.n_tiles > kTilesSummed) {
    n_before = p.tile_sums[blockIdx.x];
    n_all = p.tile_sums[p.n_tiles];
  } else {
    uint64_t all = 0, before = 0;
    for (uint32_t i = tid; i < p.n_tiles; i += kScanBlock) {
      const uint64_t v = p.tile_sums[i];
      all += v;
      before += i < blockIdx.x ? v : 0u;
    }
    block_exclusive_scan(all, smem, n_all);
    block_exclusive_scan(before, smem, n_before);
  }
  const uint64_t base = p.add_base ? p.offsets[0] : 0;
  const uint64_t r = (uint64_t)blockIdx.x * kScanTile + tid * kScanItems;
  uint32_t c[kScanItems], sum = 0;
#pragma unroll
  for (uint32_t k = 0; k < kScanItems; ++k) {
    c[k] = r + k < p.n ? p.counts[r + k] : 0u;
    sum += c[k];
  }
  uint64_t at = base + n_before + block_exclusive_scan(sum, smem, n_mine);
#pragma unroll
  for (uint32_t k = 0; k < kScanItems; ++k) {
    if (r + k < p.n && (r + k > 0 || !p.add_base)) p.offsets[r + k] = at;
    at += c[k];
  }
  if (blockIdx.x == 0 && tid == 0) {
    p.offsets[p.n] = base + n_all;
    report_records(p, *p.overflow_count, base + n_all);
  }
}

// A small batch of one range at once: offsets and records of 256 rays, the
// workgroups all summing the batch's counts.
template <typename E>
__global__ __launch_bounds__(kScanBlock) void finish_records(FinishParams p) {
  __shared__ uint64_t smem[4];
  const uint32_t tid = threadIdx.x, lane = tid & 63u;
  const uint32_t first = blockIdx.x * kScanBlock;  // the workgroup's first ray
  // records of all rays, and of those before the workgroup's
  uint64_t all = 0, before = 0;
  uint32_t over = 0;
#pragma unroll 4
  for (uint32_t i = tid; i < p.n; i += kScanBlock) {
    const uint32_t v = p.counts[i];
    all += v;
    before += i < first ? v : 0u;
    over += v > p.slab ? 1u : 0u;
  }
  uint64_t n_all, n_before, n_over = 0, n_mine;
  block_exclusive_scan(all, smem, n_all);
  block_exclusive_scan(before, smem, n_before);
  block_exclusive_scan(over, smem, n_over);
  const uint32_t r = first + tid;
  const uint32_t cnt = r < p.n ? p.counts[r] : 0u;
  if (cnt > p.slab) p.overflow_list[atomicAdd(p.overflow_count, 1u)] = p.ray_base + r;
  const uint64_t at = n_before + block_exclusive_scan(cnt, smem, n_mine);
  if (r < p.n) p.offsets[r] = at;
  if (blockIdx.x == 0 && tid == 0) {
    p.offsets[p.n] = n_all;
    report_records(p, (uint32_t)n_over, n_all);
  }
  if (n_all > p.capacity) return;  // the caller reports RTX_ERR_TRACE_OVERFLOW
  for (uint32_t i = lane >> 3; i < 64; i += 8) {  // lanes 8g .. 8g + 7: rays g, g + 8, ... of the wave
    const uint32_t c = min((uint32_t)__shfl(cnt, (int)i, 64), p.slab);
    const uint64_t o = (uint64_t)__shfl((uint32_t)at, (int)i, 64) | ((uint64_t)__shfl((uint32_t)(at >> 32), (int)i, 64) << 32);
    expand_row<E>(p, first + (tid & ~63u) + i, reinterpret_cast<uint4*>(p.records) + o, c, lane & 7u);
  }
}

// Waves take chunks of kExpandChunk consecutive records, and find their first ray
// by a 64-way search of the offsets.  Lane f takes record f of a window of 64: its
// ray is the last one that starts at or before f, counted in a bitmap of the rays'
// starts.
constexpr uint32_t kExpandChunk = 1024;
template <typename E>
__global__ __launch_bounds__(kScanBlock) void expand_records(FinishParams p) {
  __shared__ uint64_t starts_of[kScanBlock / 64][kExpandChunk / 64];
  __shared__ int2 row_of[kScanBlock / 64][64];  // a batch's rays in the chunk: first record, ray
  const uint32_t lane = threadIdx.x & 63u, wave = blockIdx.x * (kScanBlock / 64) + (threadIdx.x >> 6);
  uint64_t* starts = starts_of[threadIdx.x >> 6];
  int2* rows = row_of[threadIdx.x >> 6];
  auto wave_sync = []() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  };
  const uint64_t begin = p.offsets[0], end = p.offsets[p.n];
  if (end > p.capacity) return;  // the caller reports RTX_ERR_TRACE_OVERFLOW
  const uint32_t front = slab_front(p.slab), rest = slab_stride(p.slab) - front;
  const uint64_t stride = (uint64_t)gridDim.x * (kScanBlock / 64) * kExpandChunk;
  for (uint64_t f0 = begin + (uint64_t)wave * kExpandChunk; f0 < end; f0 += stride) {
    const uint32_t size = (uint32_t)min((uint64_t)kExpandChunk, end - f0);
    // the last ray whose offset is at most f0, among lo .. lo + len - 1
    uint32_t lo = 0, len = p.n;
    while (len > 1) {
      const uint32_t step = (len + 63) / 64, at = lane * step;
      const bool below = at < len && p.offsets[lo + at] <= f0;
      const uint32_t k = (uint32_t)__popcll(__ballot(below)) - 1u;  // (lane 0 always is)
      lo += k * step;
      len = min(step, len - k * step);
    }
    for (uint32_t r0 = lo; r0 < p.n; r0 += 64) {
      const uint32_t r = min(r0 + lane, p.n - 1);
      const int64_t off = (int64_t)(p.offsets[r] - f0), next = (int64_t)(p.offsets[r + 1] - f0);
      const bool mine = r0 + lane < p.n && off < (int64_t)size;
      const bool some = mine && next > 0 && next > off;  // has records in the chunk
      // (a ray of the chunk starts at most a slab's rows and 2^24 steps before it)
      const uint32_t s = (uint32_t)max(off, (int64_t)0);
      const uint64_t have = __ballot(some);
      if (lane < kExpandChunk / 64) starts[lane] = 0;
      wave_sync();
      if (some) {
        atomicOr(reinterpret_cast<unsigned long long*>(&starts[s >> 6]), 1ull << (s & 63u));
        rows[lanes_below(have)] = make_int2((int)off, (int)(r0 + lane));
      }
      wave_sync();
      if (have) {
        const int first = (int)__builtin_ctzll(have), last = 63 - (int)__builtin_clzll(have);
        const uint32_t b0 = (uint32_t)__builtin_amdgcn_readlane((int)s, first);
        const uint32_t b1 = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)min(next, (int64_t)size), last);
        uint32_t before = 0;  // starts in the words before w
        constexpr uint32_t kUnroll = 4;
        for (uint32_t w = b0 >> 6; w * 64 < b1; w += kUnroll) {
          E v[kUnroll];
          uint32_t slot[kUnroll], tl[kUnroll];
          uint64_t roff[kUnroll];
          bool ok[kUnroll];
#pragma unroll
          for (uint32_t u = 0; u < kUnroll; ++u) {
            const uint64_t m = starts[min(w + u, kExpandChunk / 64 - 1)];
            const uint32_t f = (w + u) * 64 + lane;
            const uint32_t k = before + lanes_below(m) + (uint32_t)((m >> lane) & 1u);
            const int2 row = rows[k ? min(k, 64u) - 1u : 0u];
            const uint32_t j = f - (uint32_t)row.x;
            ok[u] = f >= b0 && f < b1 && j < p.slab;
            const E* q = j < front ? reinterpret_cast<const E*>(p.slabs) + (uint64_t)(uint32_t)row.y * front + j
                                   : reinterpret_cast<const E*>(p.slabs_rest) + (uint64_t)(uint32_t)row.y * rest + (j - front);
            v[u] = ok[u] ? *q : (E)0;
            before += (uint32_t)__popcll(m);
          }
#pragma unroll
          for (uint32_t u = 0; u < kUnroll; ++u) {
            slot[u] = sizeof(E) == 4 ? (uint32_t)v[u] & ((1u << p.shift) - 1u) : (uint32_t)v[u];
            const bool in = ok[u] && slot[u] < p.slots;  // (see expand_row)
            tl[u] = p.owner && in ? p.owner[slot[u]] : RTX_NO_TREELET;
            roff[u] = p.layout_remap && in ? p.layout_remap[slot[u]] : (uint64_t)slot[u] << 6;
          }
#pragma unroll
          for (uint32_t u = 0; u < kUnroll; ++u)
            if (ok[u])
              reinterpret_cast<uint4*>(p.records)[f0 + (w + u) * 64 + lane] = record_of(v[u], p.shift, roff[u], tl[u]);
        }
      }
      if (__ballot(mine) != ~0ull) break;
    }
  }
}

TraceFn pick_batch(uint32_t mode, uint32_t lds_stack) {
  const bool plain = mode == RTX_MODE_PLAIN;
  switch (lds_stack) {
    case 4: return plain ? trace_kernel<0, false, 4, 0, true> : trace_kernel<1, false, 4, 0, true>;
    case 8: return plain ? trace_kernel<0, false, 8, 0, true> : trace_kernel<1, false, 8, 0, true>;
    case 16: return plain ? trace_kernel<0, false, 16, 0, true> : trace_kernel<1, false, 16, 0, true>;
    default: return nullptr;
  }
}

hipError_t launch_fn(TraceFn f, const TraceParams& p, uint32_t grid, uint32_t bs, hipStream_t s) {
  if (!f) return hipErrorInvalidValue;
  TraceParams arg = p;
  void* args[] = {&arg};
  return hipLaunchKernel(reinterpret_cast<const void*>(f), dim3(grid), dim3(bs), args, 0, s);
}

uint32_t blocks_per_cu(TraceFn f, uint32_t bs) {
  int nb = 0;
  if (!f || hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, reinterpret_cast<const void*>(f), (int)bs, 0) !=
                hipSuccess)
    return 0;
  return nb > 0 ? (uint32_t)nb : 0u;
}

__global__ void fill_zero_kernel(uint32_t* dst, uint32_t words) {
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < words; i += gridDim.x * blockDim.x) dst[i] = 0u;
}

}  // namespace

hipError_t launch_trace_batch(const TraceParams& p, uint32_t mode, uint32_t lds_stack, uint32_t grid,
                              hipStream_t s) {
  if (p.n_jobs == 0 || p.n_jobs > kMaxBatchJobs) return hipErrorInvalidValue;
  return launch_fn(pick_batch(mode, lds_stack), p, grid, 256, s);
}

uint32_t trace_batch_blocks_per_cu(uint32_t mode, uint32_t lds_stack) {
  return blocks_per_cu(pick_batch(mode, lds_stack), 256);
}

hipError_t launch_report_total(const uint64_t* total, uint32_t* host, hipStream_t s) {
  hipLaunchKernelGGL(report_total_kernel, dim3(1), dim3(64), 0, s, total, host);
  return hipGetLastError();
}

hipError_t launch_fill_zero(uint32_t* dst, uint32_t words, hipStream_t s) {
  hipLaunchKernelGGL(fill_zero_kernel, dim3(1), dim3(64), 0, s, dst, words);
  return hipGetLastError();
}

uint32_t trace_block_size(uint32_t stage_bytes) { return stage_bytes ? 64u : 256u; }

namespace {
// per-ray counters -> run totals; with no records the per-type counts follow
// from the counters: a internal nodes, b instance leaves, c primitive leaves
// (fetch = 64 + 64a + 192b + 64c, nodes = a + b + c, records = 1 + a + 2b + 2c)
__global__ __launch_bounds__(256) void k_stats_hits(const rtx_hit* hits, uint32_t n, bool derive_types,
                                                    unsigned long long* acc) {
  unsigned long long t[7] = {0, 0, 0, 0, 0, 0, 0}, nh = 0, na = 0, nodes = 0, fb = 0, ab = 0;
  uint32_t mx_nodes = 0, mx_level = 0;
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    const rtx_hit& h = hits[i];
    nh += h.hit;
    na += h.n_any_hits;
    nodes += h.n_nodes;
    fb += h.fetch_bytes;
    ab += h.accessed_bytes;
    mx_nodes = max(mx_nodes, h.n_nodes);
    mx_level = max(mx_level, h.max_level);
    if (derive_types && h.n_records) {
      const uint32_t b = ((h.fetch_bytes >> 6) - 1u - h.n_nodes) >> 1;
      const uint32_t c = h.n_records - 1u - h.n_nodes - b;
      const uint32_t a = h.n_nodes - b - c;
      t[RTX_TX_BVH_STRUCTURE] += 1u + b;
      t[RTX_TX_BVH_INTERNAL_NODE] += a;
      t[RTX_TX_BVH_INSTANCE_LEAF] += b;
      t[RTX_TX_BVH_PRIMITIVE_LEAF_DESCRIPTOR] += c;
      t[RTX_TX_BVH_QUAD_LEAF] += c;
    }
  }
  const unsigned long long v[14] = {t[0], t[1], t[2], t[3], t[4], t[5], t[6], nh, na, nodes, 0, 0, fb, ab};
  for (int k = 0; k < 14; ++k) {
    if (k == 10 || k == 11) continue;
    unsigned long long x = v[k];
    for (int o = 32; o > 0; o >>= 1) x += __shfl_xor(x, o, 64);
    if ((threadIdx.x & 63u) == 0 && x) atomicAdd(&acc[k], x);
  }
  for (int o = 32; o > 0; o >>= 1) {
    mx_nodes = max(mx_nodes, (uint32_t)__shfl_xor(mx_nodes, o, 64));
    mx_level = max(mx_level, (uint32_t)__shfl_xor(mx_level, o, 64));
  }
  if ((threadIdx.x & 63u) == 0) {
    atomicMax(&acc[10], (unsigned long long)mx_nodes);
    atomicMax(&acc[11], (unsigned long long)mx_level);
  }
}

__global__ __launch_bounds__(256) void k_stats_records(const rtx_record* rec, uint64_t n, unsigned long long* acc) {
  unsigned long long t[7] = {0, 0, 0, 0, 0, 0, 0};
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x) {
    const uint32_t ty = rec[i].type;
    if (ty < 7) t[ty]++;
  }
  for (int k = 0; k < 7; ++k) {
    unsigned long long x = t[k];
    for (int o = 32; o > 0; o >>= 1) x += __shfl_xor(x, o, 64);
    if ((threadIdx.x & 63u) == 0 && x) atomicAdd(&acc[k], x);
  }
}
}  // namespace

hipError_t launch_trace_stats(const rtx_hit* hits, uint32_t n, const rtx_record* records, uint64_t n_records,
                              unsigned long long* acc, hipStream_t s) {
  const uint32_t g = std::max(1u, std::min<uint32_t>(2048, (n + 255) / 256));
  if (n) hipLaunchKernelGGL(k_stats_hits, dim3(g), dim3(256), 0, s, hits, n, records == nullptr, acc);
  if (records && n_records) {
    const uint32_t gr = (uint32_t)std::min<uint64_t>(4096, (n_records + 255) / 256);
    hipLaunchKernelGGL(k_stats_records, dim3(gr), dim3(256), 0, s, records, n_records, acc);
  }
  return hipGetLastError();
}

hipError_t launch_finish_records(FinishParams p, uint64_t* tile_sums, hipStream_t s) {
  if (p.n == 0 || p.slab == 0) return hipSuccess;
  const uint32_t grid = (p.n + kScanBlock - 1) / kScanBlock;
  if (p.n <= kFinishAlone && !p.add_base) {
    if (p.shift)
      hipLaunchKernelGGL(finish_records<uint32_t>, dim3(grid), dim3(kScanBlock), 0, s, p);
    else
      hipLaunchKernelGGL(finish_records<uint64_t>, dim3(grid), dim3(kScanBlock), 0, s, p);
    return hipGetLastError();
  }
  p.n_tiles = (p.n + kScanTile - 1) / kScanTile;
  p.tile_sums = tile_sums;
  hipLaunchKernelGGL(sum_record_tiles, dim3(p.n_tiles), dim3(kScanBlock), 0, s, p.counts, p.n, p.slab, tile_sums,
                     p.ray_base, p.overflow_list, p.overflow_count);
  if (p.n_tiles > kTilesSummed)
    hipLaunchKernelGGL(scan_sums, dim3(1), dim3(kScanBlock), 0, s, tile_sums, p.n_tiles, tile_sums, p.n_tiles);
  hipLaunchKernelGGL(place_records, dim3(p.n_tiles), dim3(kScanBlock), 0, s, p);
  const uint32_t chunks = std::min<uint32_t>(2048, grid);
  if (p.shift)
    hipLaunchKernelGGL(expand_records<uint32_t>, dim3(chunks), dim3(kScanBlock), 0, s, p);
  else
    hipLaunchKernelGGL(expand_records<uint64_t>, dim3(chunks), dim3(kScanBlock), 0, s, p);
  return hipGetLastError();
}

hipError_t launch_level_pass(const TraceParams& p, uint32_t mode, uint32_t grid, hipStream_t s) {
  if (!p.lm_table || !p.lm_list || p.lm_cap < 2 || (p.lm_cap & (p.lm_cap - 1))) return hipErrorInvalidValue;
  TraceFn f = mode == RTX_MODE_PLAIN ? trace_kernel<0, kRecNone, 8, 0, false, true>
                                     : trace_kernel<1, kRecNone, 8, 0, false, true>;
  return launch_fn(f, p, grid, 256, s);
}

namespace {
typedef void (*WideFn)(TraceParams, uint32_t, uint32_t);
WideFn pick_wide(uint32_t mode, bool records) {
  if (mode == RTX_MODE_PLAIN) return records ? trace_wide<0, true> : trace_wide<0, false>;
  return records ? trace_wide<1, true> : trace_wide<1, false>;
}
uint32_t wide_lds_bytes(uint32_t mode, uint32_t groups) {
  return kWideBlock / 64 * groups * (mode == RTX_MODE_PLAIN ? 1u : 2u) * kWideCap * (uint32_t)sizeof(uint64_t);
}
}  // namespace

hipError_t launch_trace_wide(const TraceParams& p, uint32_t mode, bool records, uint32_t cap, uint32_t grid,
                             uint32_t groups, hipStream_t s) {
  if (cap > kWideCap || groups < 1 || groups > 64 / kWideLanes) return hipErrorInvalidValue;
  hipLaunchKernelGGL(pick_wide(mode, records), dim3(grid), dim3(kWideBlock), wide_lds_bytes(mode, groups), s, p, cap,
                     groups);
  return hipGetLastError();
}

uint32_t trace_wide_blocks_per_cu(uint32_t mode, bool records, uint32_t groups) {
  int nb = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, reinterpret_cast<const void*>(pick_wide(mode, records)),
                                                   (int)kWideBlock, wide_lds_bytes(mode, groups)) != hipSuccess)
    return 0;
  return nb > 0 ? (uint32_t)nb : 0u;
}

hipError_t launch_trace(const TraceParams& p, uint32_t mode, int records, uint32_t lds_stack, uint32_t stage_bytes,
                        uint32_t grid, hipStream_t s) {
  return launch_fn(pick_trace(mode, records, lds_stack, stage_bytes), p, grid, trace_block_size(stage_bytes), s);
}

uint32_t trace_blocks_per_cu(uint32_t mode, int records, uint32_t lds_stack, uint32_t stage_bytes) {
  return blocks_per_cu(pick_trace(mode, records, lds_stack, stage_bytes), trace_block_size(stage_bytes));
}

hipError_t launch_scan_records(const rtx_hit* hits, uint32_t n, uint64_t* offsets, uint64_t* tile_sums, hipStream_t s) {
  const uint32_t tiles = (n + kScanTile - 1) / kScanTile;
  if (tiles > 0) {
    hipLaunchKernelGGL(scan_tiles, dim3(tiles), dim3(kScanBlock), 0, s, hits, n, offsets, tile_sums);
  }
  hipLaunchKernelGGL(scan_sums, dim3(1), dim3(kScanBlock), 0, s, tile_sums, tiles, offsets, n);
  if (tiles > 0) {
    hipLaunchKernelGGL(scan_add, dim3(tiles), dim3(kScanBlock), 0, s, offsets, n, tile_sums);
  }
  return hipGetLastError();
}

}  // namespace rtxk
