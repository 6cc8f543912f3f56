// partition.hip — device treelet partitioner.
//
// Restates createTreelets (vulkan_ray_tracing.cc:823-1470) and
// buildNodeToRootMap (:475-489) for the GPU:
//  * A treelet is the longest breadth-first prefix of its root's subtree whose
//    byte sizes fit the budget (internal node 64, instance leaf 128 plus its
//    BLAS header 64, primitive leaf 64); the root always enters and must fit
//    (:893,962,976).  The first treelet is the TLAS header plus the prefix
//    that starts at the TLAS root with budget-64 bytes left (:846-866).
//  * When the next breadth-first entry does not fit, every entry still queued
//    becomes a pending root (:1132-1211).
//  * A treelet depends only on its root, so all pending roots of one round
//    are formed in parallel, by eight lanes or a wave each, and a root reached
//    twice (a BLAS shared by several instances) is formed once; the reference
//    forms it again with an identical result.
//  * The lanes walk the breadth-first queue in chunks of 8 or 64 entries: an
//    inclusive scan of the entry sizes finds how many fit, the accepted
//    entries append their children in order (exclusive scan of child counts),
//    which is exactly the sequential pop-front / push-back order whatever the
//    chunk.
//  * Forming the treelets visits every reachable node and checks what the
//    structural walk (run_validate) checks; the walk itself runs only on a
//    failure, to report the error it finds first.
//  * Node lists keep first occurrences (:1310-1336); roots are numbered in
//    ascending offset order (:1332); a node belongs to the largest root offset
//    whose list holds it, which is what iterating the ordered root map and
//    overwriting produces (:479-488).
#include <algorithm>
#include <vector>

#include "kernels.h"
#include "layout.h"
#include "partition.h"

namespace rtxk {
namespace {

// queue entry kinds
constexpr uint32_t kTopInternal = 0, kTopLeaf = 1, kBotInternal = 2, kBotLeaf = 3;
// node kinds recorded per slot by the validator
constexpr uint8_t kSlotNone = 0, kSlotHeader = 1, kSlotInternal = 2, kSlotInstance = 3, kSlotPrim = 4;

__device__ __forceinline__ uint64_t qentry(uint32_t slot, uint32_t kind) { return (uint64_t)slot | ((uint64_t)kind << 32); }
__device__ __forceinline__ uint32_t q_slot(uint64_t e) { return (uint32_t)e; }
__device__ __forceinline__ uint32_t q_kind(uint64_t e) { return (uint32_t)(e >> 32); }

template <typename T>
__device__ __forceinline__ T wave_incl_scan(T v, uint32_t lane) {
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    T y = __shfl_up(v, d, 64);
    if (lane >= (uint32_t)d) v += y;
  }
  return v;
}

// [off, off + len) lies in the arena (no overflow for any offset)
__device__ __forceinline__ bool in_arena(uint64_t off, uint64_t len, uint64_t bytes) {
  return off <= bytes && bytes - off >= len;
}

// Running totals of a partition: list entries (also the next free place of the
// raw lists), treelet bytes, error bits, whether some node is in two lists or
// twice in one, and the largest treelet.
struct FormTotals {
  unsigned long long listed, bytes;
  uint32_t error, shared, max_bytes, max_nodes;
};

// Rounds launched between two host synchronisations: round j of a batch reads
// its frontier's size from cnt[j], which round j - 1 counted up, so the host
// waits once per batch (a 1M-triangle scene takes four rounds at 8 KiB).
constexpr uint32_t kRoundBatch = 4;

struct FormParams {
  const uint8_t* A;
  uint64_t bytes;
  uint64_t tlas;
  uint32_t budget;
  uint32_t first;  // the frontier is the TLAS header (one treelet)
  uint32_t round;  // within the batch
  uint32_t n0;     // frontier entries of the batch's first round
  uint32_t base0;  // treelets of all earlier batches
  uint32_t* cnt;   // [kRoundBatch + 1] frontier entries of round j (j > 0)
  uint32_t* nbig;  // [kRoundBatch] entries of round j left to form_large
  const uint64_t* in;
  uint64_t* out;
  uint32_t* big;  // their frontier indices
  uint32_t* root_flag;
  uint32_t* owner_root1;
  uint8_t* kind;
  uint32_t* raw_list;
  uint64_t raw_cap;
  uint4* desc;  // per treelet: root slot, place and length of its raw list, bytes
  FormTotals* tot;
  // form_large's queues when they do not fit in LDS, queue_bytes per workgroup
  uint8_t* scratch;
  uint64_t queue_bytes;
  uint32_t qcap, lcap;
};

__device__ __forceinline__ uint32_t frontier_count(const FormParams& p) { return p.round ? p.cnt[p.round] : p.n0; }
// index of the round's first treelet
__device__ __forceinline__ uint32_t treelet_base(const FormParams& p) {
  uint32_t b = p.base0;
  for (uint32_t j = 0; j < p.round; ++j) b += j ? p.cnt[j] : p.n0;
  return b;
}

__device__ __forceinline__ uint8_t slot_kind(uint32_t qkind) {
  return qkind == kTopLeaf ? kSlotInstance : qkind == kBotLeaf ? kSlotPrim : kSlotInternal;
}

// Child offset and the six size/type bytes (22..27) of the internal node at off.
struct NodeKids {
  uint64_t first;
  uint32_t lo, hi;  // info bytes of children 0-3, 4-5
  __device__ __forceinline__ uint32_t info(int i) const { return ((i < 4 ? lo >> (8 * i) : hi >> (8 * (i - 4)))) & 0x3fu; }
};
__device__ __forceinline__ NodeKids load_kids(const uint8_t* A, uint64_t off) {
  const uint4 a = *reinterpret_cast<const uint4*>(A + off);
  const uint4 b = *reinterpret_cast<const uint4*>(A + off + 16);
  NodeKids k;
  k.first = off + (uint64_t)((int64_t)(int32_t)a.w * 64);
  k.lo = __builtin_amdgcn_alignbyte(b.z, b.y, 2);
  k.hi = b.z >> 16;
  return k;
}

// The structural walk's checks of one internal node's children; counts them.
__device__ __forceinline__ uint32_t check_kids(const NodeKids& n, uint32_t kind, uint64_t bytes, uint32_t& count) {
  uint32_t err = 0;
  uint64_t c = n.first;
  count = 0;
#pragma unroll
  for (int i = 0; i < 6; ++i) {
    const uint32_t info = n.info(i), size = info & 3u, type = info >> 2;
    if (size == 0) continue;
    count++;
    if (!in_arena(c, (uint64_t)size * 64, bytes)) err |= kErrRange;
    if (kind == kTopInternal ? (type > 1u || (type == 1u && size != 2u)) : type == 1u) err |= kErrType;
    c += (uint64_t)size * 64;
  }
  return err;
}

template <typename F>
__device__ __forceinline__ void each_kid(const NodeKids& n, uint32_t kind, F&& f) {
  uint32_t slot = (uint32_t)(n.first >> 6);
#pragma unroll
  for (int i = 0; i < 6; ++i) {
    const uint32_t info = n.info(i), size = info & 3u;
    if (size == 0) continue;
    f(slot, kind + (info >> 2 ? 1u : 0u));  // the leaf kind follows the internal one
    slot += size;
  }
}
static_assert(kTopLeaf == kTopInternal + 1 && kBotLeaf == kBotInternal + 1, "each_kid");

__device__ __forceinline__ void wave_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// ---- small treelets: eight lanes each, 32 per workgroup ----------------------
// Most treelets are small (5.5 nodes on average on the 1M-triangle scene at 8
// KiB: what a BLAS's first treelet leaves over), so a wave per treelet idles
// 58 of its 64 lanes, and the time was its chain of queue writes, device-scope
// fences and four atomics on shared counters.  Here eight treelets share a
// wave, their queues stay in LDS, and a workgroup's 32 treelets reserve their
// list, frontier and statistics with one atomic each.  A treelet with an
// instance leaf, or whose queue outgrows kSmallQueue, is left to form_large.
// On the 1M-triangle scene at 8 KiB (253,071 treelets) forming them took 12.3
// ms with a wave each and takes 0.44 ms; bound now by the dependent reads of a
// treelet (entry, node, its leaves' flags) and the shared counters.
// Frontiers of fewer than kSmallMin entries go to form_large at once: they are
// the scene's few large treelets (TLAS, BLAS roots), which 64 lanes walk
// faster, and a wave each does not fill the chip.  The whole build at 1,024 /
// 2,048 / 16,384: 16 instances of 1,024 triangles 242 / 244 / 386 us (8 KiB),
// 256 instances 500 / 464 / 788, and at 1 KiB 603 / 616 / 748.
constexpr uint32_t kSmallLanes = 8;
constexpr uint32_t kSmallGroups = 256 / kSmallLanes;
constexpr uint32_t kSmallQueue = 128;
constexpr uint32_t kSmallStride = kSmallQueue + kSmallLanes;  // the groups of a wave start in different banks
constexpr uint32_t kSmallMin = 2048;

__global__ __launch_bounds__(256) void form_small(FormParams p) {
  const uint32_t n_in = frontier_count(p);
  if (p.first || n_in < kSmallMin) return;
  __shared__ uint32_t qs[kSmallGroups * kSmallStride];
  __shared__ uint8_t qk[kSmallGroups * kSmallStride];
  __shared__ uint32_t g_list[kSmallGroups], g_pend[kSmallGroups], g_big[kSmallGroups];
  __shared__ unsigned long long list_base;
  __shared__ bool listed;  // the workgroup's lists have their place
  const uint32_t lane = threadIdx.x & 63u, j = threadIdx.x & (kSmallLanes - 1), g = threadIdx.x / kSmallLanes;
  const uint32_t gsh = lane & ~(kSmallLanes - 1);  // the group's first lane in its wave
  uint32_t* Q = qs + g * kSmallStride;
  uint8_t* K = qk + g * kSmallStride;
  const uint32_t base = treelet_base(p);
  const uint32_t room = p.budget / 64;
  uint32_t sum_nodes = 0, max_nodes = 0;  // of the workgroup's treelets (thread 0)
  auto group_any = [&](bool v) -> bool { return ((__ballot(v) >> gsh) & 0xffull) != 0; };
  for (uint32_t b = blockIdx.x; b * kSmallGroups < n_in; b += gridDim.x) {
    const uint32_t idx = b * kSmallGroups + g;
    uint32_t head = 0, tail = 0, err = 0, root_slot = 0;
    bool large = false;
    if (idx < n_in) {
      const uint64_t e = p.in[idx];
      root_slot = q_slot(e);
      large = q_kind(e) == kTopLeaf;
      if (j == 0) {
        Q[0] = q_slot(e);
        K[0] = (uint8_t)q_kind(e);
      }
      tail = 1;
    }
    wave_fence();
    // every entry is 64 bytes here: the budget is a node count
    bool more = tail != 0 && !large;
    while (more) {
      const uint32_t chunk = min(kSmallLanes, tail - head), take = min(chunk, room - head);
      if (take == 0) break;
      uint32_t kind = kBotLeaf, slot = 0, count = 0, bad = 0;
      NodeKids kids{0, 0, 0};
      if (j < take) {
        slot = Q[head + j];
        kind = K[head + j];
        if (kind == kTopInternal || kind == kBotInternal) {
          kids = load_kids(p.A, (uint64_t)slot << 6);
          bad = check_kids(kids, kind, p.bytes, count);
        }
      }
      if (group_any(kind == kTopLeaf)) {
        large = true;
        break;
      }
      if (group_any(bad != 0)) {
        err |= bad;
        break;
      }
      uint32_t incl = count;
#pragma unroll
      for (uint32_t d = 1; d < kSmallLanes; d <<= 1) {
        const uint32_t y = __shfl_up(incl, d, kSmallLanes);
        if (j >= d) incl += y;
      }
      const uint32_t total = __shfl(incl, kSmallLanes - 1, kSmallLanes);
      if (tail + total > kSmallQueue) {
        large = true;
        break;
      }
      uint32_t at = tail + incl - count;
      if (count)
        each_kid(kids, kind, [&](uint32_t s, uint32_t k) {
          Q[at] = s;
          K[at] = (uint8_t)k;
          at++;
        });
      wave_fence();
      head += take;
      tail += total;
      more = take == chunk && head < tail;
    }
    if (err) atomicOr(&p.tot->error, err);
    const bool done = idx < n_in && !large && !group_any(err != 0);
    // entries still queued become roots, each once: the new ones move to the front
    uint32_t pend = 0;
    if (done)
      for (uint32_t k0 = head; k0 < tail; k0 += kSmallLanes) {
        const uint32_t k = k0 + j;
        uint32_t s = 0, kd = 0;
        bool fresh = false;
        if (k < tail) {
          s = Q[k];
          kd = K[k];
          fresh = atomicCAS(&p.root_flag[s], 0u, 1u) == 0u;
        }
        const uint32_t m = (uint32_t)(__ballot(fresh) >> gsh) & 0xffu;
        wave_fence();
        if (fresh) {
          const uint32_t at = head + pend + (uint32_t)__popc(m & ((1u << j) - 1u));
          Q[at] = s;
          K[at] = (uint8_t)kd;
        }
        wave_fence();
        pend += (uint32_t)__popc(m);
      }
    if (j == 0) {
      g_list[g] = done ? head : 0u;
      g_pend[g] = pend;
      g_big[g] = large ? 1u : 0u;
    }
    __syncthreads();
    if (threadIdx.x < 64) {
      // The first wave reserves the workgroup's places (exclusive prefixes per group).
      // Roots are counted into the next frontier only once the lists have theirs: the
      // host looks at the error word after a few rounds, and until then every counted
      // frontier place has to hold an entry.
      const bool in = lane < kSmallGroups;
      const uint32_t nl = in ? g_list[lane] : 0u, np = in ? g_pend[lane] : 0u, nb = in ? g_big[lane] : 0u;
      const uint32_t li = wave_incl_scan<uint32_t>(nl, lane), pi = wave_incl_scan<uint32_t>(np, lane),
                     bi = wave_incl_scan<uint32_t>(nb, lane);
      const uint32_t lt = __shfl(li, 63, 64), pt = __shfl(pi, 63, 64), bt = __shfl(bi, 63, 64);
      uint32_t mx = nl;
      for (int o = 32; o > 0; o >>= 1) mx = max(mx, (uint32_t)__shfl_xor(mx, o, 64));
      uint32_t po = 0, bo = 0;
      if (lane == 0) {
        list_base = lt ? atomicAdd(&p.tot->listed, (unsigned long long)lt) : 0ull;
        sum_nodes += lt;
        max_nodes = max(max_nodes, mx);
        listed = lt == 0 || list_base + lt <= p.raw_cap;
        if (!listed) atomicOr(&p.tot->error, kErrQueue);
        if (pt && listed) po = atomicAdd(&p.cnt[p.round + 1], pt);
        if (bt) bo = atomicAdd(&p.nbig[p.round], bt);
      }
      po = __shfl(po, 0, 64);
      bo = __shfl(bo, 0, 64);
      if (in) {
        g_list[lane] = li - nl;
        g_pend[lane] = po + pi - np;
        g_big[lane] = bo + bi - nb;
      }
    }
    __syncthreads();
    if (large && j == 0) p.big[g_big[g]] = idx;
    if (done && listed) {
      const unsigned long long pos = list_base + g_list[g];
      // Q[0, head) was overwritten by nothing: the roots moved to head and on
      bool twice = false;
      for (uint32_t k = j; k < head; k += kSmallLanes) {
        const uint32_t s = Q[k];
        p.raw_list[pos + k] = s;
        p.kind[s] = slot_kind(K[k]);
        twice |= atomicMax(&p.owner_root1[s], root_slot + 1) != 0u;
      }
      if (twice) atomicOr(&p.tot->shared, 1u);
      if (j == 0) p.desc[base + idx] = make_uint4(root_slot, (uint32_t)pos, head, head * 64u);
      for (uint32_t k = j; k < pend; k += kSmallLanes)
        p.out[g_pend[g] + k] = qentry(Q[head + k], K[head + k]);
    }
    __syncthreads();
  }
  if (threadIdx.x == 0 && sum_nodes) {
    atomicAdd(&p.tot->bytes, (unsigned long long)sum_nodes * 64ull);
    atomicMax(&p.tot->max_nodes, max_nodes);
    atomicMax(&p.tot->max_bytes, max_nodes * 64u);
  }
}

// ---- large treelets: one wave each ---------------------------------------------
// The breadth-first queue and the list are in LDS when qcap entries fit (5
// bytes each; budgets up to 64 KiB), else in global memory.
typedef __attribute__((address_space(3))) uint32_t lds_u32;
typedef __attribute__((address_space(3))) uint8_t lds_u8;
typedef __attribute__((address_space(1))) uint32_t glb_u32;
typedef __attribute__((address_space(1))) uint8_t glb_u8;

template <bool LDS, typename W, typename B>
__device__ __forceinline__ void form_one(const FormParams& p, uint32_t idx, uint32_t base, W* Q, W* L, B* K) {
  const uint32_t lane = threadIdx.x;
  auto fence = [&]() {
    if constexpr (!LDS) __threadfence_block();
    wave_fence();
  };
  uint32_t err = 0, head = 0, tail = 1, nl = 0;
  int64_t remaining = p.budget;
  uint32_t root_slot;
  if (p.first) {
    root_slot = (uint32_t)(p.tlas >> 6);
    const uint64_t top = p.tlas + *reinterpret_cast<const uint64_t*>(p.A + p.tlas);
    if ((top & 63) || !in_arena(top, 64, p.bytes)) err |= kErrRange;
    if (lane == 0) {
      L[0] = root_slot;
      Q[0] = (uint32_t)(top >> 6);
      K[0] = (uint8_t)kTopInternal;
      p.kind[root_slot] = kSlotHeader;
    }
    nl = 1;
    remaining -= 64;
  } else {
    const uint64_t e = p.in[idx];
    root_slot = q_slot(e);
    if (lane == 0) {
      Q[0] = q_slot(e);
      K[0] = (uint8_t)q_kind(e);
    }
  }
  fence();
  bool first_chunk = true;
  while (err == 0) {
    const uint32_t chunk = min(64u, tail - head);
    uint32_t slot = 0, kind = kBotLeaf, sz = 0;
    if (lane < chunk) {
      slot = Q[head + lane];
      kind = K[head + lane];
      sz = kind == kTopLeaf ? 192u : 64u;
    }
    const uint32_t incl = wave_incl_scan<uint32_t>(sz, lane);
    const bool acc = lane < chunk && (int64_t)incl <= remaining;
    const uint32_t count = (uint32_t)__popcll(__ballot(acc));
    if (count == 0) {
      if (first_chunk) err |= kErrBudget;
      break;
    }
    // children and list additions of accepted entries
    uint32_t ladd = 0, nch = 0, header = 0, blas_root = 0;
    NodeKids kids{0, 0, 0};
    if (acc) {
      const uint64_t off = (uint64_t)slot << 6;
      ladd = 1;
      p.kind[slot] = slot_kind(kind);
      if (kind == kTopInternal || kind == kBotInternal) {
        kids = load_kids(p.A, off);
        err |= check_kids(kids, kind, p.bytes, nch);
      } else if (kind == kTopLeaf) {
        const uint64_t h = off + *reinterpret_cast<const uint64_t*>(p.A + off + 64);
        if ((h & 63) || !in_arena(h, 64, p.bytes)) {
          err |= kErrRange;
        } else {
          const uint64_t r = h + *reinterpret_cast<const uint64_t*>(p.A + h);
          if ((r & 63) || !in_arena(r, 64, p.bytes)) err |= kErrRange;
          header = (uint32_t)(h >> 6);
          blas_root = (uint32_t)(r >> 6);
          ladd = 2;
          nch = 1;
        }
      }
    }
    if (__ballot(err != 0)) {
      for (int o = 32; o > 0; o >>= 1) err |= __shfl_xor(err, o, 64);
      break;
    }
    const uint32_t lincl = wave_incl_scan<uint32_t>(ladd, lane);
    const uint32_t cincl = wave_incl_scan<uint32_t>(nch, lane);
    const uint32_t ltot = __shfl(lincl, 63, 64);
    const uint32_t ctot = __shfl(cincl, 63, 64);
    if (nl + ltot > p.lcap || tail + ctot > p.qcap) {
      err |= kErrQueue;
      break;
    }
    if (acc) {
      const uint32_t lp = nl + lincl - ladd;
      uint32_t cp = tail + cincl - nch;
      L[lp] = slot;
      if (kind == kTopLeaf) {
        p.kind[header] = kSlotHeader;
        L[lp + 1] = header;
        Q[cp] = blas_root;
        K[cp] = (uint8_t)kBotInternal;
      } else if (nch) {
        each_kid(kids, kind, [&](uint32_t s, uint32_t k) {
          Q[cp] = s;
          K[cp] = (uint8_t)k;
          cp++;
        });
      }
    }
    fence();
    remaining -= __shfl(incl, (int)count - 1, 64);
    head += count;
    tail += ctot;
    nl += ltot;
    first_chunk = false;
    if (count < chunk || head == tail) break;
  }
  if (err) {
    if (lane == 0) atomicOr(&p.tot->error, err);
    return;
  }
  // publish the node list, owner candidates, descriptor and pending roots
  const uint32_t used = p.budget - (uint32_t)remaining;
  unsigned long long pos = 0;
  if (lane == 0) {
    pos = atomicAdd(&p.tot->listed, (unsigned long long)nl);
    atomicAdd(&p.tot->bytes, (unsigned long long)used);
    atomicMax(&p.tot->max_bytes, used);
    atomicMax(&p.tot->max_nodes, nl);
  }
  pos = __shfl(pos, 0, 64);
  if (pos + nl > p.raw_cap) {
    if (lane == 0) atomicOr(&p.tot->error, kErrQueue);
    return;
  }
  bool twice = false;
  for (uint32_t k = lane; k < nl; k += 64) {
    const uint32_t s = L[k];
    p.raw_list[pos + k] = s;
    twice |= atomicMax(&p.owner_root1[s], root_slot + 1) != 0u;
  }
  if (twice) atomicOr(&p.tot->shared, 1u);
  if (lane == 0) p.desc[base + idx] = make_uint4(root_slot, (uint32_t)pos, nl, used);
  for (uint32_t k0 = head; k0 < tail; k0 += 64) {
    const uint32_t k = k0 + lane;
    uint32_t s = 0;
    bool fresh = false;
    if (k < tail) {
      s = Q[k];
      fresh = atomicCAS(&p.root_flag[s], 0u, 1u) == 0u;
    }
    const uint64_t m = __ballot(fresh);
    uint32_t o = 0;
    if (m) {
      if (lane == 0) o = atomicAdd(&p.cnt[p.round + 1], (uint32_t)__popcll(m));
      o = __shfl(o, 0, 64);
    }
    if (fresh) p.out[o + (uint32_t)__popcll(m & ((1ull << lane) - 1ull))] = qentry(s, K[k]);
  }
}

template <bool LDS>
__global__ __launch_bounds__(64) void form_large(FormParams p) {
  extern __shared__ uint32_t smem[];
  const uint32_t n_in = frontier_count(p);
  const bool all = p.first || n_in < kSmallMin;
  const uint32_t n = all ? n_in : p.nbig[p.round];
  if (blockIdx.x >= n) return;
  const uint32_t base = treelet_base(p);
  for (uint32_t i = blockIdx.x; i < n; i += gridDim.x) {
    const uint32_t idx = all ? i : p.big[i];
    if constexpr (LDS) {
      form_one<true>(p, idx, base, (lds_u32*)smem, (lds_u32*)smem + p.qcap, (lds_u8*)((lds_u32*)smem + p.qcap + p.lcap));
    } else {
      glb_u32* q = (glb_u32*)(p.scratch + (uint64_t)blockIdx.x * p.queue_bytes);
      form_one<false>(p, idx, base, q, q + p.qcap, (glb_u8*)(q + p.qcap + p.lcap));
    }
    wave_fence();
  }
}

// ---- generic exclusive scans ------------------------------------------------
__device__ __forceinline__ uint64_t block_excl(uint64_t v, uint64_t* sm, uint64_t& total) {
  const uint32_t lane = threadIdx.x & 63u, w = threadIdx.x >> 6;
  uint64_t x = wave_incl_scan<uint64_t>(v, lane);
  if (lane == 63) sm[w] = x;
  __syncthreads();
  uint64_t off = 0;
  for (uint32_t k = 0; k < w; ++k) off += sm[k];
  total = sm[0] + sm[1] + sm[2] + sm[3];
  __syncthreads();
  return off + x - v;
}

constexpr uint32_t kTile = 1024;  // 256 threads x 4 items

template <typename In>
__global__ __launch_bounds__(256) void scan_tile_k(In in, uint64_t n, uint64_t* out, uint64_t* sums) {
  __shared__ uint64_t sm[4];
  const uint64_t base = (uint64_t)blockIdx.x * kTile + threadIdx.x * 4;
  uint64_t v[4], s = 0;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    v[k] = base + k < n ? (uint64_t)in(base + k) : 0;
    s += v[k];
  }
  uint64_t tot;
  uint64_t ex = block_excl(s, sm, tot);
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    if (base + k < n) out[base + k] = ex;
    ex += v[k];
  }
  if (threadIdx.x == 0) sums[blockIdx.x] = tot;
}

__global__ __launch_bounds__(256) void scan_sums_k(uint64_t* sums, uint64_t tiles, uint64_t* total_out) {
  __shared__ uint64_t sm[4];
  uint64_t carry = 0;
  for (uint64_t b = 0; b < tiles; b += 256) {
    const uint64_t i = b + threadIdx.x;
    uint64_t v = i < tiles ? sums[i] : 0, tot;
    uint64_t ex = block_excl(v, sm, tot);
    if (i < tiles) sums[i] = carry + ex;
    carry += tot;
  }
  if (threadIdx.x == 0) *total_out = carry;
}

__global__ __launch_bounds__(256) void scan_add_k(uint64_t* out, uint64_t n, const uint64_t* sums) {
  const uint64_t base = (uint64_t)blockIdx.x * kTile + threadIdx.x * 4;
  const uint64_t a = sums[blockIdx.x];
#pragma unroll
  for (int k = 0; k < 4; ++k)
    if (base + k < n) out[base + k] += a;
}

struct FlagIn {
  const uint32_t* f;
  __device__ uint64_t operator()(uint64_t i) const { return f[i] != 0 ? 1u : 0u; }
};
struct U32In {
  const uint32_t* v;
  __device__ uint64_t operator()(uint64_t i) const { return v[i]; }
};

template <typename In>
hipError_t exclusive_scan(In in, uint64_t n, uint64_t* out, uint64_t* sums, uint64_t* total, hipStream_t s) {
  const uint64_t tiles = (n + kTile - 1) / kTile;
  if (tiles) hipLaunchKernelGGL((scan_tile_k<In>), dim3((uint32_t)tiles), dim3(256), 0, s, in, n, out, sums);
  hipLaunchKernelGGL(scan_sums_k, dim3(1), dim3(256), 0, s, sums, tiles, total);
  if (tiles) hipLaunchKernelGGL(scan_add_k, dim3((uint32_t)tiles), dim3(256), 0, s, out, n, sums);
  return hipGetLastError();
}

__global__ void owner_and_roots(uint64_t slots, const uint32_t* root_flag, const uint64_t* rank,
                                const uint32_t* owner_root1, uint32_t* owner, uint64_t* roots) {
  for (uint64_t s = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; s < slots; s += (uint64_t)gridDim.x * blockDim.x) {
    const uint32_t o1 = owner_root1[s];
    owner[s] = o1 ? (uint32_t)rank[o1 - 1] : RTX_NO_TREELET;
    if (root_flag[s]) roots[rank[s]] = s << 6;
  }
}

// ---- finalisation of a tree: every node is in exactly one list ------------------
// A treelet's list is its nodes, its image the same nodes packed, and its bytes
// (64 per node, 192 per instance leaf with its BLAS header) the image's size.
__global__ __launch_bounds__(256) void rank_treelets(const uint4* desc, uint32_t n, const uint64_t* rank,
                                                     uint64_t* roots, uint32_t* list_len, uint32_t* image_bytes,
                                                     uint32_t* desc_of_rank) {
  const uint32_t d = blockIdx.x * 256 + threadIdx.x;
  if (d >= n) return;
  const uint4 ds = desc[d];
  const uint32_t r = (uint32_t)rank[ds.x];
  roots[r] = (uint64_t)ds.x << 6;
  list_len[r] = ds.z;
  image_bytes[r] = ds.w;
  desc_of_rank[r] = d;
}

// Eight lanes per treelet (5.5 nodes on average): list, owners and image in one
// pass over its nodes.  Bound by HBM: a node is read and written once more
// (64 B each way) beside 20 B of list, owner and unit words.  Four lanes copy
// one node, so the eight nodes of a step are four 16-byte loads per lane, all
// in flight together: 94 us for the 1.47M nodes of the 1M-triangle scene, where
// a wave per treelet and a kernel per array took 290 us.
__global__ __launch_bounds__(256) void emit_treelets(const uint4* desc, uint32_t n, const uint32_t* raw,
                                                     const uint32_t* desc_of_rank, const uint8_t* kind,
                                                     const uint64_t* list_offsets, const uint64_t* image_offset,
                                                     const uint8_t* A, uint64_t* list_nodes, uint32_t* owner,
                                                     uint8_t* images, uint32_t* image_slots) {
  const uint32_t j = threadIdx.x & 7u;
  for (uint32_t r = blockIdx.x * 32 + threadIdx.x / 8; r < n; r += gridDim.x * 32) {
    const uint4 ds = desc[desc_of_rank[r]];
    const uint64_t lo = list_offsets[r];
    uint64_t unit = image_offset[r] / 64;
    for (uint32_t k0 = 0; k0 < ds.z; k0 += 8) {
      const uint32_t k = k0 + j;
      const bool in = k < ds.z;
      uint32_t s = 0, units = 0;
      if (in) {
        s = raw[ds.y + k];
        units = kind[s] == kSlotInstance ? 2u : 1u;
      }
      uint32_t incl = units;
#pragma unroll
      for (uint32_t d = 1; d < 8; d <<= 1) {
        const uint32_t y = __shfl_up(incl, d, 8);
        if (j >= d) incl += y;
      }
      const uint64_t at = unit + incl - units;
      if (in) {
        list_nodes[lo + k] = (uint64_t)s << 6;
        owner[s] = r;
        image_slots[at] = s;
        if (units == 2u) image_slots[at + 1] = 0xffffffffu;
      }
      uint4 v[4];
#pragma unroll
      for (uint32_t q = 0; q < 4; ++q) {
        const uint32_t from = 2 * q + (j >> 2);
        const uint32_t src = __shfl(s, (int)from, 8);
        // entries past the list read slot 0 and are not stored
        v[q] = *reinterpret_cast<const uint4*>(A + ((uint64_t)src << 6) + (j & 3u) * 16);
      }
#pragma unroll
      for (uint32_t q = 0; q < 4; ++q) {
        const uint32_t from = 2 * q + (j >> 2);
        const uint32_t src = __shfl(s, (int)from, 8), un = __shfl(units, (int)from, 8);
        const uint64_t place = (unit + __shfl(incl, (int)from, 8) - un) * 64 + (j & 3u) * 16;
        if (un) *reinterpret_cast<uint4*>(images + place) = v[q];
        if (un == 2u)
          *reinterpret_cast<uint4*>(images + place + 64) =
              *reinterpret_cast<const uint4*>(A + ((uint64_t)src << 6) + 64 + (j & 3u) * 16);
      }
      unit += __shfl(incl, 7, 8);
    }
  }
}

// ---- finalisation where nodes are shared ------------------------------------------
// One wave per descriptor: de-duplicated length (first occurrence kept).
__global__ __launch_bounds__(256) void dedupe_count(const uint4* desc, uint32_t n_desc, const uint32_t* raw,
                                                    const uint64_t* rank, uint32_t* dlen, uint32_t* desc_of_rank) {
  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t wave = blockIdx.x * 4 + (threadIdx.x >> 6);
  for (uint32_t d = wave; d < n_desc; d += gridDim.x * 4) {
    const uint4 ds = desc[d];
    const uint32_t* l = raw + ds.y;
    uint32_t kept = 0;
    for (uint32_t j = lane; j < ds.z; j += 64) {
      bool keep = true;
      const uint32_t v = l[j];
      for (uint32_t k = 0; k < j; ++k)
        if (l[k] == v) {
          keep = false;
          break;
        }
      kept += keep ? 1u : 0u;
    }
    for (int o = 32; o > 0; o >>= 1) kept += __shfl_xor(kept, o, 64);
    if (lane == 0) {
      const uint32_t r = (uint32_t)rank[ds.x];
      dlen[r] = kept;
      desc_of_rank[r] = d;
    }
  }
}

__global__ __launch_bounds__(256) void dedupe_copy(const uint4* desc, uint32_t n, const uint32_t* raw,
                                                   const uint32_t* desc_of_rank, const uint64_t* list_offsets,
                                                   uint64_t* list_nodes) {
  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t wave = blockIdx.x * 4 + (threadIdx.x >> 6);
  for (uint32_t r = wave; r < n; r += gridDim.x * 4) {
    const uint4 ds = desc[desc_of_rank[r]];
    const uint32_t* l = raw + ds.y;
    uint64_t out = list_offsets[r];
    for (uint32_t j0 = 0; j0 < ds.z; j0 += 64) {
      const uint32_t j = j0 + lane;
      bool keep = j < ds.z;
      uint32_t v = 0;
      if (keep) {
        v = l[j];
        for (uint32_t k = 0; k < j; ++k)
          if (l[k] == v) {
            keep = false;
            break;
          }
      }
      const uint64_t m = __ballot(keep);
      if (keep) {
        const uint32_t pos = __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
        list_nodes[out + pos] = (uint64_t)v << 6;
      }
      out += (uint64_t)__popcll(m);
    }
  }
}

// ---- structural validation: breadth-first walk with per-slot reference counts
struct ValParams {
  const uint8_t* A;
  uint64_t bytes;
  const uint64_t* in;
  uint32_t n_in;
  uint64_t* out;
  uint32_t* n_out;
  uint32_t* refs;
  uint8_t* kind;
  uint32_t* shared;
  uint32_t* error;
  uint32_t* irregular;  // set when a node has a gap before a child, or a child of another size than its kind's
  uint32_t* unordered;  // set when a valid child box has a lower bound byte above its upper one, or its node a
                        // NaN origin or a scale above 2^103 (the sign-ordered slab test's conditions)
  // tree levels (tree_level_map values): nodes processed in this round are at
  // level round + 1 (the TLAS root at 1), their children and a BLAS root
  // reached through an instance leaf at round + 2; lvl[slot] keeps the first
  // level seen and `inconsistent` is set when a node is reached at another
  uint32_t* lvl;
  uint32_t round;
  uint32_t* inconsistent;
};

__device__ __forceinline__ void level_ref(const ValParams& p, uint64_t off, uint32_t level) {
  const uint32_t prev = atomicCAS(&p.lvl[off >> 6], 0u, level);
  if (prev != 0u && prev != level) atomicOr(p.inconsistent, 1u);
}

__device__ void val_ref(const ValParams& p, uint64_t off, uint8_t k, bool push, uint32_t qkind) {
  const uint32_t s = (uint32_t)(off >> 6);
  const uint32_t old = atomicAdd(&p.refs[s], 1u);
  if (old != 0) {
    atomicOr(p.shared, 1u);
    return;
  }
  p.kind[s] = k;
  if (push) {
    const uint32_t o = atomicAdd(p.n_out, 1u);
    p.out[o] = qentry(s, qkind);
  }
}

__global__ void validate_level(ValParams p) {
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < p.n_in; i += gridDim.x * blockDim.x) {
    const uint64_t e = p.in[i];
    const uint64_t off = (uint64_t)q_slot(e) << 6;
    const uint32_t kind = q_kind(e);
    const uint8_t* nd = p.A + off;
    const int32_t co = *reinterpret_cast<const int32_t*>(nd + 12);
    uint64_t c = off + (uint64_t)((int64_t)co * 64);
    const uint32_t child_level = p.round + 2;
    const float* org = reinterpret_cast<const float*>(nd);
    const int8_t* ex = reinterpret_cast<const int8_t*>(nd + 18);
    if (__builtin_isnan(org[0]) || __builtin_isnan(org[1]) || __builtin_isnan(org[2]) || ex[0] > 111 || ex[1] > 111 ||
        ex[2] > 111)
      atomicOr(p.unordered, 1u);
    bool gap = false;
    for (int k = 0; k < 6; ++k) {
      const uint32_t info = nd[22 + k] & 0x3fu;
      const uint32_t size = info & 3u, type = info >> 2;
      if (size == 0) {
        gap = true;
        continue;
      }
      if (gap || size != (kind == kTopInternal && type != 0 ? 2u : 1u)) atomicOr(p.irregular, 1u);
      // lower x/y/z at bytes 28/40/52 + k, upper at 34/46/58 + k
      if (nd[28 + k] > nd[34 + k] || nd[40 + k] > nd[46 + k] || nd[52 + k] > nd[58 + k]) atomicOr(p.unordered, 1u);
      const uint64_t len = (uint64_t)size * 64;
      if ((c & 63) || !in_arena(c, len, p.bytes)) {
        atomicOr(p.error, kErrRange);
        return;
      }
      level_ref(p, c, child_level);
      if (type == 0) {
        val_ref(p, c, kSlotInternal, true, kind);
      } else if (kind == kTopInternal) {
        if (type != 1 || size != 2) {
          atomicOr(p.error, kErrType);
          return;
        }
        const uint64_t h = c + *reinterpret_cast<const uint64_t*>(p.A + c + 64);
        if ((h & 63) || !in_arena(h, 64, p.bytes)) {
          atomicOr(p.error, kErrRange);
          return;
        }
        const uint64_t r = h + *reinterpret_cast<const uint64_t*>(p.A + h);
        if ((r & 63) || !in_arena(r, 64, p.bytes)) {
          atomicOr(p.error, kErrRange);
          return;
        }
        val_ref(p, c, kSlotInstance, false, 0);
        level_ref(p, r, child_level);  // tree_level_map[botLevelRootAddr] = tree_level_map[leaf_addr]
        const uint32_t hs = (uint32_t)(h >> 6);
        if (atomicAdd(&p.refs[hs], 1u) == 0u) {
          p.kind[hs] = kSlotHeader;
          val_ref(p, r, kSlotInternal, true, kBotInternal);
        } else {
          atomicOr(p.shared, 1u);
        }
      } else {
        if (type == 1) {
          atomicOr(p.error, kErrType);
          return;
        }
        val_ref(p, c, kSlotPrim, false, 0);
      }
      c += len;
    }
  }
}

// ---- cycle check: Kahn's peeling over the graph the walk above counted ------
// refs[s] holds each reachable slot's in-degree from the walk (every reference
// an expanded node made; a BLAS header one per instance leaf, its root one from
// the header).  A round takes the internal nodes whose in-degree reached zero
// and removes their edges in the same order the walk added them; the graph has
// a cycle exactly when some count never reaches zero.
struct KahnParams {
  const uint8_t* A;
  const uint64_t* in;
  uint32_t n_in;
  uint64_t* out;
  uint32_t* n_out;
  uint32_t* refs;
};

__device__ __forceinline__ void kahn_push(const KahnParams& p, uint64_t off, uint32_t kind) {
  const uint32_t o = atomicAdd(p.n_out, 1u);
  p.out[o] = qentry((uint32_t)(off >> 6), kind);
}

__global__ void kahn_level(KahnParams p) {
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < p.n_in; i += gridDim.x * blockDim.x) {
    const uint64_t e = p.in[i];
    const uint64_t off = (uint64_t)q_slot(e) << 6;
    const uint32_t kind = q_kind(e);
    const uint8_t* nd = p.A + off;
    const int32_t co = *reinterpret_cast<const int32_t*>(nd + 12);
    uint64_t c = off + (uint64_t)((int64_t)co * 64);
    for (int k = 0; k < 6; ++k) {
      const uint32_t info = nd[22 + k] & 0x3fu;
      const uint32_t size = info & 3u, type = info >> 2;
      if (size == 0) continue;
      if (type == 0) {
        if (atomicSub(&p.refs[c >> 6], 1u) == 1u) kahn_push(p, c, kind);
      } else if (kind == kTopInternal) {
        atomicSub(&p.refs[c >> 6], 1u);
        const uint64_t h = c + *reinterpret_cast<const uint64_t*>(p.A + c + 64);
        const uint64_t r = h + *reinterpret_cast<const uint64_t*>(p.A + h);
        if (atomicSub(&p.refs[h >> 6], 1u) == 1u && atomicSub(&p.refs[r >> 6], 1u) == 1u) kahn_push(p, r, kBotInternal);
      } else {
        atomicSub(&p.refs[c >> 6], 1u);
      }
      c += (uint64_t)size * 64;
    }
  }
}

__global__ void count_nonzero(const uint32_t* v, uint64_t n, uint32_t* count) {
  uint32_t local = 0;
  for (uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x)
    local += v[i] != 0u ? 1u : 0u;
  if (local) atomicAdd(count, local);
}

template <typename T>
rtx_status dmalloc(T** p, size_t count) {
  *p = nullptr;
  if (count == 0) count = 1;
  if (hipMalloc((void**)p, count * sizeof(T)) != hipSuccess) {
    (void)hipGetLastError();
    *p = nullptr;
    return RTX_ERR_OUT_OF_MEMORY;
  }
  return RTX_OK;
}

struct Scratch {
  std::vector<void*> ptrs;
  ~Scratch() {
    for (void* q : ptrs) hipFree(q);
  }
  template <typename T>
  rtx_status alloc(T** p, size_t count) {
    rtx_status st = dmalloc(p, count);
    if (st == RTX_OK) ptrs.push_back(*p);
    return st;
  }
};

// Offsets of several 256-byte aligned arrays in one allocation.
struct Layout {
  size_t size = 0;
  size_t add(size_t bytes) {
    const size_t at = size;
    size += (bytes + 255) & ~(size_t)255;
    return at;
  }
};

// Device memory that lives as long as the partition.
template <typename T>
rtx_status own_alloc(Partition& p, T** q, size_t count) {
  rtx_status st = dmalloc(q, count);
  if (st == RTX_OK) p.owned.push_back(*q);
  return st;
}

rtx_status map_err(uint32_t bits) {
  if (bits & kErrRange) return RTX_ERR_OFFSET_OUT_OF_ARENA;
  if (bits & kErrType) return RTX_ERR_BAD_NODE_TYPE;
  if (bits & kErrBudget) return RTX_ERR_NODE_LARGER_THAN_BUDGET;
  if (bits & kErrQueue) return RTX_ERR_OUT_OF_MEMORY;
  return bits ? RTX_ERR_HIP : RTX_OK;
}

#define CK(expr)                          \
  do {                                    \
    if ((expr) != hipSuccess) {           \
      (void)hipGetLastError();            \
      return RTX_ERR_HIP;                 \
    }                                     \
  } while (0)
#define CS(expr)                  \
  do {                            \
    rtx_status _s = (expr);       \
    if (_s != RTX_OK) return _s;  \
  } while (0)

// Walks the DAG; fills kind[] and reports whether any node is referenced twice.
rtx_status run_validate(const uint8_t* A, uint64_t bytes, uint64_t tlas, hipStream_t s, Scratch& sc, uint8_t* kind,
                        uint32_t* shared_out, uint64_t* n_nodes, uint32_t* unordered_out = nullptr,
                        SceneCheck* check = nullptr) {
  const uint64_t slots = bytes / 64;
  uint32_t *refs, *lvl;
  uint64_t *qa, *qb;
  uint32_t* ctr;  // [0] n_out, [1] error, [2] shared, [3] unordered, [4] inconsistent, [5] nonzero, [6] irregular
  CS(sc.alloc(&refs, slots));
  CS(sc.alloc(&lvl, slots));
  CS(sc.alloc(&qa, slots));
  CS(sc.alloc(&qb, slots));
  CS(sc.alloc(&ctr, 8));
  CK(hipMemsetAsync(refs, 0, slots * 4, s));
  CK(hipMemsetAsync(lvl, 0, slots * 4, s));
  CK(hipMemsetAsync(kind, 0, slots, s));
  CK(hipMemsetAsync(ctr, 0, 32, s));
  uint64_t hdr[1];
  CK(hipMemcpyAsync(hdr, A + tlas, 8, hipMemcpyDeviceToHost, s));
  CK(hipStreamSynchronize(s));
  const uint64_t root = tlas + hdr[0];
  if ((root & 63) || root > bytes || bytes - root < 64) return RTX_ERR_OFFSET_OUT_OF_ARENA;
  const uint32_t one = 1;
  const uint8_t khdr = kSlotHeader, kint = kSlotInternal;
  CK(hipMemcpyAsync(refs + tlas / 64, &one, 4, hipMemcpyHostToDevice, s));
  CK(hipMemcpyAsync(kind + tlas / 64, &khdr, 1, hipMemcpyHostToDevice, s));
  CK(hipMemcpyAsync(refs + root / 64, &one, 4, hipMemcpyHostToDevice, s));
  CK(hipMemcpyAsync(lvl + root / 64, &one, 4, hipMemcpyHostToDevice, s));  // tree_level_map[topRootAddr] = 1
  CK(hipMemcpyAsync(kind + root / 64, &kint, 1, hipMemcpyHostToDevice, s));
  uint64_t e0 = (root / 64) | ((uint64_t)kTopInternal << 32);
  CK(hipMemcpyAsync(qa, &e0, 8, hipMemcpyHostToDevice, s));
  uint32_t n_in = 1;
  uint64_t total = 2;
  uint32_t round = 0;
  while (n_in > 0) {
    CK(hipMemsetAsync(ctr, 0, 4, s));
    ValParams vp{A, bytes, qa, n_in, qb, ctr, refs, kind, ctr + 2, ctr + 1, ctr + 6, ctr + 3, lvl, round++, ctr + 4};
    uint32_t grid = std::min<uint32_t>(4096, (n_in + 255) / 256);
    hipLaunchKernelGGL(validate_level, dim3(grid), dim3(256), 0, s, vp);
    CK(hipGetLastError());
    uint32_t c[3];
    CK(hipMemcpyAsync(c, ctr, 12, hipMemcpyDeviceToHost, s));
    CK(hipStreamSynchronize(s));
    if (c[1]) return map_err(c[1]);
    total += c[0];
    n_in = c[0];
    std::swap(qa, qb);
  }
  // count every referenced slot (leaves and headers included)
  uint32_t c[7];
  CK(hipMemcpyAsync(c, ctr, 28, hipMemcpyDeviceToHost, s));
  CK(hipStreamSynchronize(s));
  if (shared_out) *shared_out = c[2];
  if (unordered_out) *unordered_out = c[3];
  if (check) {
    check->ordered = c[3] == 0;
    check->regular = c[6] == 0;
    check->level_consistent = c[4] == 0;
    check->max_level = round + 1;  // the last walked nodes are at level `round`, their leaves one below
    check->cyclic = false;
    // A cycle reaches a node at two levels, so only inconsistent scenes are peeled.
    if (!check->level_consistent) {
      uint32_t r0 = 0;
      CK(hipMemcpyAsync(&r0, refs + root / 64, 4, hipMemcpyDeviceToHost, s));
      CK(hipStreamSynchronize(s));
      r0 -= 1;  // the walk's seed reference
      CK(hipMemcpyAsync(refs + root / 64, &r0, 4, hipMemcpyHostToDevice, s));
      const uint32_t zero = 0;
      CK(hipMemcpyAsync(refs + tlas / 64, &zero, 4, hipMemcpyHostToDevice, s));
      n_in = r0 == 0 ? 1u : 0u;  // an edge into the TLAS root closes a cycle
      CK(hipMemcpyAsync(qa, &e0, 8, hipMemcpyHostToDevice, s));
      while (n_in > 0) {
        CK(hipMemsetAsync(ctr, 0, 4, s));
        KahnParams kp{A, qa, n_in, qb, ctr, refs};
        uint32_t grid = std::min<uint32_t>(4096, (n_in + 255) / 256);
        hipLaunchKernelGGL(kahn_level, dim3(grid), dim3(256), 0, s, kp);
        CK(hipGetLastError());
        CK(hipMemcpyAsync(&n_in, ctr, 4, hipMemcpyDeviceToHost, s));
        CK(hipStreamSynchronize(s));
        std::swap(qa, qb);
      }
      const uint32_t g = (uint32_t)std::max<uint64_t>(1, std::min<uint64_t>(4096, (slots + 255) / 256));
      hipLaunchKernelGGL(count_nonzero, dim3(g), dim3(256), 0, s, refs, slots, ctr + 5);
      CK(hipGetLastError());
      uint32_t left = 0;
      CK(hipMemcpyAsync(&left, ctr + 5, 4, hipMemcpyDeviceToHost, s));
      CK(hipStreamSynchronize(s));
      check->cyclic = left != 0;
    }
  }
  if (n_nodes) {
    std::vector<uint8_t> k(slots);
    CK(hipMemcpyAsync(k.data(), kind, slots, hipMemcpyDeviceToHost, s));
    CK(hipStreamSynchronize(s));
    uint64_t cnt = 0;
    for (uint8_t v : k) cnt += v != kSlotNone;
    *n_nodes = cnt;
  }
  (void)total;
  return RTX_OK;
}

// ---- treelet-contiguous images (LDS staging source) -------------------------
// Image t = the nodes owned by treelet t, in list order; an instance leaf takes
// 128 bytes, every other node 64.  One wave per treelet.
__global__ __launch_bounds__(256) void image_layout(uint32_t n, const uint64_t* lo, const uint64_t* ln,
                                                    const uint32_t* owner, const uint8_t* kind, uint32_t* stage_slot,
                                                    uint32_t* image_bytes) {
  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t wave = blockIdx.x * 4 + (threadIdx.x >> 6);
  for (uint32_t t = wave; t < n; t += gridDim.x * 4) {
    uint32_t pos = 0;
    for (uint64_t j0 = lo[t]; j0 < lo[t + 1]; j0 += 64) {
      const uint64_t j = j0 + lane;
      uint32_t units = 0, s = 0;
      if (j < lo[t + 1]) {
        s = (uint32_t)(ln[j] >> 6);
        if (owner[s] == t) units = kind[s] == kSlotInstance ? 2u : 1u;
      }
      const uint32_t incl = wave_incl_scan<uint32_t>(units, lane);
      if (units) stage_slot[s] = pos + incl - units;
      pos += __shfl(incl, 63, 64);
    }
    if (lane == 0) image_bytes[t] = pos * 64;
  }
}

__global__ __launch_bounds__(256) void image_copy(uint32_t n, const uint64_t* lo, const uint64_t* ln,
                                                  const uint32_t* owner, const uint8_t* kind,
                                                  const uint32_t* stage_slot, const uint64_t* image_offset,
                                                  const uint8_t* A, uint8_t* images, uint32_t* image_slots) {
  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t wave = blockIdx.x * 4 + (threadIdx.x >> 6);
  for (uint32_t t = wave; t < n; t += gridDim.x * 4) {
    uint8_t* img = images + image_offset[t];
    for (uint64_t j = lo[t] + lane; j < lo[t + 1]; j += 64) {
      const uint32_t s = (uint32_t)(ln[j] >> 6);
      if (owner[s] != t) continue;
      const uint32_t units = kind[s] == kSlotInstance ? 2u : 1u;
      const uint4* src = reinterpret_cast<const uint4*>(A + ((uint64_t)s << 6));
      uint4* dst = reinterpret_cast<uint4*>(img + (uint64_t)stage_slot[s] * 64);
      for (uint32_t k = 0; k < 4 * units; ++k) dst[k] = src[k];
      uint32_t* idx = image_slots + image_offset[t] / 64 + stage_slot[s];
      idx[0] = s;
      if (units == 2) idx[1] = 0xffffffffu;
    }
  }
}

}  // namespace

// Children owned by the first treelet, one byte per node slot after the owner
// words: for an internal node bit i is set when child i is in the arena and
// owner[child i] == first; for an instance leaf bit 0 is set when its BLAS
// root is.  Treelet-order traversal tests exactly these ownerships before its
// first treelet switch, so it reads this byte instead of six owner words.
__global__ void first_bits_kernel(const uint8_t* A, uint64_t bytes, const uint8_t* kind, const uint32_t* owner,
                                  uint32_t first, uint64_t slots, uint8_t* out) {
  for (uint64_t sl = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; sl < slots;
       sl += (uint64_t)gridDim.x * blockDim.x) {
    const uint64_t off = sl << 6;
    uint32_t bits = 0;
    if (kind[sl] == kSlotInternal) {
      const uint8_t* nd = A + off;
      uint64_t c = off + (uint64_t)((int64_t)*reinterpret_cast<const int32_t*>(nd + 12) * 64);
      for (int i = 0; i < 6; ++i) {
        const uint32_t size = nd[22 + i] & 3u;
        if (size != 0 && !(c & 63) && c + 64 <= bytes && owner[c >> 6] == first) bits |= 1u << i;
        c += (uint64_t)size * 64;
      }
    } else if (kind[sl] == kSlotInstance && off + 128 <= bytes) {
      const uint64_t h = off + *reinterpret_cast<const uint64_t*>(A + off + 64);
      if (!(h & 63) && h + 64 <= bytes) {
        const uint64_t r = h + *reinterpret_cast<const uint64_t*>(A + h);
        if (!(r & 63) && r + 64 <= bytes && owner[r >> 6] == first) bits = 1u;
      }
    }
    out[sl] = (uint8_t)bits;
  }
}

hipError_t launch_first_bits(const uint8_t* A, uint64_t bytes, hipStream_t s, const uint8_t* kind, Partition& p) {
  const uint64_t slots = bytes / 64;
  hipLaunchKernelGGL(first_bits_kernel, dim3((uint32_t)std::min<uint64_t>(8192, (slots + 255) / 256)), dim3(256), 0, s, A,
                     bytes, kind, p.owner, p.first_treelet, slots, reinterpret_cast<uint8_t*>(p.owner + slots));
  return hipGetLastError();
}

// Images of a partition whose lists and owners are in place (shared nodes, or
// installed by the caller).
rtx_status build_images(const uint8_t* A, uint64_t bytes, hipStream_t s, const uint8_t* kind, Partition& p) {
  const uint64_t slots = bytes / 64;
  CK(launch_first_bits(A, bytes, s, kind, p));
  Scratch sc;
  uint32_t* stage_slot;  // the 64-byte position of a node inside its owner's image
  uint64_t* sums;
  CS(sc.alloc(&stage_slot, slots));
  CS(sc.alloc(&sums, p.n / kTile + 2));
  CS(own_alloc(p, &p.image_bytes, p.n));
  CS(own_alloc(p, &p.image_offset, (size_t)p.n + 1));
  CK(hipMemsetAsync(stage_slot, 0xff, slots * 4, s));
  const uint32_t g = std::min<uint32_t>(4096, (p.n + 3) / 4);
  hipLaunchKernelGGL(image_layout, dim3(g), dim3(256), 0, s, p.n, p.list_offsets, p.list_nodes, p.owner, kind,
                     stage_slot, p.image_bytes);
  CK(hipGetLastError());
  CK(exclusive_scan(U32In{p.image_bytes}, p.n, p.image_offset, sums, p.image_offset + p.n, s));
  uint64_t total = 0;
  CK(hipMemcpyAsync(&total, p.image_offset + p.n, 8, hipMemcpyDeviceToHost, s));
  CK(hipStreamSynchronize(s));
  p.images_total = total;
  CS(own_alloc(p, &p.images, total));
  CS(own_alloc(p, &p.image_slots, total / 64));
  // units no node claims stay "none", so staging never inserts them
  if (total) CK(hipMemsetAsync(p.image_slots, 0xff, total / 64 * 4, s));
  hipLaunchKernelGGL(image_copy, dim3(g), dim3(256), 0, s, p.n, p.list_offsets, p.list_nodes, p.owner, kind,
                     stage_slot, p.image_offset, A, p.images, p.image_slots);
  CK(hipGetLastError());
  CK(hipStreamSynchronize(s));  // stage_slot is freed on return
  return RTX_OK;
}

// ---- treelet layout: remapBVHToTreeletLayout (vulkan_ray_tracing.cc:1473-1509) ----
// Treelet t's block starts at t * (budget + stride): its root first, then the
// other nodes of its list in order, each advancing by its size (instance leaf
// 128 bytes, every other node 64).  A node listed by several treelets keeps
// the place of the first (lowest index, i.e. lowest root address): each list
// entry proposes (treelet << 32 | place in block) and the slot keeps the
// minimum.  A wave scans one treelet's list.
__global__ __launch_bounds__(256) void layout_propose(uint32_t n, const uint64_t* roots, const uint64_t* lo,
                                                      const uint64_t* ln, const uint8_t* kind,
                                                      unsigned long long* key) {
  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t wave = blockIdx.x * 4 + (threadIdx.x >> 6);
  for (uint32_t t = wave; t < n; t += gridDim.x * 4) {
    const uint32_t rs = (uint32_t)(roots[t] >> 6);
    // the root sits at the block start; the others follow it
    uint32_t place = kind[rs] == kSlotInstance ? 128u : 64u;
    if (lane == 0) atomicMin(&key[rs], (unsigned long long)t << 32);
    for (uint64_t j0 = lo[t]; j0 < lo[t + 1]; j0 += 64) {
      const uint64_t j = j0 + lane;
      uint32_t sz = 0, s = 0;
      if (j < lo[t + 1]) {
        s = (uint32_t)(ln[j] >> 6);
        if (s != rs) sz = kind[s] == kSlotInstance ? 128u : 64u;
      }
      const uint32_t incl = wave_incl_scan<uint32_t>(sz, lane);
      if (sz) atomicMin(&key[s], ((unsigned long long)t << 32) | (place + incl - sz));
      place += __shfl(incl, 63, 64);
    }
  }
}

__global__ __launch_bounds__(256) void layout_place(uint64_t slots, const unsigned long long* key, uint64_t block,
                                                    uint64_t* remap, unsigned long long* placed) {
  uint64_t count = 0;
  for (uint64_t s = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; s < slots; s += (uint64_t)gridDim.x * blockDim.x) {
    const unsigned long long k = key[s];
    remap[s] = k == ~0ull ? ~0ull : (k >> 32) * block + (k & 0xffffffffull);
    count += k == ~0ull ? 0u : 1u;
  }
  for (int o = 32; o > 0; o >>= 1) count += __shfl_xor(count, o, 64);
  if ((threadIdx.x & 63u) == 0 && count) atomicAdd(placed, (unsigned long long)count);
}

// metadata[t][j]: place of list entry j relative to the root's place; also
// flags a root that an earlier treelet placed (the reference asserts there)
__global__ __launch_bounds__(256) void layout_metadata_kernel(uint32_t n, uint32_t per, const uint64_t* roots,
                                                              const uint64_t* lo, const uint64_t* ln,
                                                              const unsigned long long* key, const uint64_t* remap,
                                                              int32_t* meta, uint32_t* conflict) {
  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t wave = blockIdx.x * 4 + (threadIdx.x >> 6);
  for (uint32_t t = wave; t < n; t += gridDim.x * 4) {
    const uint32_t rs = (uint32_t)(roots[t] >> 6);
    if (lane == 0 && (uint32_t)(key[rs] >> 32) != t) atomicOr(conflict, 1u);
    const int64_t r = (int64_t)remap[rs];
    const uint64_t len = lo[t + 1] - lo[t];
    for (uint32_t j = lane; j < per; j += 64) {
      int32_t v = -1;
      if (j < len) v = (int32_t)((int64_t)remap[ln[lo[t] + j] >> 6] - r);
      meta[(uint64_t)t * per + j] = v;
    }
  }
}

void partition_free(Partition& p) {
  hipFree(p.layout_remap);
  hipFree(p.layout_metadata);
  for (void* q : p.owned) hipFree(q);
  p = Partition{};
}

rtx_status partition_layout(const uint8_t* A, uint64_t bytes, uint64_t tlas, uint32_t stride, hipStream_t s,
                            Partition& p) {
  if (!p.valid) return RTX_ERR_NO_PARTITION;
  const uint64_t slots = bytes / 64;
  const uint32_t per = p.budget / 64;
  hipFree(p.layout_remap);
  hipFree(p.layout_metadata);
  p.layout_remap = nullptr;
  p.layout_metadata = nullptr;
  Scratch sc;
  uint8_t* kind;
  unsigned long long* key;
  unsigned long long* placed;
  uint32_t* conflict;
  CS(sc.alloc(&kind, slots));
  CS(sc.alloc(&key, slots));
  CS(sc.alloc(&placed, 1));
  CS(sc.alloc(&conflict, 1));
  CS(run_validate(A, bytes, tlas, s, sc, kind, nullptr, nullptr));
  uint64_t* remap;
  int32_t* meta;
  CS(dmalloc(&remap, slots));
  rtx_status st = dmalloc(&meta, (size_t)p.n * per);
  if (st != RTX_OK) {
    hipFree(remap);
    return st;
  }
  auto fail = [&](rtx_status e) {
    hipFree(remap);
    hipFree(meta);
    return e;
  };
  if (hipMemsetAsync(key, 0xff, slots * 8, s) != hipSuccess || hipMemsetAsync(placed, 0, 8, s) != hipSuccess ||
      hipMemsetAsync(conflict, 0, 4, s) != hipSuccess)
    return fail(RTX_ERR_HIP);
  const uint32_t g = std::max(1u, std::min<uint32_t>(4096, (p.n + 3) / 4));
  hipLaunchKernelGGL(layout_propose, dim3(g), dim3(256), 0, s, p.n, p.roots, p.list_offsets, p.list_nodes, kind, key);
  const uint32_t gs = (uint32_t)std::min<uint64_t>(8192, (slots + 255) / 256);
  hipLaunchKernelGGL(layout_place, dim3(std::max(gs, 1u)), dim3(256), 0, s, slots, key,
                     (uint64_t)p.budget + stride, remap, placed);
  hipLaunchKernelGGL(layout_metadata_kernel, dim3(g), dim3(256), 0, s, p.n, per, p.roots, p.list_offsets,
                     p.list_nodes, key, remap, meta, conflict);
  if (hipGetLastError() != hipSuccess) return fail(RTX_ERR_HIP);
  uint32_t bad = 0;
  unsigned long long mapped = 0;
  if (hipMemcpyAsync(&bad, conflict, 4, hipMemcpyDeviceToHost, s) != hipSuccess ||
      hipMemcpyAsync(&mapped, placed, 8, hipMemcpyDeviceToHost, s) != hipSuccess ||
      hipStreamSynchronize(s) != hipSuccess)
    return fail(RTX_ERR_HIP);
  if (bad) return fail(RTX_ERR_UNSUPPORTED);
  p.layout_remap = remap;
  p.layout_metadata = meta;
  p.layout_stride = stride;
  p.layout_mapped = mapped;
  return RTX_OK;
}

// Whether every internal node reachable from the TLAS has, for each child it
// uses, lower bound bytes no greater than the upper ones on all three axes (so
// the child's decoded box has lo <= hi).  False as well when the walk finds a
// malformed arena or cannot allocate its scratch: traversal then keeps the
// compare-select slab tests, and a malformed arena still reports at trace time.
SceneCheck scene_check(const uint8_t* A, uint64_t bytes, uint64_t tlas, hipStream_t s) {
  SceneCheck out;
  Scratch sc;
  uint8_t* kind;
  if (sc.alloc(&kind, bytes / 64) != RTX_OK) return out;
  SceneCheck ck;
  if (run_validate(A, bytes, tlas, s, sc, kind, nullptr, nullptr, nullptr, &ck) != RTX_OK) {
    (void)hipGetLastError();
    (void)hipStreamSynchronize(s);
    return out;
  }
  ck.valid = true;
  return ck;
}

rtx_status partition_validate(const uint8_t* A, uint64_t bytes, uint64_t tlas, hipStream_t s, uint64_t* n_nodes) {
  Scratch sc;
  uint8_t* kind;
  CS(sc.alloc(&kind, bytes / 64));
  SceneCheck ck;
  CS(run_validate(A, bytes, tlas, s, sc, kind, nullptr, n_nodes, nullptr, &ck));
  return ck.cyclic ? RTX_ERR_CYCLE : RTX_OK;
}

rtx_status partition_build(const uint8_t* A, uint64_t bytes, uint64_t tlas, uint32_t budget, hipStream_t s,
                           Partition& out) {
  partition_free(out);
  const uint64_t slots = bytes / 64;
  const uint32_t qcap = (6 * (budget / 64) + 8 + 3) & ~3u;
  const uint32_t lcap = budget / 64 + 4;
  const uint64_t queue_bytes = ((uint64_t)qcap * 5 + (uint64_t)lcap * 4 + 15) & ~15ull;
  const bool lds = queue_bytes <= 48 * 1024;
  uint32_t large_grid = 4096;  // form_large workgroups of one wave
  while (!lds && large_grid > 64 && queue_bytes * large_grid > (256ull << 20)) large_grid /= 2;
  const uint64_t raw_cap = std::min<uint64_t>(0xffffffffull, 3 * slots + 1024);

  // One block of scratch; the words before `zeroed` are cleared together.
  struct Control {
    FormTotals tot;
    uint32_t cnt[kRoundBatch + 1], nbig[kRoundBatch];
  };
  Scratch sc;
  Layout lay;
  const size_t o_ctl = lay.add(sizeof(Control)), o_flag = lay.add(slots * 4), o_owner1 = lay.add(slots * 4),
               o_kind = lay.add(slots), zeroed = lay.size, o_fa = lay.add(slots * 8), o_fb = lay.add(slots * 8),
               o_big = lay.add(slots * 4), o_desc = lay.add(slots * 16), o_raw = lay.add(raw_cap * 4),
               o_rank = lay.add(slots * 8), o_sums = lay.add((slots / kTile + 2) * 8), o_tot = lay.add(16),
               o_len = lay.add(slots * 4), o_dor = lay.add(slots * 4),
               o_queues = lay.add(lds ? 0 : queue_bytes * large_grid);
  uint8_t* mem;
  CS(sc.alloc(&mem, lay.size));
  Control* ctl = reinterpret_cast<Control*>(mem + o_ctl);
  uint32_t* root_flag = reinterpret_cast<uint32_t*>(mem + o_flag);
  uint32_t* owner_root1 = reinterpret_cast<uint32_t*>(mem + o_owner1);
  uint8_t* kind = mem + o_kind;
  uint64_t* fa = reinterpret_cast<uint64_t*>(mem + o_fa);
  uint64_t* fb = reinterpret_cast<uint64_t*>(mem + o_fb);
  uint4* desc = reinterpret_cast<uint4*>(mem + o_desc);
  uint32_t* raw_list = reinterpret_cast<uint32_t*>(mem + o_raw);
  uint64_t* rank = reinterpret_cast<uint64_t*>(mem + o_rank);
  uint64_t* sums = reinterpret_cast<uint64_t*>(mem + o_sums);
  uint64_t* tot = reinterpret_cast<uint64_t*>(mem + o_tot);
  uint32_t* list_len = reinterpret_cast<uint32_t*>(mem + o_len);
  uint32_t* desc_of_rank = reinterpret_cast<uint32_t*>(mem + o_dor);

  CK(hipMemsetAsync(mem, 0, zeroed, s));
  const uint32_t one = 1;
  CK(hipMemcpyAsync(root_flag + tlas / 64, &one, 4, hipMemcpyHostToDevice, s));
  Control h{};
  uint32_t n_in = 1, n = 0;
  bool first = true;
  while (n_in > 0) {
    if (!first) CK(hipMemsetAsync(ctl->cnt, 0, sizeof(Control) - offsetof(Control, cnt), s));
    for (uint32_t j = 0; j < kRoundBatch; ++j) {
      FormParams fp{A,  bytes, tlas, budget, first ? 1u : 0u, j, n_in, n, ctl->cnt, ctl->nbig, fa, fb,
                    reinterpret_cast<uint32_t*>(mem + o_big), root_flag, owner_root1, kind, raw_list, raw_cap, desc,
                    &ctl->tot, mem + o_queues, queue_bytes, qcap, lcap};
      if (!first) hipLaunchKernelGGL(form_small, dim3(2048), dim3(256), 0, s, fp);
      const uint32_t g = first ? 1u : large_grid;
      if (lds)
        hipLaunchKernelGGL(form_large<true>, dim3(g), dim3(64), queue_bytes, s, fp);
      else
        hipLaunchKernelGGL(form_large<false>, dim3(g), dim3(64), 0, s, fp);
      CK(hipGetLastError());
      std::swap(fa, fb);
      first = false;
    }
    CK(hipMemcpyAsync(&h, ctl, sizeof(h), hipMemcpyDeviceToHost, s));
    CK(hipStreamSynchronize(s));
    if (h.tot.error) {
      // a malformed arena reports what its structural walk finds first
      uint8_t* k2;
      CS(sc.alloc(&k2, slots));
      CS(run_validate(A, bytes, tlas, s, sc, k2, nullptr, nullptr));
      return map_err(h.tot.error);
    }
    n += n_in;
    for (uint32_t j = 1; j < kRoundBatch; ++j) n += h.cnt[j];
    n_in = h.cnt[kRoundBatch];
  }

  // dense numbering of roots in ascending offset order
  CK(exclusive_scan(FlagIn{root_flag}, slots, rank, sums, tot, s));
  Partition p;
  p.budget = budget;
  p.n = n;
  const bool shared = h.tot.shared != 0;
  auto give_back = [&](rtx_status st) {
    partition_free(p);
    return st;
  };
#define CKP(expr)                                                \
  do {                                                           \
    if ((expr) != hipSuccess) {                                  \
      (void)hipGetLastError();                                   \
      return give_back(RTX_ERR_HIP);                             \
    }                                                            \
  } while (0)
#define CSP(expr)                                   \
  do {                                              \
    rtx_status _s = (expr);                         \
    if (_s != RTX_OK) return give_back(_s);         \
  } while (0)
  p.summary.n_treelets = n;
  p.summary.budget_bytes = budget;
  p.summary.total_bytes = h.tot.bytes;
  p.summary.max_treelet_bytes = h.tot.max_bytes;
  p.summary.max_treelet_nodes = h.tot.max_nodes;
  uint64_t n_roots = 0, first_rank = 0;
  if (!shared) {
    // a tree: list and image sizes are known, and one pass writes both
    p.n_list = h.tot.listed;
    p.images_total = h.tot.bytes;
    Layout pl;
    const size_t q_owner = pl.add((slots + (slots + 3) / 4) * 4), q_roots = pl.add((uint64_t)n * 8),
                 q_lo = pl.add(((uint64_t)n + 1) * 8), q_ln = pl.add(p.n_list * 8), q_img = pl.add(p.images_total),
                 q_io = pl.add(((uint64_t)n + 1) * 8), q_ib = pl.add((uint64_t)n * 4),
                 q_is = pl.add(p.images_total / 64 * 4);
    uint8_t* pm;
    CSP(own_alloc(p, &pm, pl.size));
    p.owner = reinterpret_cast<uint32_t*>(pm + q_owner);  // owner words, then the first-treelet bytes
    p.roots = reinterpret_cast<uint64_t*>(pm + q_roots);
    p.list_offsets = reinterpret_cast<uint64_t*>(pm + q_lo);
    p.list_nodes = reinterpret_cast<uint64_t*>(pm + q_ln);
    p.images = pm + q_img;
    p.image_offset = reinterpret_cast<uint64_t*>(pm + q_io);
    p.image_bytes = reinterpret_cast<uint32_t*>(pm + q_ib);
    p.image_slots = reinterpret_cast<uint32_t*>(pm + q_is);
    CKP(hipMemsetAsync(p.owner, 0xff, slots * 4, s));
    hipLaunchKernelGGL(rank_treelets, dim3((n + 255) / 256), dim3(256), 0, s, desc, n, rank, p.roots, list_len,
                       p.image_bytes, desc_of_rank);
    CKP(hipGetLastError());
    CKP(exclusive_scan(U32In{list_len}, n, p.list_offsets, sums, p.list_offsets + n, s));
    CKP(exclusive_scan(U32In{p.image_bytes}, n, p.image_offset, sums, p.image_offset + n, s));
    hipLaunchKernelGGL(emit_treelets, dim3(std::min<uint32_t>(8192, (n + 31) / 32)), dim3(256), 0, s, desc, n, raw_list,
                       desc_of_rank, kind, p.list_offsets, p.image_offset, A, p.list_nodes, p.owner, p.images,
                       p.image_slots);
    CKP(hipGetLastError());
  } else {
    CSP(own_alloc(p, &p.owner, slots + (slots + 3) / 4));
    CSP(own_alloc(p, &p.roots, n));
    CSP(own_alloc(p, &p.list_offsets, (size_t)n + 1));
    hipLaunchKernelGGL(owner_and_roots, dim3(2048), dim3(256), 0, s, slots, root_flag, rank, owner_root1, p.owner,
                       p.roots);
    CKP(hipGetLastError());
    const uint32_t g = std::min<uint32_t>(4096, (n + 3) / 4);
    hipLaunchKernelGGL(dedupe_count, dim3(g), dim3(256), 0, s, desc, n, raw_list, rank, list_len, desc_of_rank);
    CKP(hipGetLastError());
    CKP(exclusive_scan(U32In{list_len}, n, p.list_offsets, sums, p.list_offsets + n, s));
    uint64_t n_list = 0;
    std::vector<uint32_t> hl(n);
    CKP(hipMemcpyAsync(&n_list, p.list_offsets + n, 8, hipMemcpyDeviceToHost, s));
    CKP(hipMemcpyAsync(hl.data(), list_len, (size_t)n * 4, hipMemcpyDeviceToHost, s));
    CKP(hipStreamSynchronize(s));
    p.n_list = n_list;
    p.summary.max_treelet_nodes = *std::max_element(hl.begin(), hl.end());
    CSP(own_alloc(p, &p.list_nodes, n_list));
    hipLaunchKernelGGL(dedupe_copy, dim3(g), dim3(256), 0, s, desc, n, raw_list, desc_of_rank, p.list_offsets,
                       p.list_nodes);
    CKP(hipGetLastError());
  }
  p.summary.n_list_entries = p.n_list;
  CKP(hipMemcpyAsync(&n_roots, tot, 8, hipMemcpyDeviceToHost, s));
  CKP(hipMemcpyAsync(&first_rank, rank + tlas / 64, 8, hipMemcpyDeviceToHost, s));
  CKP(hipStreamSynchronize(s));
  if (n_roots != n || n_roots == 0) return give_back(RTX_ERR_HIP);
  p.first_treelet = (uint32_t)first_rank;
  if (shared) {
    CSP(build_images(A, bytes, s, kind, p));
  } else {
    CKP(launch_first_bits(A, bytes, s, kind, p));
    CKP(hipStreamSynchronize(s));
  }
#undef CKP
#undef CSP
  p.valid = true;
  out = p;
  return RTX_OK;
}

rtx_status partition_copy_out(const Partition& p, uint64_t bytes, hipStream_t s, uint64_t* roots, uint64_t* lo,
                              uint64_t* ln, uint32_t* owner) {
  if (!p.valid) return RTX_ERR_NO_PARTITION;
  if (roots) CK(hipMemcpyAsync(roots, p.roots, (size_t)p.n * 8, hipMemcpyDeviceToHost, s));
  if (lo) CK(hipMemcpyAsync(lo, p.list_offsets, ((size_t)p.n + 1) * 8, hipMemcpyDeviceToHost, s));
  if (ln && p.n_list) CK(hipMemcpyAsync(ln, p.list_nodes, p.n_list * 8, hipMemcpyDeviceToHost, s));
  if (owner) CK(hipMemcpyAsync(owner, p.owner, (bytes / 64) * 4, hipMemcpyDeviceToHost, s));
  CK(hipStreamSynchronize(s));
  return RTX_OK;
}

rtx_status partition_install(const uint8_t* A, uint64_t bytes, uint64_t tlas, uint32_t budget, uint32_t n,
                             const uint64_t* roots, const uint64_t* lo, const uint64_t* ln, const uint32_t* owner,
                             hipStream_t s, Partition& out) {
  const uint64_t slots = bytes / 64;
  // host-side consistency checks
  for (uint32_t i = 0; i < n; ++i) {
    if (roots[i] % 64 || roots[i] >= bytes || (i && roots[i] <= roots[i - 1])) return RTX_ERR_INVALID_ARGUMENT;
    if (lo[i + 1] < lo[i]) return RTX_ERR_INVALID_ARGUMENT;
  }
  if (lo[0] != 0) return RTX_ERR_INVALID_ARGUMENT;
  const uint64_t n_list = lo[n];
  for (uint64_t i = 0; i < n_list; ++i)
    if (ln[i] % 64 || ln[i] >= bytes) return RTX_ERR_INVALID_ARGUMENT;
  // Each list must be de-duplicated (VRT:1312-1356 removes repeats): a node
  // listed twice would get two image positions, and image_layout keeps only one.
  {
    std::vector<uint64_t> sorted;
    for (uint32_t i = 0; i < n; ++i) {
      sorted.assign(ln + lo[i], ln + lo[i + 1]);
      std::sort(sorted.begin(), sorted.end());
      if (std::adjacent_find(sorted.begin(), sorted.end()) != sorted.end()) return RTX_ERR_INVALID_ARGUMENT;
    }
  }
  uint32_t ft = RTX_NO_TREELET;
  for (uint32_t i = 0; i < n; ++i)
    if (roots[i] == tlas) ft = i;
  if (ft == RTX_NO_TREELET) return RTX_ERR_INVALID_ARGUMENT;
  for (uint64_t sidx = 0; sidx < slots; ++sidx)
    if (owner[sidx] != RTX_NO_TREELET && owner[sidx] >= n) return RTX_ERR_INVALID_ARGUMENT;
  partition_free(out);
  Scratch sc;
  uint8_t* kind;
  CS(sc.alloc(&kind, slots));
  CS(run_validate(A, bytes, tlas, s, sc, kind, nullptr, nullptr));
  Partition p;
  p.budget = budget;
  p.n = n;
  p.n_list = n_list;
  p.first_treelet = ft;
  CS(own_alloc(p, &p.owner, slots + (slots + 3) / 4));  // owner words, then the first-treelet bytes
  CS(own_alloc(p, &p.roots, n));
  CS(own_alloc(p, &p.list_offsets, (size_t)n + 1));
  CS(own_alloc(p, &p.list_nodes, n_list));
  CK(hipMemcpyAsync(p.owner, owner, slots * 4, hipMemcpyHostToDevice, s));
  CK(hipMemcpyAsync(p.roots, roots, (size_t)n * 8, hipMemcpyHostToDevice, s));
  CK(hipMemcpyAsync(p.list_offsets, lo, ((size_t)n + 1) * 8, hipMemcpyHostToDevice, s));
  if (n_list) CK(hipMemcpyAsync(p.list_nodes, ln, n_list * 8, hipMemcpyHostToDevice, s));
  rtx_treelet_summary sm{};
  sm.n_treelets = n;
  sm.budget_bytes = budget;
  sm.n_list_entries = n_list;
  for (uint32_t i = 0; i < n; ++i) sm.max_treelet_nodes = std::max<uint32_t>(sm.max_treelet_nodes, (uint32_t)(lo[i + 1] - lo[i]));
  p.summary = sm;
  rtx_status st = build_images(A, bytes, s, kind, p);
  if (st != RTX_OK) {
    partition_free(p);
    return st;
  }
  CK(hipStreamSynchronize(s));
  p.valid = true;
  out = p;
  return RTX_OK;
}

}  // namespace rtxk
