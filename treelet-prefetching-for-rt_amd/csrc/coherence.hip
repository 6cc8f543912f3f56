// coherence.hip — the RT unit's ray coherence engine as a claim order.
//
// The reference's engine (src/gpgpu-sim/ray_coherency_engine.cc) hashes each
// ray a warp brings in (:43), pools rays of equal hash in insertion order
// (:46-54), and whenever a packet slot is free moves up to warp_size rays
// from the largest pool into it (:155-175, get_largest_packet :182-193: the
// first maximum in ascending hash order).  For a batch whose rays are all
// present, that schedule is a sort: pool g of size S contributes chunks
// k = 0, 1, ... with S - k * W rays left before each, and always taking the
// largest remaining pool merges those decreasing sequences, so the chunks
// come out ordered by (rays left before the chunk, descending; hash,
// ascending), each chunk holding its pool's next W rays in input order.
//
// Here: a hash per ray (the four functions of :393-470), a stable radix sort
// of the rays by hash, and a stable radix sort of the chunks by rays left: they
// are listed by pool, so equal counts stay in hash order.  The permutation is
// rtx_trace's claim order: rays of one packet start together in one wave.
//
// Every step is a few passes over 4- or 8-byte arrays that fit the last-level
// cache, so what counts is how many there are: only the bits a hash function can
// set are sorted (12 for the grid hashes: two passes), the second sort takes
// chunks, not rays (1.3M rays make some 25,000), and the scratch memory is the
// context's.  1.29M rays: 1,040 us with two full-width sorts of all rays and
// their allocations, 205 us now, most of it the latency of 24 launches.
#include <algorithm>
#include <cmath>

#include "kernels.h"
#include "rtx.h"

namespace rtxk {
namespace {

struct CohParams {
  const rtx_ray* rays;
  uint32_t n;
  uint32_t hash;  // 'f', 'g', 't', 'd'
  uint32_t francois_bits, grid_bits, sphere_bits;
  float two_point_ratio;
  float wmin[3], wmax[3];
};

// hash_comp (:393-402): sign, the top `b` exponent bits and the top `b`
// mantissa bits of the float's pattern
__device__ __forceinline__ uint64_t hash_comp(float x, uint32_t b) {
  const uint32_t mask = 0xffffffffu >> (32 - b);
  const uint32_t o = __float_as_uint(x);
  const uint64_t sign = o >> 31;
  const uint64_t ex = (o >> (31 - b)) & mask;
  const uint64_t mant = (o >> (23 - b)) & mask;
  return (sign << (2 * b)) | (ex << b) | mant;
}

// float -> uint64 as the reference's implicit conversions; a NaN (a world
// axis of zero extent) becomes 0, where the reference's conversion is undefined
__device__ __forceinline__ uint64_t to_u64(float v) { return __builtin_isnan(v) ? 0ull : (uint64_t)v; }

// clamp (vector-math.cc:68-71): std::max(std::min(x, hi), lo)
__device__ __forceinline__ float vm_clamp(float x, float lo, float hi) {
  const float m = hi < x ? hi : x;
  return m < lo ? lo : m;
}

// hash_origin_grid (:423-430)
__device__ __forceinline__ uint64_t hash_grid(const CohParams& c, float ox, float oy, float oz, uint32_t b) {
  const uint32_t g = 1u << b;
  const float gs = (float)g, top = (float)g - 1.f;
  const uint64_t x = to_u64(vm_clamp((ox - c.wmin[0]) / (c.wmax[0] - c.wmin[0]) * gs, 0.f, top));
  const uint64_t y = to_u64(vm_clamp((oy - c.wmin[1]) / (c.wmax[1] - c.wmin[1]) * gs, 0.f, top));
  const uint64_t z = to_u64(vm_clamp((oz - c.wmin[2]) / (c.wmax[2] - c.wmin[2]) * gs, 0.f, top));
  return (x << (2 * b)) | (y << b) | z;
}

// hash_direction_spherical (:408-421)
__device__ __forceinline__ uint64_t hash_sphere(float dx, float dy, float dz, uint32_t b) {
  const float kPi = 3.14159265358979323846f;
  const uint64_t theta = to_u64(acosf(vm_clamp(dz, -1.f, 1.f)) / kPi * 180.f);
  const uint64_t phi = to_u64((atan2f(dy, dx) + kPi) / kPi * 180.f);
  const uint64_t q_theta = theta >> (8 - b);
  const uint64_t q_phi = phi >> (9 - (b + 1));
  return (q_phi << b) | q_theta;
}

__global__ __launch_bounds__(256) void k_ray_hash(CohParams c, uint32_t* keys, uint32_t* hashes_out) {
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < c.n; i += gridDim.x * blockDim.x) {
    const rtx_ray r = c.rays[i];
    const float ox = r.org[0], oy = r.org[1], oz = r.org[2];
    const float dx = r.dir[0], dy = r.dir[1], dz = r.dir[2];
    uint64_t h = 0;
    if (c.hash == 'f') {  // hash_francois (:432-445)
      const uint32_t b = c.francois_bits, cb = 2 * b + 1;
      const uint64_t hd = (hash_comp(dz, b) << (2 * cb)) | (hash_comp(dy, b) << cb) | hash_comp(dx, b);
      const uint64_t ho = (hash_comp(ox, b) << (2 * cb)) | (hash_comp(oy, b) << cb) | hash_comp(oz, b);
      h = ho ^ hd;
    } else if (c.hash == 'g') {  // hash_grid_spherical (:447-456)
      h = hash_grid(c, ox, oy, oz, c.grid_bits) ^ hash_sphere(dx, dy, dz, c.sphere_bits);
    } else if (c.hash == 't') {  // hash_two_point (:462-469)
      const float ex = c.wmax[0] - c.wmin[0], ey = c.wmax[1] - c.wmin[1], ez = c.wmax[2] - c.wmin[2];
      const float mx = ex > ey ? ex : ey;  // std::max(std::max(x, y), z)
      const float ext = mx > ez ? mx : ez;
      const float s = c.two_point_ratio * ext;
      h = hash_grid(c, ox, oy, oz, c.grid_bits) ^ hash_grid(c, ox + s * dx, oy + s * dy, oz + s * dz, c.grid_bits);
    } else {  // hash_direction_only (:471-474)
      h = hash_sphere(dx, dy, dz, c.sphere_bits);
    }
    keys[i] = (uint32_t)h;  // the host keeps every configuration's hash below 2^32
    if (hashes_out) hashes_out[i] = (uint32_t)h;
  }
}

// Upper bound of the bits a configuration's hash can set.
uint32_t hash_bits(const rtx_coherence_config& c) {
  // theta <= 180 and phi <= 360 degrees, shifted by 8 - b each: below 2^b and 2^(b + 1)
  const uint32_t sphere = 2 * c.sphere_bits + 1, grid = 3 * c.grid_bits;
  switch (c.hash) {
    case 'f': return 3 * (2 * c.francois_bits + 1);
    case 'g': return std::max(grid, sphere);
    case 't': return grid;
    default: return sphere;
  }
}

// ---- stable radix sort, one digit of up to 8 bits per pass ---------------------
// A workgroup takes kTile consecutive items, each of its waves a contiguous
// quarter.  k_digit_counts tabulates the digits per workgroup (digit-major),
// k_digit_scan turns each digit's row into exclusive prefixes and a total, and
// k_digit_scatter gives every item its place: digits before, workgroups before,
// waves before, and its rank among the wave's items of its digit (one ballot per
// digit bit).  The item count is a device word, so that a pass over a count the
// host does not know is launched for its upper bound.
constexpr uint32_t kTile = 2048, kWaveItems = kTile / 4, kWaveSteps = kWaveItems / 64;

__global__ __launch_bounds__(256) void k_digit_counts(const uint32_t* keys, const uint32_t* count, uint32_t shift,
                                                      uint32_t bits, uint32_t* table) {
  __shared__ uint32_t hist[256];
  const uint32_t n = *count, b0 = blockIdx.x * kTile;
  hist[threadIdx.x] = 0;
  __syncthreads();
  if (b0 < n) {
    const uint32_t e = min(n - b0, kTile);
    for (uint32_t i = threadIdx.x; i < e; i += 256) atomicAdd(&hist[(keys[b0 + i] >> shift) & ((1u << bits) - 1u)], 1u);
  }
  __syncthreads();
  if (threadIdx.x < 1u << bits) table[(size_t)threadIdx.x * gridDim.x + blockIdx.x] = hist[threadIdx.x];
}

// inclusive sums over a workgroup; sm: a word per wave
__device__ __forceinline__ uint32_t block_incl(uint32_t v, uint32_t* sm) {
  const uint32_t lane = threadIdx.x & 63u, w = threadIdx.x >> 6;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const uint32_t y = __shfl_up(v, d, 64);
    if (lane >= (uint32_t)d) v += y;
  }
  __syncthreads();
  if (lane == 63) sm[w] = v;
  __syncthreads();
  for (uint32_t k = 0; k < w; ++k) v += sm[k];
  return v;
}

__global__ __launch_bounds__(256) void k_digit_scan(uint32_t* table, uint32_t groups, uint32_t* totals) {
  __shared__ uint32_t sm[4];
  __shared__ uint32_t sum;
  uint32_t* row = table + (size_t)blockIdx.x * groups;
  uint32_t carry = 0;
  for (uint32_t b = 0; b < groups; b += 256) {
    const uint32_t i = b + threadIdx.x, v = i < groups ? row[i] : 0u;
    const uint32_t incl = block_incl(v, sm);
    if (i < groups) row[i] = carry + incl - v;
    if (threadIdx.x == 255) sum = incl;
    __syncthreads();
    carry += sum;
  }
  if (threadIdx.x == 0) totals[blockIdx.x] = carry;
}

// vals null: the items' values are their positions
__global__ __launch_bounds__(256) void k_digit_scatter(const uint32_t* keys, const uint32_t* vals, const uint32_t* count,
                                                       uint32_t shift, uint32_t bits, const uint32_t* table,
                                                       const uint32_t* totals, uint32_t* keys_out, uint32_t* vals_out) {
  __shared__ uint32_t place[4][256];
  __shared__ uint32_t sm[4];
  const uint32_t n = *count, b0 = blockIdx.x * kTile;
  if (b0 >= n) return;
  const uint32_t lane = threadIdx.x & 63u, w = threadIdx.x >> 6, mask = (1u << bits) - 1u;
  for (uint32_t k = 0; k < 4; ++k) place[k][threadIdx.x] = 0;
  __syncthreads();
  const uint32_t w0 = b0 + w * kWaveItems;
  const uint32_t we = w0 < n ? min(n - w0, kWaveItems) : 0u;
  // the wave's items, all loads in flight together
  uint32_t key[kWaveSteps], val[kWaveSteps];
#pragma unroll
  for (uint32_t k = 0; k < kWaveSteps; ++k) {
    const uint32_t i = k * 64 + lane;
    key[k] = i < we ? keys[w0 + i] : 0u;
    val[k] = vals ? (i < we ? vals[w0 + i] : 0u) : w0 + i;
  }
#pragma unroll
  for (uint32_t k = 0; k < kWaveSteps; ++k)
    if (k * 64 + lane < we) atomicAdd(&place[w][(key[k] >> shift) & mask], 1u);
  const bool digit = threadIdx.x < 1u << bits;
  const uint32_t tot = digit ? totals[threadIdx.x] : 0u;
  uint32_t at = block_incl(tot, sm) - tot + (digit ? table[(size_t)threadIdx.x * gridDim.x + blockIdx.x] : 0u);
  __syncthreads();
  for (uint32_t k = 0; k < 4; ++k) {
    const uint32_t c = place[k][threadIdx.x];
    place[k][threadIdx.x] = at;
    at += c;
  }
  __syncthreads();
#pragma unroll
  for (uint32_t k = 0; k < kWaveSteps; ++k) {
    const bool in = k * 64 + lane < we;
    const uint32_t d = (key[k] >> shift) & mask;
    uint64_t same = __ballot(in);
    for (uint32_t b = 0; b < bits; ++b) {
      const uint64_t m = __ballot((d >> b) & 1u);
      same &= (d >> b) & 1u ? m : ~m;
    }
    if (in) {
      const uint32_t pos = place[w][d] + (uint32_t)__popcll(same & ((1ull << lane) - 1ull));
      keys_out[pos] = key[k];
      vals_out[pos] = val[k];
      // the digit's last item of this step moves its place on
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
      if ((same >> lane) == 1ull) place[w][d] = pos + 1;
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }
}

// ---- chunks ----------------------------------------------------------------------
// first position with h's value, searching [0, p]
__device__ __forceinline__ uint32_t pool_start(const uint32_t* h, uint32_t p) {
  const uint32_t v = h[p];
  uint32_t lo = 0, hi = p;  // h[hi] == v
  while (lo < hi) {
    const uint32_t mid = (lo + hi) >> 1;
    if (h[mid] == v)
      hi = mid;
    else
      lo = mid + 1;
  }
  return lo;
}

// The chunk starts among 1,024 sorted positions: positions whose distance from
// their pool's start is a multiple of the packet.  Each thread takes four
// consecutive positions; `starts` keeps their pools' starts.
__device__ __forceinline__ uint32_t chunk_flags(const uint32_t* h, uint32_t n, uint32_t packet, uint32_t p0,
                                                uint32_t starts[4]) {
  uint32_t flags = 0;
  for (uint32_t k = 0; k < 4; ++k) {
    const uint32_t p = p0 + k;
    if (p >= n) break;
    starts[k] = k == 0 ? pool_start(h, p) : h[p] == h[p - 1] ? starts[k - 1] : p;
    if ((p - starts[k]) % packet == 0) flags |= 1u << k;
  }
  return flags;
}

__global__ __launch_bounds__(256) void k_chunk_counts(const uint32_t* h, uint32_t n, uint32_t packet, uint32_t* sums) {
  __shared__ uint32_t sm[4];
  uint32_t starts[4];
  const uint32_t f = chunk_flags(h, n, packet, blockIdx.x * 1024 + threadIdx.x * 4, starts);
  const uint32_t incl = block_incl((uint32_t)__popc(f), sm);
  if (threadIdx.x == 255) sums[blockIdx.x] = incl;
}

// exclusive prefixes of `tiles` sums, in place; the total to *total
__global__ __launch_bounds__(1024) void k_scan_sums(uint32_t* sums, uint32_t tiles, uint32_t* total) {
  __shared__ uint32_t sm[16];
  __shared__ uint32_t sum;
  uint32_t carry = 0;
  for (uint32_t b = 0; b < tiles; b += 1024) {
    const uint32_t i = b + threadIdx.x, v = i < tiles ? sums[i] : 0u;
    const uint32_t incl = block_incl(v, sm);
    if (i < tiles) sums[i] = carry + incl - v;
    if (threadIdx.x == 1023) sum = incl;
    __syncthreads();
    carry += sum;
  }
  if (threadIdx.x == 0) *total = carry;
}

// Key of each chunk in pool order: the batch's rays without those left in its
// pool before it, so that the most rays left sort first.
__global__ __launch_bounds__(256) void k_chunk_keys(const uint32_t* h, uint32_t n, uint32_t packet, const uint32_t* sums,
                                                    uint32_t* keys) {
  __shared__ uint32_t sm[4];
  uint32_t starts[4];
  const uint32_t p0 = blockIdx.x * 1024 + threadIdx.x * 4;
  uint32_t f = chunk_flags(h, n, packet, p0, starts);
  const uint32_t own = (uint32_t)__popc(f);
  uint32_t at = sums[blockIdx.x] + block_incl(own, sm) - own;
  // the lanes' searches run together: one round unless packets are below four
  for (; f; f &= f - 1) {
    const uint32_t p = p0 + (uint32_t)__ffs((int)f) - 1u;
    // the pool ends where the value changes (or at n)
    const uint32_t v = h[p];
    uint32_t lo = p, hi = n;
    while (lo + 1 < hi) {
      const uint32_t mid = (lo + hi) >> 1;
      if (h[mid] == v)
        lo = mid;
      else
        hi = mid;
    }
    keys[at++] = n - (hi - p);
  }
}

// rays of sorted chunk c: min(packet, rays left)
__device__ __forceinline__ uint32_t chunk_size(const uint32_t* keys, uint32_t n, uint32_t packet, uint32_t c) {
  return min(packet, n - keys[c]);
}

__global__ __launch_bounds__(256) void k_size_sums(const uint32_t* keys, const uint32_t* count, uint32_t n,
                                                   uint32_t packet, uint32_t* sums) {
  __shared__ uint32_t sm[4];
  const uint32_t c = blockIdx.x * 256 + threadIdx.x;
  const uint32_t incl = block_incl(c < *count ? chunk_size(keys, n, packet, c) : 0u, sm);
  if (threadIdx.x == 255) sums[blockIdx.x] = incl;
}

// place[id] of the sorted chunks: where chunk id's rays begin in the schedule
__global__ __launch_bounds__(256) void k_chunk_places(const uint32_t* keys, const uint32_t* ids, const uint32_t* count,
                                                      uint32_t n, uint32_t packet, const uint32_t* sums,
                                                      uint32_t* place) {
  __shared__ uint32_t sm[4];
  const uint32_t m = *count, c = blockIdx.x * 256 + threadIdx.x;
  if (blockIdx.x * 256 >= m) return;
  const uint32_t sz = c < m ? chunk_size(keys, n, packet, c) : 0u;
  const uint32_t at = sums[blockIdx.x] + block_incl(sz, sm) - sz;
  if (c < m) place[ids[c]] = at;
}

// Every pooled ray to its chunk's place (a thread per ray, so that a packet of
// any size is copied evenly).
__global__ __launch_bounds__(256) void k_copy_chunks(const uint32_t* h, uint32_t n, uint32_t packet,
                                                     const uint32_t* sums, const uint32_t* place, const uint32_t* rays,
                                                     uint32_t* order) {
  __shared__ uint32_t sm[4];
  uint32_t starts[4];
  const uint32_t p0 = blockIdx.x * 1024 + threadIdx.x * 4;
  const uint32_t f = chunk_flags(h, n, packet, p0, starts);
  const uint32_t own = (uint32_t)__popc(f);
  const uint32_t before = sums[blockIdx.x] + block_incl(own, sm) - own;
  for (uint32_t k = 0; k < 4; ++k) {
    const uint32_t p = p0 + k;
    if (p >= n) break;
    const uint32_t id = before + (uint32_t)__popc(f & ((2u << k) - 1u)) - 1u;
    order[place[id] + (p - starts[k]) % packet] = rays[p];
  }
}

__global__ void k_set_count(uint32_t* word, uint32_t n) {
  if (threadIdx.x == 0) *word = n;
}

}  // namespace

size_t coherence_scratch_bytes(uint32_t n) {
  const size_t groups = ((size_t)n + kTile - 1) / kTile, tiles = ((size_t)n + 255) / 256;
  return (6 * (size_t)n + 256 * groups + 256 + 2 * tiles + 64) * 4;
}

hipError_t coherence_order(const rtx_ray* rays, uint32_t n, const rtx_coherence_config& cfg, const float wmin[3],
                           const float wmax[3], uint32_t* order, uint32_t* hashes_out, void* scratch, hipStream_t s) {
  if (n == 0) return hipSuccess;
  CohParams c{};
  c.rays = rays;
  c.n = n;
  c.hash = (uint32_t)(uint8_t)cfg.hash;
  c.francois_bits = cfg.francois_bits;
  c.grid_bits = cfg.grid_bits;
  c.sphere_bits = cfg.sphere_bits;
  c.two_point_ratio = cfg.two_point_ratio;
  for (int a = 0; a < 3; ++a) {
    c.wmin[a] = wmin[a];
    c.wmax[a] = wmax[a];
  }
  const uint32_t packet = cfg.packet ? cfg.packet : 64u;
  const uint32_t groups = (n + kTile - 1) / kTile, tiles = (n + 1023) / 1024, chunk_tiles = (n + 255) / 256;
  uint32_t* w = static_cast<uint32_t*>(scratch);
  auto take = [&](size_t words) {
    uint32_t* q = w;
    w += words;
    return q;
  };
  uint32_t *hash = take(n), *ray = take(n), *k0 = take(n), *k1 = take(n), *v0 = take(n), *v1 = take(n);
  uint32_t *table = take(256 * (size_t)groups), *totals = take(256), *tile_sums = take(chunk_tiles),
           *size_sums = take(chunk_tiles), *words = take(64);
  uint32_t *n_dev = words, *m_dev = words + 1;
  // stable sort of (keys, positions) by the keys' low `bits` bits; the result is in ka, va
  auto sort = [&](const uint32_t* count, uint32_t bits, uint32_t*& ka, uint32_t*& va, uint32_t*& kb, uint32_t*& vb) {
    const uint32_t* vals = nullptr;
    for (uint32_t shift = 0; shift < bits;) {
      const uint32_t passes = (bits - shift + 7) / 8, d = (bits - shift + passes - 1) / passes;
      hipLaunchKernelGGL(k_digit_counts, dim3(groups), dim3(256), 0, s, ka, count, shift, d, table);
      hipLaunchKernelGGL(k_digit_scan, dim3(1u << d), dim3(256), 0, s, table, groups, totals);
      hipLaunchKernelGGL(k_digit_scatter, dim3(groups), dim3(256), 0, s, ka, vals, count, shift, d, table, totals, kb,
                         vb);
      std::swap(ka, kb);
      std::swap(va, vb);
      vals = va;
      shift += d;
    }
  };
  hipLaunchKernelGGL(k_set_count, dim3(1), dim3(64), 0, s, n_dev, n);
  hipLaunchKernelGGL(k_ray_hash, dim3(std::max(1u, std::min<uint32_t>(8192, (n + 255) / 256))), dim3(256), 0, s, c,
                     hash, hashes_out);
  // pools: rays of one hash, in input order
  sort(n_dev, std::min(32u, hash_bits(cfg)), hash, ray, k0, v0);
  // their chunks in pool order, then by rays left
  hipLaunchKernelGGL(k_chunk_counts, dim3(tiles), dim3(256), 0, s, hash, n, packet, tile_sums);
  hipLaunchKernelGGL(k_scan_sums, dim3(1), dim3(1024), 0, s, tile_sums, tiles, m_dev);
  hipLaunchKernelGGL(k_chunk_keys, dim3(tiles), dim3(256), 0, s, hash, n, packet, tile_sums, k0);
  uint32_t bits = 1;
  while (bits < 32 && (n >> bits)) ++bits;
  sort(m_dev, bits, k0, v0, k1, v1);
  hipLaunchKernelGGL(k_size_sums, dim3(chunk_tiles), dim3(256), 0, s, k0, m_dev, n, packet, size_sums);
  hipLaunchKernelGGL(k_scan_sums, dim3(1), dim3(1024), 0, s, size_sums, chunk_tiles, words + 2);
  hipLaunchKernelGGL(k_chunk_places, dim3(chunk_tiles), dim3(256), 0, s, k0, v0, m_dev, n, packet, size_sums, k1);
  hipLaunchKernelGGL(k_copy_chunks, dim3(tiles), dim3(256), 0, s, hash, n, packet, tile_sums, k1, ray, order);
  return hipGetLastError();
}

}  // namespace rtxk
