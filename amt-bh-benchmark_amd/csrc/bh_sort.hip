// Bounding box, Morton keys and the stable (key, index) sort on CDNA4.
//
// Reference semantics:
//   particle_bounds          flat_build_ttg.h:93-113
//   domain_from_bounds       domain.h:23-30
//   morton_key/spread_bits3  flat_tree.h:104-125
//   sort order               flat_build_ttg.h:62-66 (ascending key, ties by input index)
//   gather to Morton order   flat_build_ttg.h:180-188
//
// This file is compiled with -ffp-contract=off: the domain and key
// arithmetic must round exactly as the reference's FP64 code does.
//
// The sort is an LSD radix sort over the leading 8 p bits of the 63-bit keys
// with the input index as payload, p passes of 8-bit digits, and a last pass
// over the result (k_fix_runs) that orders the runs of keys whose leading bits
// are equal by the bits below. LSD radix sorting is stable, so the result is
// exactly the (key, index) order. p is chosen so that such runs are short
// (sort_passes): 32, 40 or 48 bits hold 10 to 16 octree levels, and the keys
// below them decide only between particles closer together than that. With
// all 63 bits (p = 8) there is nothing to fix. Each radix pass is a single
// "onesweep" kernel: a workgroup ranks a tile of 4,096 or 2,048 keys in LDS with wavefront
// ballots, obtains its global digit offsets by decoupled look-back over the
// preceding tiles, and writes the tile out digit-sorted so stores coalesce.
#include <utility>

#include "bh_internal.h"

namespace bhk {

namespace {

constexpr int kBlock = 256;
constexpr int kSortThreads = 512;
constexpr int kFixTile = 1024;  // positions per k_fix_runs workgroup

__device__ inline uint64_t lanemask_lt() {
  const int lane = __lane_id();
  return lane == 0 ? 0ull : (~0ull >> (64 - lane));
}

// domain.h:23-30 from the reduced bounds lohi = {lo.x, lo.y, lo.z, hi.x, hi.y, hi.z}.
__device__ inline void domain_from_lohi(const double* lohi, double c[3], double* hw) {
  c[0] = 0.5 * (lohi[0] + lohi[3]);
  c[1] = 0.5 * (lohi[1] + lohi[4]);
  c[2] = 0.5 * (lohi[2] + lohi[5]);
  const double ex = lohi[3] - lohi[0], ey = lohi[4] - lohi[1], ez = lohi[5] - lohi[2];
  // std::max({ex, ey, ez}): the first largest; equal values are identical
  double m = ex;
  if (m < ey) m = ey;
  if (m < ez) m = ez;
  double h = 0.5 * m;
  if (!(h > 0.0)) h = 1.0;
  h *= 1.0 + 1e-9;
  *hw = h;
}

__device__ inline uint64_t spread_bits3(uint32_t v) {
  uint64_t x = v & 0x1fffffu;
  x = (x | (x << 32)) & 0x1f00000000ffffull;
  x = (x | (x << 16)) & 0x1f0000ff0000ffull;
  x = (x | (x << 8)) & 0x100f00f00f00f00full;
  x = (x | (x << 4)) & 0x10c30c30c30c30c3ull;
  x = (x | (x << 2)) & 0x1249249249249249ull;
  return x;
}

__device__ inline uint32_t quantize(double v, double lo, double scale) {
  const double cells = 2097152.0;
  double t = floor((v - lo) * scale);
  t = t < 0.0 ? 0.0 : (cells - 1.0 < t ? cells - 1.0 : t);  // std::clamp(t, 0, cells - 1)
  return static_cast<uint32_t>(t);
}

// Zeroes several ranges in one launch.
__global__ __launch_bounds__(kBlock) void k_zero_ranges(ZeroRanges r) {
  zero_ranges(r, blockIdx.x * uint64_t(kBlock) + threadIdx.x, gridDim.x * uint64_t(kBlock));
}

__device__ inline double wave_min(double v) {
  for (int o = 32; o > 0; o >>= 1) v = fmin(v, __shfl_xor(v, o));
  return v;
}
__device__ inline double wave_max(double v) {
  for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o));
  return v;
}

// Where the build reads a particle's position: its record, or the compact
// copy a resident step's walk wrote for its output, four blocks of n
// doubles (x, y, z, m), of which the build reads x, y, z. `finite` checks
// what the source holds (the walk that wrote the compact copy flagged any
// non-finite position, velocity or mass itself).
struct RecordSrc {
  const bh_particle* p;
};
struct CompactSrc {
  const double* p;
  uint64_t n;
};
__device__ inline void pos_of(const RecordSrc& s, uint32_t i, double* x, double* y, double* z, bool* finite) {
  const bh_particle& q = s.p[i];
  *x = q.pos[0];
  *y = q.pos[1];
  *z = q.pos[2];
  *finite = isfinite(*x) && isfinite(*y) && isfinite(*z) && isfinite(q.mass) && isfinite(q.vel[0]) &&
            isfinite(q.vel[1]) && isfinite(q.vel[2]);
}
__device__ inline void pos_of(const CompactSrc& s, uint32_t i, double* x, double* y, double* z, bool* finite) {
  *x = s.p[i];
  *y = s.p[s.n + i];
  *z = s.p[2 * s.n + i];
  *finite = isfinite(*x) && isfinite(*y) && isfinite(*z);
}
// x, y, z and mass
__device__ inline double4 posm_of(const RecordSrc& s, uint32_t i) {
  const bh_particle& q = s.p[i];
  return make_double4(q.pos[0], q.pos[1], q.pos[2], q.mass);
}
__device__ inline double4 posm_of(const CompactSrc& s, uint32_t i) {
  return make_double4(s.p[i], s.p[s.n + i], s.p[2 * s.n + i], s.p[3 * s.n + i]);
}

// The Morton key of a position in the domain whose lowest corner is (lx, ly,
// lz); scale = cells per unit length.
__device__ inline uint64_t morton_key(double x, double y, double z, double lx, double ly, double lz, double scale) {
  return spread_bits3(quantize(x, lx, scale)) | (spread_bits3(quantize(y, ly, scale)) << 1) |
         (spread_bits3(quantize(z, lz, scale)) << 2);
}

// A step's first kernel. Small systems wait for each of a step's launches in
// turn (5 us each), so one takes all that needs nothing but the input: the
// system table, read from pinned host memory, the zeroing, each particle's
// system, and block b < n_chunks the min/max of the positions of chunk b
// (flat_build_ttg.h:93-113; min/max is exact, so the chunking does not matter).
// A chunk with a non-finite position, velocity or mass leaves NaN in place of
// its lower x. (With copies and launches of their own for these, and events and
// copies in place of the report below, a step of 1,000 particles took 252 us,
// now 217; of 65,536 in FP64 800 and 760; of 1M 1,710 and 1,688.)
template <typename Src>
__global__ __launch_bounds__(kBlock) void k_start(Src src, StartArgs a) {
  stamp(a.misc, kStampStart);
  const uint64_t t = blockIdx.x * uint64_t(kBlock) + threadIdx.x, threads = gridDim.x * uint64_t(kBlock);
  const bool mine = blockIdx.x < a.n_chunks;
  uint4 c = make_uint4(0u, blockIdx.x * a.chunk, 0u, 0u);
  if (a.n_sys == 1)
    c.z = a.n - c.y < a.chunk ? a.n : c.y + a.chunk;
  else if (mine)
    c = a.host_chunks[blockIdx.x];
  for (uint64_t i = t; i < a.table_quads; i += threads) a.table[i] = a.host_table[i];
  if (a.host_hist)
    for (uint64_t i = t; i < 2 * 256 / 4; i += threads) a.hist[i] = a.host_hist[i];
  zero_ranges(a.zero, t, threads);
  if (!mine) return;
  for (uint32_t i = c.y + threadIdx.x; i < c.z; i += kBlock) a.sid[i] = static_cast<uint16_t>(c.x);
  const double inf = __builtin_huge_val();
  double lo[3] = {inf, inf, inf}, hi[3] = {-inf, -inf, -inf};
  bool bad = false;
  // kB elements per lane and round, all loads issued before the first use
  // (indices clamped into the chunk, extra elements dropped after the load)
  constexpr int kB = 4;
  for (uint32_t i0 = c.y + threadIdx.x; i0 < c.z; i0 += kB * kBlock) {
    double x[kB], y[kB], z[kB];
    bool fin[kB];
#pragma unroll
    for (int r = 0; r < kB; ++r) {
      const uint32_t i = i0 + r * kBlock < c.z ? i0 + r * kBlock : c.z - 1;
      pos_of(src, i, &x[r], &y[r], &z[r], &fin[r]);
    }
#pragma unroll
    for (int r = 0; r < kB; ++r) {
      if (i0 + r * kBlock >= c.z) break;
      bad |= !fin[r];
      lo[0] = fmin(lo[0], x[r]);
      lo[1] = fmin(lo[1], y[r]);
      lo[2] = fmin(lo[2], z[r]);
      hi[0] = fmax(hi[0], x[r]);
      hi[1] = fmax(hi[1], y[r]);
      hi[2] = fmax(hi[2], z[r]);
    }
  }
  __shared__ double s[4][6];
  const int w = threadIdx.x >> 6, lane = __lane_id();
  double r[6];
  for (int k = 0; k < 3; ++k) {
    r[k] = wave_min(lo[k]);
    r[3 + k] = wave_max(hi[k]);
  }
  if (lane == 0)
    for (int k = 0; k < 6; ++k) s[w][k] = r[k];
  bad = __syncthreads_or(bad);
  if (threadIdx.x < 6) {
    const int k = threadIdx.x;
    double v = s[0][k];
    for (int j = 1; j < 4; ++j) v = k < 3 ? fmin(v, s[j][k]) : fmax(v, s[j][k]);
    a.partial[blockIdx.x * 6 + k] = bad && k == 0 ? __builtin_nan("") : v;
  }
}

// Per system: reduce its chunks' partials to lohi[6 s .. 6 s + 6), and flag a
// chunk with a non-finite value (and, from a compact copy, its writer's flag).
__global__ __launch_bounds__(kBlock) void k_bounds_final(const double* __restrict__ partial,
                                                         const uint32_t* __restrict__ chunk_first,
                                                         const uint32_t* __restrict__ carried_bad, double* __restrict__ lohi,
                                                         uint32_t* __restrict__ nonfinite) {
  const double inf = __builtin_huge_val();
  __shared__ double s[4][6];
  double r[6] = {inf, inf, inf, -inf, -inf, -inf};
  const uint32_t b0 = chunk_first[blockIdx.x], b1 = chunk_first[blockIdx.x + 1];
  bool bad = carried_bad && *carried_bad;
  for (uint32_t b = b0 + threadIdx.x; b < b1; b += kBlock) {
    bad |= partial[b * 6] != partial[b * 6];
    for (int a = 0; a < 3; ++a) {
      r[a] = fmin(r[a], partial[b * 6 + a]);
      r[3 + a] = fmax(r[3 + a], partial[b * 6 + 3 + a]);
    }
  }
  const int w = threadIdx.x >> 6, lane = __lane_id();
  for (int a = 0; a < 3; ++a) {
    r[a] = wave_min(r[a]);
    r[3 + a] = wave_max(r[3 + a]);
  }
  if (lane == 0)
    for (int a = 0; a < 6; ++a) s[w][a] = r[a];
  bad = __syncthreads_or(bad);
  if (bad && threadIdx.x == 0) atomicOr(nonfinite, 1u);
  if (threadIdx.x < 6) {
    const int a = threadIdx.x;
    double v = s[0][a];
    for (int k = 1; k < 4; ++k) v = a < 3 ? fmin(v, s[k][a]) : fmax(v, s[k][a]);
    lohi[6 * blockIdx.x + a] = v;
  }
}

// Morton key per particle (input order) and the histograms of the kDigits
// leading 8-bit digits of all keys, for the onesweep passes' global digit
// offsets.
template <typename Src, int kDigits>
__global__ __launch_bounds__(kBlock) void k_keys_hist(Src src, uint32_t n,
                                                      const uint16_t* __restrict__ sid, const double* __restrict__ lohi,
                                                      uint64_t* __restrict__ keys, uint32_t* __restrict__ hist) {
  constexpr int kShift = kDigits == 8 ? 0 : 63 - 8 * kDigits;
  __shared__ uint32_t s_h[kDigits * 256];
  for (int i = threadIdx.x; i < kDigits * 256; i += kBlock) s_h[i] = 0;
  __syncthreads();
  const int lane = __lane_id();
  const uint32_t stride = gridDim.x * kBlock;
  // each particle's position and system are loaded one round ahead, so the
  // loads of round r + 1 are in flight while round r computes
  double nx = 0.0, ny = 0.0, nz = 0.0;
  uint32_t ns = 0;
  // the domain of the lane's system, computed when it changes
  double lx = 0.0, ly = 0.0, lz = 0.0, scale = 0.0;
  uint32_t have = 0xffffffffu;
  {
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i < n) {
      bool fin;
      pos_of(src, i, &nx, &ny, &nz, &fin);
      ns = sid[i];
    }
  }
  for (uint32_t i0 = blockIdx.x * kBlock; i0 < n; i0 += stride) {
    // the wave's lanes hold consecutive particles; those below n are a
    // prefix of the wave
    const uint32_t i = i0 + threadIdx.x;
    const bool ok = i < n;
    const double x = nx, y = ny, z = nz;
    const uint32_t sys_i = ns;
    if (i + stride < n) {
      bool fin;
      pos_of(src, i + stride, &nx, &ny, &nz, &fin);
      ns = sid[i + stride];
    }
    uint64_t key = 0;
    if (ok) {
      if (sys_i != have) {
        double c[3], hw;
        domain_from_lohi(lohi + 6 * sys_i, c, &hw);
        scale = 2097152.0 / (2.0 * hw);
        lx = c[0] - hw;
        ly = c[1] - hw;
        lz = c[2] - hw;
        have = sys_i;
      }
      key = morton_key(x, y, z, lx, ly, lz, scale);
      keys[i] = key;
    }
    // Input in (or near) Morton order, as a resident step's is, gives long
    // runs of equal digits across the wave, whose atomics on one LDS word
    // would serialise: the first lane of each run adds the run's length.
    const uint32_t nvalid = static_cast<uint32_t>(__popcll(__ballot(ok)));
    const uint64_t prev = __shfl_up(key, 1);
#pragma unroll
    for (int b = 0; b < kDigits; ++b) {
      const uint32_t d = static_cast<uint32_t>(key >> (kShift + 8 * b)) & 255u;
      const uint32_t pd = static_cast<uint32_t>(prev >> (kShift + 8 * b)) & 255u;
      const bool head = ok && (lane == 0 || d != pd);
      const uint64_t heads = __ballot(head);
      const uint64_t after = lane == 63 ? 0ull : heads & (~0ull << (lane + 1));
      const uint32_t end = after ? static_cast<uint32_t>(__ffsll(static_cast<long long>(after)) - 1) : nvalid;
      if (head) atomicAdd(&s_h[b * 256 + d], end - static_cast<uint32_t>(lane));
    }
  }
  __syncthreads();
  for (int i = threadIdx.x; i < kDigits * 256; i += kBlock)
    if (s_h[i]) atomicAdd(&hist[i], s_h[i]);
}

// Exclusive block scan of one value per thread.
template <int kWavesB>
__device__ inline uint32_t block_excl_scan(uint32_t v, uint32_t* s_wsum) {
  const int lane = __lane_id(), w = threadIdx.x >> 6;
  uint32_t x = v;
  for (int o = 1; o < 64; o <<= 1) {
    uint32_t u = __shfl_up(x, o);
    if (lane >= o) x += u;
  }
  if (lane == 63) s_wsum[w] = x;
  __syncthreads();
  uint32_t off = 0;
  for (int k = 0; k < kWavesB; ++k)
    if (k < w) off += s_wsum[k];
  __syncthreads();
  return off + x - v;
}

// kMode 0: first key pass (payload = input index); 1: key pass; 2: system
// pass (digit of sid[payload], keys carried along). hist: this pass's digit
// counts over all keys (each workgroup scans the 256 of them for itself).
//
// For small inputs a pass is a chain of latencies (few tiles, one per CU):
// 512 threads hold 8 keys each, so ranking and scattering take half the
// rounds of 256 with 16, and the look-back reads kWindow tiles at a time
// (one by one it was most of the pass when all tiles publish together). For
// large ones the same tile has twice the wavefronts to hide its loads. A pass
// at 65,536 particles 12 -> 10 us, 1M 22 -> 19, 16M 146 -> 134.
template <int kMode, uint32_t kTile>
__global__ __launch_bounds__(kSortThreads) void k_onesweep(const uint64_t* __restrict__ kin,
                                                           const uint32_t* __restrict__ vin, uint64_t* __restrict__ kout,
                                                           uint32_t* __restrict__ vout, uint32_t n, uint32_t shift,
                                                           const uint16_t* __restrict__ sid,
                                                           const uint32_t* __restrict__ hist,
                                                           uint32_t* __restrict__ lookback,
                                                           uint32_t* __restrict__ tile_counter) {
  constexpr int kW = kSortThreads / 64;
  constexpr int kI = static_cast<int>(kTile) / kSortThreads;
  constexpr uint32_t kPerWave = kTile / kW;
  constexpr int kWindow = 8;
  __shared__ uint32_t s_hist[kW][256];  // per-wave digit counters, then per-wave exclusive bases
  __shared__ uint32_t s_lexcl[256];     // tile-local exclusive digit offsets
  __shared__ uint32_t s_adj[256];       // global position - local position, per digit
  __shared__ uint64_t s_k[kTile];   // the tile in digit order: keys, then (reused) payloads
  __shared__ uint8_t s_d[kTile];
  uint32_t* s_v = reinterpret_cast<uint32_t*>(s_k);
  __shared__ uint32_t s_w[kW];
  __shared__ uint32_t s_tile;

  const int tid = threadIdx.x, w = tid >> 6, lane = __lane_id();
  if (tid == 0) s_tile = atomicAdd(tile_counter, 1u);
  const uint32_t count = tid < 256 ? hist[tid] : 0u;
  for (int i = tid; i < kW * 256; i += kSortThreads) (&s_hist[0][0])[i] = 0;
  __syncthreads();
  const uint32_t tile = s_tile;
  const uint32_t base = tile * kTile;

  uint64_t k[kI];
  uint32_t v[kI];
  uint32_t r[kI];
  uint32_t dg[kI];
#pragma unroll
  for (int j = 0; j < kI; ++j) {
    const uint32_t idx = base + w * kPerWave + j * 64 + lane;
    const bool ok = idx < n;
    k[j] = ok ? kin[idx] : ~0ull;
    v[j] = kMode == 0 ? idx : (ok ? vin[idx] : 0u);
    if (kMode == 2)
      dg[j] = ok ? (static_cast<uint32_t>(sid[v[j]]) >> shift) & 255u : 255u;
    else
      dg[j] = static_cast<uint32_t>(k[j] >> shift) & 255u;
  }
  const uint32_t dbase = block_excl_scan<kW>(count, s_w);  // keys with smaller digits
  const uint64_t lt = lanemask_lt();
  // Stable in-tile ranking: items in (wave, item, lane) order follow the
  // input order; lanes with an equal digit are found with 8 ballots.
#pragma unroll
  for (int j = 0; j < kI; ++j) {
    const uint32_t idx = base + w * kPerWave + j * 64 + lane;
    const bool ok = idx < n;
    const uint32_t d = dg[j];
    uint64_t peers = __ballot(ok);
#pragma unroll
    for (int b = 0; b < 8; ++b) {
      const bool bit = (d >> b) & 1u;
      const uint64_t bb = __ballot(bit);
      peers &= bit ? bb : ~bb;
    }
    const uint32_t below = __popcll(peers & lt);
    const uint32_t cnt = s_hist[w][d];
    r[j] = cnt + below;
    __builtin_amdgcn_wave_barrier();
    if (ok && below == 0) s_hist[w][d] = cnt + __popcll(peers);
    __builtin_amdgcn_wave_barrier();
  }
  __syncthreads();
  // per digit (thread t < 256): totals over waves and per-wave exclusive bases
  const uint32_t t = tid;
  uint32_t total = 0;
  uint32_t* my = &lookback[uint64_t(tile) * 256 + t];
  if (t < 256) {
#pragma unroll
    for (int q = 0; q < kW; ++q) {
      const uint32_t c = s_hist[q][t];
      s_hist[q][t] = total;
      total += c;
    }
    __hip_atomic_store(my, (tile == 0 ? kLbPre : kLbAgg) | total, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  const uint32_t lex = block_excl_scan<kW>(total, s_w);
  if (t < 256) {
    s_lexcl[t] = lex;
    uint32_t excl = 0;
    if (tile > 0) {
      // tiles j, j - 1, ... : aggregates up to the nearest inclusive prefix
      for (int64_t j = static_cast<int64_t>(tile) - 1;;) {
        uint32_t val[kWindow];
#pragma unroll
        for (int q = 0; q < kWindow; ++q)
          val[q] = j - q >= 0 ? __hip_atomic_load(&lookback[uint64_t(j - q) * 256 + t], __ATOMIC_RELAXED,
                                                  __HIP_MEMORY_SCOPE_AGENT)
                              : kLbPre;
        bool found = false, wait = false;
        int used = 0;
#pragma unroll
        for (int q = 0; q < kWindow; ++q) {
          const uint32_t f = val[q] & ~kLbVal;
          wait |= f == 0;
          if (!found && !wait) {
            excl += val[q] & kLbVal;
            ++used;
            found = f == kLbPre;
          }
        }
        if (found) break;
        j -= used;
      }
      __hip_atomic_store(my, kLbPre | (excl + total), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    s_adj[t] = dbase + excl - lex;
  }
  __syncthreads();
  // keys, then payloads, through the same LDS tile in digit order, so that
  // the stores coalesce (one tile buffer keeps three workgroups per CU)
#pragma unroll
  for (int j = 0; j < kI; ++j) {
    const uint32_t idx = base + w * kPerWave + j * 64 + lane;
    if (idx < n) {
      const uint32_t d = dg[j];
      const uint32_t pos = s_lexcl[d] + s_hist[w][d] + r[j];
      s_k[pos] = k[j];
      s_d[pos] = static_cast<uint8_t>(d);
      r[j] = pos;
    }
  }
  __syncthreads();
  const uint32_t tn = n - base < kTile ? n - base : kTile;
  uint32_t g[kI];
#pragma unroll
  for (int j = 0; j < kI; ++j) {
    const uint32_t e = tid + j * kSortThreads;
    g[j] = e < tn ? s_adj[s_d[e]] + e : 0u;
    if (e < tn) kout[g[j]] = s_k[e];
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < kI; ++j) {
    const uint32_t idx = base + w * kPerWave + j * 64 + lane;
    if (idx < n) s_v[r[j]] = v[j];
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < kI; ++j) {
    const uint32_t e = tid + j * kSortThreads;
    if (e < tn) vout[g[j]] = s_v[e];
  }
}

// Orders the runs of equal leading key bits (key >> shift, within a system)
// by (key, index). The radix passes left each run in index order, so a run
// whose keys ascend is done, which equal positions always are. A wavefront
// takes a run of up to 64 keys and ranks them among each other in registers. A
// fall in a longer run sets kAbortSort: the host runs the step again with full
// keys, whose passes take less time than ordering such runs would. (Ranked key
// by key against the run in memory, up to 1,024 keys: sort phase of 20,000
// particles in boxes of which runs hold some 600, 743 us; with full keys 73, and
// 1M 386 against 228.) The wavefront looks for a fall among the run's first 64
// keys, each later position's thread at its own (read by one wavefront to its
// end, a run of 100,000 equal keys among 300,000 took 0.95 of a 1.06 ms sort
// phase; now 0.12).
constexpr uint32_t kRunCap = kWave;

__global__ __launch_bounds__(kBlock) void k_fix_runs(uint64_t* keys, uint32_t* vals, uint32_t n, uint32_t shift,
                                                     const uint16_t* __restrict__ sid, uint32_t* __restrict__ abort) {
  __shared__ uint32_t s_head[kFixTile];
  __shared__ uint32_t s_n;
  const uint32_t base = blockIdx.x * kFixTile;
  const int w = threadIdx.x >> 6, lane = __lane_id();
  if (threadIdx.x == 0) s_n = 0;
  __syncthreads();
  constexpr int kI = kFixTile / kBlock;
  uint64_t k0[kI], k1[kI], kp[kI];
#pragma unroll
  for (int j = 0; j < kI; ++j) {
    const uint32_t i = base + j * kBlock + threadIdx.x;
    k0[j] = i < n ? keys[i] : 0ull;
    k1[j] = i + 1 < n ? keys[i + 1] : ~0ull;
    kp[j] = i > 0 && i < n ? keys[i - 1] : ~0ull;
  }
#pragma unroll
  for (int j = 0; j < kI; ++j) {
    const uint32_t i = base + j * kBlock + threadIdx.x;
    const uint64_t top = k0[j] >> shift;
    if (i > 0 && i < n && (kp[j] >> shift) == top && sid[i - 1] == sid[i]) {
      // a fall behind the first kRunCap keys of a run. (Another workgroup may be
      // ordering this run, but then it has no key kRunCap places back.)
      if (kp[j] > k0[j] && i >= kRunCap && (keys[i - kRunCap] >> shift) == top && sid[i - kRunCap] == sid[i])
        atomicOr(abort, kAbortSort);
      continue;
    }
    if (i + 1 >= n || (k1[j] >> shift) != top || sid[i] != sid[i + 1]) continue;
    s_head[atomicAdd(&s_n, 1u)] = i;  // the first of a run of at least two
  }
  __syncthreads();
  const uint32_t runs = s_n;
  for (uint32_t h = w; h < runs; h += kBlock / 64) {
    const uint32_t b = s_head[h];
    const uint16_t sys = sid[b];
    // the run's first keys, whether they ascend, and whether there are more
    const uint32_t i = b + lane;
    const uint64_t k = i < n ? keys[i] : 0ull;
    const uint64_t top = __shfl(k, 0) >> shift;
    const uint64_t out = __ballot(i >= n || (k >> shift) != top || sid[i] != sys);
    const uint32_t len = out ? static_cast<uint32_t>(__ffsll(static_cast<long long>(out)) - 1) : 64u;
    const bool in = static_cast<uint32_t>(lane) < len;
    const uint64_t before = __shfl_up(k, 1);
    if (!__ballot(in && lane > 0 && before > k)) continue;
    if (len == kRunCap && b + kRunCap < n && (keys[b + kRunCap] >> shift) == top && sid[b + kRunCap] == sys) {
      if (lane == 0) atomicOr(abort, kAbortSort);
      continue;
    }
    const uint32_t v = in ? vals[i] : ~0u;
    uint32_t rank = 0;
    for (uint32_t q = 0; q < len; ++q) {
      const uint64_t kq = __shfl(k, static_cast<int>(q));
      rank += kq < k || (kq == k && q < static_cast<uint32_t>(lane)) ? 1u : 0u;
    }
    if (in) {
      keys[b + rank] = k;
      vals[b + rank] = v;
    }
  }
}

// Permutes the particles into Morton order and writes the FP64 walk copy
// (x, y, z, m), as sort_particles' final loop does (flat_build_ttg.h:180-188).
// Without out only the walk copy is written (a step's walk writes the
// Morton-ordered particles from the input itself).
__global__ __launch_bounds__(kBlock) void k_gather(const bh_particle* __restrict__ in, bh_particle* __restrict__ out,
                                                   const uint32_t* __restrict__ perm, double4* __restrict__ posm, uint32_t n) {
  // four lanes per particle, one 16-byte quarter each: consecutive lanes
  // read and write consecutive 16-byte pieces
  const uint32_t t = blockIdx.x * kBlock + threadIdx.x;
  const uint32_t k = t >> 2, part = t & 3u;
  if (k >= n) return;  // whole quads leave together
  const uint32_t j = perm[k];
  // the walk copy needs quarters 0-2 only
  uint4 v = make_uint4(0, 0, 0, 0);
  if (out || part < 3) v = reinterpret_cast<const uint4*>(in + j)[part];
  if (out) reinterpret_cast<uint4*>(out + k)[part] = v;
  // quarters: 0 = {id, pad, mass}, 1 = {x, y}, 2 = {z, vx}, 3 = {vy, vz}
  const int lane = __lane_id();
  const uint32_t mlo = static_cast<uint32_t>(__shfl(static_cast<int>(v.z), lane ^ 2));
  const uint32_t mhi = static_cast<uint32_t>(__shfl(static_cast<int>(v.w), lane ^ 2));
  uint4* q = reinterpret_cast<uint4*>(posm + k);
  if (part == 1) q[0] = v;
  if (part == 2) q[1] = make_uint4(v.x, v.y, mlo, mhi);
}

// The walk copy from a carried compact copy (blocks of n x, y, z and m in
// the last resident step's order, which is the order perm indexes). The
// copy holds the same FP64 values as the records, so the result equals
// k_gather's.
// Two lanes per particle: lane half 0 moves x, y, half 1 z, m (one 16-byte
// half of the walk record each).
__global__ __launch_bounds__(kBlock) void k_gather_pos(const double* __restrict__ pos, const uint32_t* __restrict__ perm,
                                                       double4* __restrict__ posm, uint32_t n) {
  const uint32_t t = blockIdx.x * kBlock + threadIdx.x;
  const uint32_t k = t >> 1, half = t & 1u;
  if (k >= n) return;
  const uint64_t j = perm[k];
  const uint64_t b0 = (2ull * half) * n + j;
  reinterpret_cast<double2*>(posm + k)[half] = make_double2(pos[b0], pos[b0 + n]);
}

// What k_start, k_bounds_final, the keys, the sort and the gather do, for one
// system of at most kSmallSort particles: nine launches that each wait for the
// one before take 5 us apiece, whatever they hold. Block b orders particles
// [1024 b, 1024 b + 1024) by (key, index), each block from bounds of its own over
// all particles, and k_small_merge merges the blocks (a single block writes
// the result itself). The sort is bitonic, on the key's leading 54 bits (18
// levels) with the index in the block below them, one element per thread, with
// shuffles inside a wavefront and LDS, two buffers in turn so that a step needs
// one barrier, beyond. Runs that share the 54 bits are then ordered by the rest
// of the key (a count over the run).
//
// The code runs once a step, from cold instruction caches: loops stay rolled
// where no load waits in them. (All 4,096 in one workgroup: 48 us, with an
// unrolled body 53.) Sort phase, nine launches -> here: 1,000 particles 45 -> 20
// us, 4,096 53 -> 29, 8,192 58 -> 38, 12,000 59 -> 48; 16,384 57 -> 56: the line
// is at 12,288.
constexpr int kSmallThreads = 1024;
constexpr int kSmallBits = 54;  // 64 - 10 for the index in the block

template <typename Src>
__global__ __launch_bounds__(kSmallThreads) void k_small_sort(Src src, const uint32_t* __restrict__ carried_bad, StartArgs a,
                                                              uint64_t* __restrict__ keys, uint32_t* __restrict__ perm,
                                                              double4* __restrict__ posm) {
  constexpr int kWaves = kSmallThreads / 64;
  constexpr int kLoads = 4;
  __shared__ uint64_t s_x[2][kSmallThreads], s_key[kSmallThreads];
  __shared__ double s_red[6][kWaves];
  __shared__ double s_lohi[6];
  stamp(a.misc, kStampStart);
  const uint32_t t = threadIdx.x, base = blockIdx.x * kSmallThreads;
  const uint32_t cnt = a.n - base < kSmallThreads ? a.n - base : kSmallThreads;
  const double inf = __builtin_huge_val();
  double b[6] = {inf, inf, inf, inf, inf, inf};  // lo, and -hi
  bool bad = t == 0 && carried_bad && *carried_bad != 0;
  double mx, my, mz;  // this thread's particle
  {
    bool fin;
    pos_of(src, base + (t < cnt ? t : cnt - 1), &mx, &my, &mz, &fin);
  }
#pragma unroll 1
  for (uint32_t i0 = 0; i0 < a.n; i0 += kLoads * kSmallThreads) {
    double x[kLoads], y[kLoads], z[kLoads];
#pragma unroll
    for (int j = 0; j < kLoads; ++j) {
      // past the end the last particle again
      const uint32_t i = i0 + t + j * kSmallThreads;
      bool fin;
      if (j > 0 && i0 + j * kSmallThreads >= a.n) {
        x[j] = x[0];
        y[j] = y[0];
        z[j] = z[0];
        continue;
      }
      pos_of(src, i < a.n ? i : a.n - 1, &x[j], &y[j], &z[j], &fin);
      bad |= !fin;
    }
#pragma unroll
    for (int j = 0; j < kLoads; ++j) {
      b[0] = fmin(b[0], x[j]);
      b[1] = fmin(b[1], y[j]);
      b[2] = fmin(b[2], z[j]);
      b[3] = fmin(b[3], -x[j]);
      b[4] = fmin(b[4], -y[j]);
      b[5] = fmin(b[5], -z[j]);
    }
  }
#pragma unroll 1
  for (uint32_t i = base + t; i < a.table_quads; i += gridDim.x * kSmallThreads) a.table[i] = a.host_table[i];
  // misc (range 0) is the first block's, which also writes to it
#pragma unroll 1
  for (int k = blockIdx.x ? 1 : 0; k < ZeroRanges::kMax; ++k) {
    uint32_t* p = a.zero.p[k];
#pragma unroll 1
    for (uint64_t i = k ? base + t : t; i < a.zero.n[k]; i += k ? gridDim.x * kSmallThreads : kSmallThreads) p[i] = 0u;
  }
  if (t < cnt) a.sid[base + t] = 0;
#pragma unroll 1
  for (int o = 32; o > 0; o >>= 1)
#pragma unroll
    for (int k = 0; k < 6; ++k) b[k] = fmin(b[k], __shfl_xor(b[k], o));
  if (__lane_id() == 0)
#pragma unroll
    for (int k = 0; k < 6; ++k) s_red[k][t >> 6] = b[k];
  bad = __syncthreads_or(bad);  // and misc is zero
  if (bad && t == 0 && blockIdx.x == 0) a.misc[kMiscNonfinite] = 1u;
  if (t < 6) {
    double v = s_red[t][0];
#pragma unroll 1
    for (int q = 1; q < kWaves; ++q) v = fmin(v, s_red[t][q]);
    if (t >= 3) v = -v;
    s_lohi[t] = v;
    if (blockIdx.x == 0) a.lohi[t] = v;
  }
  __syncthreads();
  uint64_t v;
  {
    double c[3], hw;
    domain_from_lohi(s_lohi, c, &hw);
    const uint64_t key = morton_key(mx, my, mz, c[0] - hw, c[1] - hw, c[2] - hw, 2097152.0 / (2.0 * hw));
    s_key[t] = key;
    v = t < cnt ? (key >> (63 - kSmallBits)) << (64 - kSmallBits) | t : ~0ull;
  }
  uint32_t turn = 0;
#pragma unroll 1
  for (uint32_t k = 2; k <= kSmallThreads; k <<= 1)
#pragma unroll 1
    for (uint32_t m = k >> 1; m > 0; m >>= 1) {
      // the smaller element stays here in the lower half of an ascending
      // block and in the upper half of a descending one
      const bool keep_min = ((t & m) == 0) == ((t & k) == 0);
      uint64_t o;
      if (m < 64) {
        o = __shfl_xor(static_cast<unsigned long long>(v), static_cast<int>(m));
      } else {
        s_x[turn][t] = v;
        __syncthreads();
        o = s_x[turn][t ^ m];
        turn ^= 1;
      }
      v = (v < o) == keep_min ? v : o;
    }
  __syncthreads();
  // the whole key at place t
  const uint32_t i = static_cast<uint32_t>(v) & (kSmallThreads - 1);
  const uint64_t key = s_key[i], lead = key >> (63 - kSmallBits);
  s_x[0][t] = key;
  __syncthreads();
  if (t >= cnt) return;
  uint32_t at = t;
  if ((t > 0 && s_x[0][t - 1] >> (63 - kSmallBits) == lead) || (t + 1 < cnt && s_x[0][t + 1] >> (63 - kSmallBits) == lead)) {
    // the run of these leading bits, in input order, starts at r0
    uint32_t r0 = 0;
    for (uint32_t q = t; r0 < q;) {
      const uint32_t mid = (r0 + q) / 2;
      if (s_x[0][mid] >> (63 - kSmallBits) < lead)
        r0 = mid + 1;
      else
        q = mid;
    }
    at = r0;
    for (uint32_t q = r0; q < cnt && s_x[0][q] >> (63 - kSmallBits) == lead; ++q)
      at += s_x[0][q] < key || (s_x[0][q] == key && q < t);
  }
  keys[base + at] = key;
  perm[base + at] = base + i;
  if (posm) posm[base + at] = posm_of(src, base + i);
}

// Merges the ordered blocks of k_small_sort: an element's place is its own in
// its block, and in every other block the number of elements that go before it
// (of equal keys those of earlier blocks).
template <typename Src>
__global__ __launch_bounds__(kBlock) void k_small_merge(Src src, uint32_t n, const uint64_t* __restrict__ bkeys,
                                                        const uint32_t* __restrict__ bperm, uint64_t* __restrict__ keys,
                                                        uint32_t* __restrict__ perm, double4* __restrict__ posm) {
  extern __shared__ uint64_t s_k[];  // n
#pragma unroll 8
  for (uint32_t i = threadIdx.x; i < n; i += kBlock) s_k[i] = bkeys[i];
  const uint32_t e = blockIdx.x * kBlock + threadIdx.x, mine = e / kSmallThreads;
  const uint32_t i = e < n ? bperm[e] : 0u;
  const double4 q = posm_of(src, i);
  __syncthreads();
  if (e >= n) return;
  const uint64_t key = s_k[e];
  uint32_t at = e - mine * kSmallThreads;
#pragma unroll 1
  for (uint32_t b = 0; b * kSmallThreads < n; ++b) {
    if (b == mine) continue;
    uint32_t lo = b * kSmallThreads, hi = n - lo < kSmallThreads ? n : lo + kSmallThreads;
    const uint32_t first = lo;
    while (lo < hi) {
      const uint32_t mid = (lo + hi) / 2;
      if (s_k[mid] < key || (s_k[mid] == key && b < mine))
        lo = mid + 1;
      else
        hi = mid;
    }
    at += lo - first;
  }
  keys[at] = key;
  perm[at] = i;
  if (posm) posm[at] = q;
}

// The report, written to pinned host memory by the step itself (no copies
// back, and the phases' times come with it: no events between them).
__global__ __launch_bounds__(128) void k_report(uint32_t* __restrict__ misc, uint32_t* __restrict__ host) {
  static_assert(kReportWords <= 128, "one thread per word");
  stamp(misc, kStampEnd);
  __syncthreads();
  if (threadIdx.x < kReportWords)
    __hip_atomic_store(&host[threadIdx.x], misc[threadIdx.x], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

inline uint32_t grid_for(uint64_t n, uint32_t cap) {
  uint64_t g = (n + kBlock - 1) / kBlock;
  if (g < 1) g = 1;
  return static_cast<uint32_t>(g < cap ? g : cap);
}

}  // namespace

hipError_t launch_zero(const ZeroRanges& r, hipStream_t s) {
  uint64_t most = 0;
  for (int k = 0; k < ZeroRanges::kMax; ++k) most = r.n[k] > most ? r.n[k] : most;
  if (most == 0) return hipSuccess;
  hipLaunchKernelGGL(k_zero_ranges, dim3(grid_for(most, 4096)), dim3(kBlock), 0, s, r);
  return hipGetLastError();
}

namespace {
template <typename Src>
hipError_t start(Src src, const uint32_t* carried_bad, const StartArgs& a, hipStream_t s) {
  // blocks beyond the chunks only zero: 16 KB a block
  uint64_t words = 0;
  for (int k = 0; k < ZeroRanges::kMax; ++k) words += a.zero.n[k];
  const uint64_t zeroing = words / 4096 + 1 < 2048 ? words / 4096 + 1 : 2048;
  const uint32_t blocks = a.n_chunks > zeroing ? a.n_chunks : static_cast<uint32_t>(zeroing);
  hipLaunchKernelGGL(k_start<Src>, dim3(blocks), dim3(kBlock), 0, s, src, a);
  hipLaunchKernelGGL(k_bounds_final, dim3(a.n_sys), dim3(kBlock), 0, s, a.partial, a.chunk_first, carried_bad, a.lohi,
                     a.misc + kMiscNonfinite);
  return hipGetLastError();
}
}  // namespace

hipError_t launch_start(const bh_particle* p, const StartArgs& a, hipStream_t s) {
  return start(RecordSrc{p}, nullptr, a, s);
}

hipError_t launch_start(const double* pos, const uint32_t* carried_bad, const StartArgs& a, hipStream_t s) {
  return start(CompactSrc{pos, a.n}, carried_bad, a, s);
}

namespace {
template <typename Src>
hipError_t small_sort(Src src, const uint32_t* carried_bad, const StartArgs& a, uint64_t* keys, uint32_t* perm,
                      uint64_t* bkeys, uint32_t* bperm, double4* posm, hipStream_t s) {
  if (a.n == 0 || a.n > kSmallSort || a.n_sys != 1) return hipErrorInvalidValue;
  const uint32_t blocks = (a.n + kSmallThreads - 1) / kSmallThreads;
  const bool one = blocks == 1;
  hipLaunchKernelGGL(k_small_sort<Src>, dim3(blocks), dim3(kSmallThreads), 0, s, src, carried_bad, a, one ? keys : bkeys,
                     one ? perm : bperm, one ? posm : nullptr);
  if (!one)
    hipLaunchKernelGGL(k_small_merge<Src>, dim3((a.n + kBlock - 1) / kBlock), dim3(kBlock), a.n * sizeof(uint64_t), s,
                       src, a.n, bkeys, bperm,
                       keys, perm, posm);
  return hipGetLastError();
}
}  // namespace

hipError_t launch_small_sort(const bh_particle* p, const StartArgs& a, uint64_t* keys, uint32_t* perm, uint64_t* bkeys,
                             uint32_t* bperm, double4* posm, hipStream_t s) {
  return small_sort(RecordSrc{p}, nullptr, a, keys, perm, bkeys, bperm, posm, s);
}

hipError_t launch_small_sort(const double* pos, const uint32_t* carried_bad, const StartArgs& a, uint64_t* keys,
                             uint32_t* perm, uint64_t* bkeys, uint32_t* bperm, double4* posm, hipStream_t s) {
  return small_sort(CompactSrc{pos, a.n}, carried_bad, a, keys, perm, bkeys, bperm, posm, s);
}

hipError_t launch_report(uint32_t* misc, uint32_t* host, hipStream_t s) {
  hipLaunchKernelGGL(k_report, dim3(1), dim3(128), 0, s, misc, host);
  return hipGetLastError();
}

namespace {
template <typename Src>
hipError_t keys_hist(Src src, uint32_t n, int passes, const uint16_t* sid, const double* lohi, uint64_t* keys,
                     uint32_t* hist, hipStream_t s) {
  // Every workgroup adds its digit counts to the global ones, kDigits * 256
  // atomics on the same words: a thread takes 2 to 16 particles so that they
  // stay few (us, by particles per thread: 65,536 1: 8.7, 2: 6.3, 8: 10.8;
  // 262,144 1: 24, 8: 12.1; 1M 2: 49, 16: 19.9; 4M 8: 68, 16: 54).
  const uint32_t few = n / 512 < 128 ? n / 512 + 1 : 128, many = n / 4096 < 2048 ? n / 4096 : 2048;
  const dim3 g(few > many ? few : many), b(kBlock);
  switch (passes) {
    case 4: hipLaunchKernelGGL((k_keys_hist<Src, 4>), g, b, 0, s, src, n, sid, lohi, keys, hist); break;
    case 5: hipLaunchKernelGGL((k_keys_hist<Src, 5>), g, b, 0, s, src, n, sid, lohi, keys, hist); break;
    case 6: hipLaunchKernelGGL((k_keys_hist<Src, 6>), g, b, 0, s, src, n, sid, lohi, keys, hist); break;
    case 8: hipLaunchKernelGGL((k_keys_hist<Src, 8>), g, b, 0, s, src, n, sid, lohi, keys, hist); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}
}  // namespace

hipError_t launch_keys_hist(const bh_particle* p, uint32_t n, int passes, const uint16_t* sid, const double* lohi,
                            uint64_t* keys, uint32_t* hist, hipStream_t s) {
  return keys_hist(RecordSrc{p}, n, passes, sid, lohi, keys, hist, s);
}

hipError_t launch_keys_hist(const double* pos, uint32_t n, int passes, const uint16_t* sid, const double* lohi,
                            uint64_t* keys, uint32_t* hist, hipStream_t s) {
  return keys_hist(CompactSrc{pos, n}, n, passes, sid, lohi, keys, hist, s);
}

namespace {
template <int kMode>
void onesweep(uint32_t tile, uint32_t tiles, const uint64_t* kin, const uint32_t* vin, uint64_t* ko, uint32_t* vo, uint32_t n,
              uint32_t shift, const uint16_t* sid, const uint32_t* hist, uint32_t* lookback, uint32_t* counter,
              hipStream_t s) {
  if (tile == kSortTile)
    hipLaunchKernelGGL((k_onesweep<kMode, kSortTile>), dim3(tiles), dim3(kSortThreads), 0, s, kin, vin, ko, vo, n, shift,
                       sid, hist, lookback, counter);
  else
    hipLaunchKernelGGL((k_onesweep<kMode, kSortTile / 2>), dim3(tiles), dim3(kSortThreads), 0, s, kin, vin, ko, vo, n,
                       shift, sid, hist, lookback, counter);
}
}  // namespace

hipError_t launch_radix_sort(uint64_t* keys_a, uint32_t* vals_a, uint64_t* keys_b, uint32_t* vals_b, uint32_t n,
                             uint32_t tile, int key_passes, int sid_passes, const uint16_t* sid, const uint32_t* hist,
                             uint32_t* lookback, uint32_t* abort, uint64_t** keys_out, uint32_t** vals_out,
                             hipStream_t s) {
  if (tile != kSortTile && tile != kSortTile / 2) return hipErrorInvalidValue;
  const uint32_t tiles = (n + tile - 1) / tile;
  const uint32_t low = key_passes == 8 ? 0u : 63u - 8u * key_passes;  // bits below the radix digits
  uint64_t* kin = keys_a;
  uint32_t* vin = vals_a;
  uint64_t* ko = keys_b;
  uint32_t* vo = vals_b;
  for (int pass = 0; pass < key_passes + sid_passes; ++pass) {
    uint32_t* lb = lookback + radix_lookback_words(n, tile, pass);
    uint32_t* counter = lookback + pass;
    if (pass == 0)
      onesweep<0>(tile, tiles, kin, vin, ko, vo, n, low, sid, hist, lb, counter, s);
    else if (pass < key_passes)
      onesweep<1>(tile, tiles, kin, vin, ko, vo, n, low + 8u * pass, sid, hist + pass * 256, lb, counter, s);
    else
      onesweep<2>(tile, tiles, kin, vin, ko, vo, n, 8u * (pass - key_passes), sid, hist + (8 + pass - key_passes) * 256, lb,
                  counter, s);
    std::swap(kin, ko);
    std::swap(vin, vo);
  }
  if (low)
    hipLaunchKernelGGL(k_fix_runs, dim3((n + kFixTile - 1) / kFixTile), dim3(kBlock), 0, s, kin, vin, n, low, sid, abort);
  *keys_out = kin;
  *vals_out = vin;
  return hipGetLastError();
}

hipError_t launch_gather(const bh_particle* in, bh_particle* out, const uint32_t* perm, double4* posm, uint32_t n,
                         hipStream_t s) {
  hipLaunchKernelGGL(k_gather, dim3((4ull * n + kBlock - 1) / kBlock), dim3(kBlock), 0, s, in, out, perm, posm, n);
  return hipGetLastError();
}

hipError_t launch_gather(const double* pos, const uint32_t* perm, double4* posm, uint32_t n, hipStream_t s) {
  hipLaunchKernelGGL(k_gather_pos, dim3((2ull * n + kBlock - 1) / kBlock), dim3(kBlock), 0, s, pos, perm, posm, n);
  return hipGetLastError();
}

}  // namespace bhk
