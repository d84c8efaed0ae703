// The grouped force walk on CDNA4: one wavefront per walk unit or piece of one.
//
// Reference semantics:
//   targets           grouped_ttg.h:253 (topmost nodes with leaf || count <= target_size)
//   MAC               multipole.h:130-153: accept iff theta^2 * near2(com) > (2*hw)^2,
//                     near2 against the FP64 bounding box of the target's particles
//   lists             grouped_ttg.h:223-249: accepted nodes -> quadrupole cells (or
//                     monopoles without quadrupole), opened leaves -> their particles
//                     (the target's own included), opened interior nodes -> children
//   P2P               grouped_ttg.h:124-163: a += m d (r^2 + eps^2)^(-3/2), r = 0 masked
//                     when eps2 == 0
//   P2C               multipole.h:171-200: monopole + traceless quadrupole
//   kick/drift        integrate.h:15-16 via integrate_ttg.h:74-77, fused
//
// Work is split into walk units, one wavefront each: walk groups (topmost
// nodes with leaf || count <= max(tsm, 128)), with runs of sibling groups
// that are single targets packed into units of up to 128 particles. A
// group that is itself a target (and not packed) walks as one target.
// Otherwise the wavefront first walks the tree for the unit's particle box
// with the reference's three-way decision at a group node
// (grouped_ttg.h:259-276): accepted (theta^2 near2 > edge^2) -> the shared
// list, rejected for every box inside (theta^2 far2 <= edge^2) -> opened
// for all, otherwise deferred. The shared list is evaluated for all the
// unit's particles at once. Then each target of the unit walks only the
// deferred nodes. This gives every
// target exactly the interaction list of its own walk from the root: near2
// and far2 are monotone in the box (also in floating point) and near2 <=
// far2, so a group's accept / reject-for-all is the decision of every
// target box inside, and a target opens whatever it does not accept
// (grouped_ttg.h:42-51). A unit of a system too small to fill the GPU is
// walked by several wavefronts, each for a piece of its particles (the walk
// itself with the whole unit's box, so the lists are the same).
//
// Per iteration a wavefront pops up to 64 nodes of the top frame of its
// LDS stack (frame d holds child ranges d levels below the walk's start),
// tests them with 64 lanes in FP64 - bit-identical to the reference's
// decisions - and compacts the outcomes with ballots: children ranges into
// frame d+1, accepted cells into the P2C ring, opened leaves' particles
// into the P2P ring. Ring entries are staged as (source - box centre) in
// FP64, then rounded to the walk precision, so FP32 arithmetic never sees
// absolute coordinates. Whenever a ring holds a batch it is evaluated. For a
// target with T particles, lane = (particle p, slice s): each of the
// S = 64 / T slices takes its share of the entries, so small leaves still use
// the whole wavefront. FP32 batch sums are accumulated per lane in FP64;
// slices, the group's share and the target's own list are combined in
// FP64.
//
// No MFMA: the only GEMM-shaped part, the quadrupole's Q.d, is a K = 4
// product; on gfx950 the FP32 MFMA does not issue beside the VALU, and a
// bf16-split form would need more registers than four waves per SIMD leave.
#include <algorithm>
#include <type_traits>

#include "bh_internal.h"

namespace bhk {

namespace {

// Staged entries that make a batch, and staging capacity: kBatch - 1 left over
// + 64 staged at once. FP64 entries take twice the LDS; with 48 only 10
// wavefronts fitted a CU, with 22 the 12 that the registers allow do (walk of
// 65,536 particles 0.575 -> 0.54 ms, 131,072 1.65 -> 1.52, 1M 5.73 -> 5.55; 16:
// 0.62, 1.60, 5.78).
template <typename Real>
constexpr int kBatch = sizeof(Real) == 4 ? 48 : 22;
template <typename Real>
constexpr int kBuf = kBatch<Real> + 64;
constexpr int kGroupChunks = kGroupCap / kWave;  // a group's particle slots per lane

template <typename Real>
struct Vec4T;
template <>
struct Vec4T<float> {
  using T = float4;
};
template <>
struct Vec4T<double> {
  using T = double4;
};
template <typename Real>
struct Vec2T;
template <>
struct Vec2T<float> {
  using T = float2;
};
template <>
struct Vec2T<double> {
  using T = double2;
};

// The P2C ring: cell i is {x, y, z, m} a[i], {Qxx, Qyy, Qzz, Qxy} b[i],
// {Qxz, Qyz} c[i] (40 bytes in FP32).
template <typename Real>
struct PcRing {
  typename Vec4T<Real>::T a[kBuf<Real>];
  typename Vec4T<Real>::T b[kBuf<Real>];
  typename Vec2T<Real>::T c[kBuf<Real>];
};

// The walk's stack: frame d holds the child ranges d levels below the
// walk's start. Frames [0, F) live in LDS; with kDeep, frames [F, kLevels)
// live in a per-group global scratch area (trees deeper than F levels).
template <typename Real, int F, bool kDeep>
struct WaveLds {
  static constexpr int kFrames = F;
  static constexpr bool kDeepFrames = kDeep;
  using V4 = typename Vec4T<Real>::T;
  uint32_t fr[F][kWave];  // child ranges: (first << 3) | (count - 1)
  unsigned long long tot[2];    // interactions of the wavefront's units so far
  V4 pp[kBuf<Real>];                  // x, y, z (relative to the target centre), m
  PcRing<Real> pc;
};

__device__ inline float rsq(float x) { return __builtin_amdgcn_rsqf(x); }
__device__ inline double rsq(double x) { return rsqrt(x); }
__device__ inline float fmaR(float a, float b, float c) { return fmaf(a, b, c); }
__device__ inline double fmaR(double a, double b, double c) { return fma(a, b, c); }

// Per-lane acceleration accumulator. The FP32 walk sums each batch in plain
// FP32 and adds the batch sums into FP64 accumulators: on CDNA4 an FP64 add
// issues at the FP32 rate, so this takes 6 instructions per batch sum where
// Kahan-compensated FP32 took 12, in the same 6 registers, with a smaller
// error. The FP64 walk adds in FP64 throughout.
template <typename Real>
struct Acc {
  double x = 0.0, y = 0.0, z = 0.0;
  __device__ inline void add(Real bx, Real by, Real bz) {
    x += static_cast<double>(bx);
    y += static_cast<double>(by);
    z += static_cast<double>(bz);
  }
  __device__ inline double sx() const { return x; }
  __device__ inline double sy() const { return y; }
  __device__ inline double sz() const { return z; }
};

// Wave64 inclusive scans on DPP (row shifts within 16-lane rows, then the
// row broadcasts of lanes 15 and 31), no LDS round trips.
__device__ inline uint32_t wave_incl_add(uint32_t v) {
  int x = static_cast<int>(v);
  x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, false);  // row_shr:1
  x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, false);  // row_shr:2
  x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, false);  // row_shr:4
  x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, false);  // row_shr:8
  x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xa, 0xf, false);  // row_bcast:15
  x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xc, 0xf, false);  // row_bcast:31
  return static_cast<uint32_t>(x);
}
// The lanes where p holds: a comparison's mask as it is (__ballot makes it a
// value per lane first and compares again).
__device__ inline uint64_t ballot(bool p) { return __builtin_amdgcn_ballot_w64(p); }
// Set bits of mask below this lane.
__device__ inline uint32_t rank_of(uint64_t mask) {
  return __builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(mask >> 32),
                                   __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(mask), 0u));
}

__device__ inline uint32_t uniform(uint32_t v) { return __builtin_amdgcn_readfirstlane(v); }
// A wave-uniform double, held in scalar registers.
__device__ inline double uniform_d(double v) {
  const uint64_t b = __builtin_bit_cast(uint64_t, v);
  const uint32_t lo = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(b));
  const uint32_t hi = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(b >> 32));
  return __builtin_bit_cast(double, (static_cast<uint64_t>(hi) << 32) | lo);
}

// k_walk's arguments, read again from the kernel's argument segment (its first
// argument). A field used here and there costs two scalar registers from the
// kernel's start to its last use, and what does not fit is moved to and from
// vector registers in the traversal's loop: all but the loop's own fields are
// read where they are used (spilled scalar registers 112 -> 44; walk of 65,536
// particles in FP64 0.525 -> 0.515 ms, 250,007 0.88 -> 0.865, 1M 1.325 -> 1.305).
// Only a kernel has the segment's address, so every function on the way from
// k_walk to here is inlined by force.
using LateArgs = const __attribute__((address_space(4))) WalkArgs;
__device__ __forceinline__ LateArgs& late_args() {
  LateArgs* p = (LateArgs*)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(p));
  return *p;
}

// A walk box (FP64): lo x, y, z, hi x, y, z.
struct Box6 {
  double v[6];
};

template <typename Real>
__device__ inline typename Vec4T<Real>::T make_entry(double x, double y, double z, double m) {
  using V4 = typename Vec4T<Real>::T;
  V4 v;
  v.x = static_cast<Real>(x);
  v.y = static_cast<Real>(y);
  v.z = static_cast<Real>(z);
  v.w = static_cast<Real>(m);
  return v;
}

// One particle (or monopole) interaction (grouped_ttg.h:137-153).
template <typename Real, bool kMask, typename V4>
__device__ inline void pp_term(const V4& q, Real tx, Real ty, Real tz, Real eps2, Real& bx, Real& by, Real& bz) {
  const Real dx = q.x - tx, dy = q.y - ty, dz = q.z - tz;
  const Real r2 = fmaR(dx, dx, fmaR(dy, dy, fmaR(dz, dz, eps2)));
  Real inv = rsq(r2);
  if (kMask) inv = r2 > Real(0) ? inv : Real(0);
  const Real s3 = q.w * inv * inv * inv;
  bx = fmaR(s3, dx, bx);
  by = fmaR(s3, dy, by);
  bz = fmaR(s3, dz, bz);
}

// Monopole + traceless quadrupole of one cell (multipole.h:171-200):
// a = M d / r^3 - Q.d / r^5 + 2.5 (d.Q.d) d / r^7, evaluated as
// r^-5 (d (M r^2 + 2.5 (d.Q.d) / r^2) - Q.d) with the softened r^2.
template <typename V4, typename V2, typename Real>
__device__ inline void p2c_term(const V4& e0, const V4& e1, const V2& e2, Real tx, Real ty, Real tz, Real eps2,
                                Real& bx, Real& by, Real& bz) {
  const Real dx = e0.x - tx, dy = e0.y - ty, dz = e0.z - tz;
  const Real r2 = fmaR(dx, dx, fmaR(dy, dy, fmaR(dz, dz, eps2)));
  const Real inv = rsq(r2);
  const Real inv2 = inv * inv;
  const Real inv5 = (inv * inv2) * inv2;
  // Q.d with Q = {xx, yy, zz, xy, xz, yz} = {e1.x, e1.y, e1.z, e1.w, e2.x, e2.y}
  const Real qx = fmaR(e1.x, dx, fmaR(e1.w, dy, e2.x * dz));
  const Real qy = fmaR(e1.w, dx, fmaR(e1.y, dy, e2.y * dz));
  const Real qz = fmaR(e2.x, dx, fmaR(e2.y, dy, e1.z * dz));
  const Real dqd = fmaR(dx, qx, fmaR(dy, qy, dz * qz));
  const Real g = fmaR(Real(2.5) * dqd, inv2, e0.w * r2);
  bx = fmaR(inv5, fmaR(g, dx, -qx), bx);
  by = fmaR(inv5, fmaR(g, dy, -qy), by);
  bz = fmaR(inv5, fmaR(g, dz, -qz), bz);
}

// How a batch of n entries is shared by S slices: slice s takes q or q + 1
// consecutive entries, the first n - q S slices the longer share. No entry
// is padding, and only the last round of the longer shares is divergent.
struct Share {
  uint32_t slices, inv;  // inv = ceil(2^16 / slices): n * inv >> 16 = n / slices for n <= kBuf
  uint32_t s;            // this lane's slice
  __device__ inline void setup(uint32_t S, uint32_t slice) {
    slices = S;
    inv = (65536u + S - 1) / S;
    s = slice;
  }
  __device__ inline void of(uint32_t n, int* q, int* first, bool* more) const {
    const uint32_t w = (n * inv) >> 16, r = n - w * slices;
    *q = static_cast<int>(w);
    *first = static_cast<int>(s * w + (s < r ? s : r));
    *more = s < r;
  }
};

// Entries [j0, j0 + n) of a batch for the NC particles of this lane, added to
// the plain partial sums.
template <typename Real, bool kMask, int NC>
__device__ inline void eval_pp(const typename Vec4T<Real>::T* e, int n, const Real* gx, const Real* gy, const Real* gz,
                               Real eps2, Real* bx, Real* by, Real* bz) {
  constexpr int kU = NC == 1 ? 4 : 2;
#pragma unroll kU
  for (int j = 0; j < n; ++j) {
    const auto q = e[j];
#pragma unroll
    for (int k = 0; k < NC; ++k) pp_term<Real, kMask>(q, gx[k], gy[k], gz[k], eps2, bx[k], by[k], bz[k]);
  }
}
template <typename Real, int NC>
__device__ inline void eval_pc(const PcRing<Real>& r, int j0, int n, const Real* gx, const Real* gy, const Real* gz,
                               Real eps2, Real* bx, Real* by, Real* bz) {
  constexpr int kU = NC == 1 && sizeof(Real) == 4 ? 2 : 1;
#pragma unroll kU
  for (int j = 0; j < n; ++j) {
    const auto e0 = r.a[j0 + j];
    const auto e1 = r.b[j0 + j];
    const auto e2 = r.c[j0 + j];
#pragma unroll
    for (int k = 0; k < NC; ++k) p2c_term(e0, e1, e2, gx[k], gy[k], gz[k], eps2, bx[k], by[k], bz[k]);
  }
}

// Evaluator of a target's particles: lane = (particle p, slice s). Batches
// are summed in walk precision and folded into the lane's FP64 accumulator
// before it has summed more than kFoldEntries entries (or one batch's, if those
// are more: 56 of 111 in two slices). (Pieces of targets of
// 33 to 128 particles come here, too: with twice as many entries a sum, the
// median error of 4,096 particles at target size 128 was 1.25 times what the
// group evaluator's sums of one batch gave; now 0.91 times. The walk of 4,096
// particles at target size 64 takes 143.9 us for it instead of 143.6.)
//
// Small targets are bound by latency, not by issue: with 9 particles and 7
// slices a 48-entry batch is 7 entries per lane, and moving the left-over
// entries of the ring to its front took as long as evaluating them. So a
// batch takes everything that is staged (48 to 111 entries, in FP64 22 to 85:
// fewer batches, no move), at any split into slices (Share). 65,536 particles in
// 16-particle units, walk 0.282 -> 0.268 ms; 1M uniform 1.58 -> 1.50.
template <typename Real, bool kMask>
struct TargetEval {
  using V4 = typename Vec4T<Real>::T;
  static constexpr int kFoldEntries = sizeof(Real) == 4 ? kBatch<Real> : 2 * kBatch<Real>;
  // a batch takes all that is staged
  static constexpr bool kTakesAll = true;
  __device__ static inline uint32_t take(uint32_t n) { return n; }
  Real tx, ty, tz, eps2;
  Share sh;
  bool active;
  int pending = 0;
  Real px = 0, py = 0, pz = 0;
  Acc<Real> acc;
  __device__ inline void fold() {
    acc.add(px, py, pz);
    px = py = pz = 0;
    pending = 0;
  }
  __device__ inline void count(int q) {
    pending += q + 1;
    if (pending > kFoldEntries) {
      fold();
      pending = q + 1;
    }
  }
  __device__ inline void pp(const V4* ring, uint32_t n) {
    int q, j0;
    bool more;
    sh.of(n, &q, &j0, &more);
    count(q);
    if (active) {
      eval_pp<Real, kMask, 1>(ring + j0, q, &tx, &ty, &tz, eps2, &px, &py, &pz);
      if (more) pp_term<Real, kMask>(ring[j0 + q], tx, ty, tz, eps2, px, py, pz);
    }
  }
  __device__ inline void pc(const PcRing<Real>& r, uint32_t n) {
    int q, j0;
    bool more;
    sh.of(n, &q, &j0, &more);
    count(q);
    if (active) {
      eval_pc<Real, 1>(r, j0, q, &tx, &ty, &tz, eps2, &px, &py, &pz);
      if (more) p2c_term(r.a[j0 + q], r.b[j0 + q], r.c[j0 + q], tx, ty, tz, eps2, px, py, pz);
    }
  }
};

// Evaluator of a whole group (G <= 128 particles). Each lane has two
// particle slots; slot k of lane l holds particle base_k + l % P_k and takes
// slice l / P_k of S_k slices of each batch. Layouts, by G:
//   G <= 42      two slots, P = ceil(G / 2), S = 64 / P (one fused loop)
//   43 .. 53     slot 0: particles 0..31 in 2 slices; slot 1: the r = G - 32
//                others, S_1 = 64 / r
//   54 .. 64     one slot, P = 64, S = 1
//   65 .. 96     slot 0: particles 0..63, every entry; slot 1: the r = G - 64
//                others, S_1 = 64 / r
//   97 .. 128    two slots, P = 64, S = 1 (one fused loop)
// A lane's sum of a batch is folded into FP64 after at most kBatch entries;
// slices are summed in FP64 at the end. A batch takes whole folds and the
// rest of the ring moves to its front: the move is small beside 48 entries
// for up to 128 particles, and odd batches would cost a second, short fold
// each (64 systems of 65,536 at target size 96: 8.42 ms against 8.11).
template <typename Real, bool kMask>
struct GroupEval {
  using V4 = typename Vec4T<Real>::T;
  // a batch takes whole folds
  static constexpr bool kTakesAll = false;
  __device__ static inline uint32_t take(uint32_t n) { return n / kBatch<Real> * kBatch<Real>; }
  Real gx[kGroupChunks], gy[kGroupChunks], gz[kGroupChunks], eps2;
  int nc;          // slots in the fused loop (1 or 2)
  bool tail;       // slot 1 has a loop of its own
  bool on0, on1;   // this lane's slots hold a slice
  Share sh0, sh1;
  uint32_t base1, rows0, rows1;
  Acc<Real> acc[kGroupChunks];

  __device__ inline void setup(uint32_t G, int lane) {
    const uint32_t l = static_cast<uint32_t>(lane);
    tail = false;
    uint32_t S0 = 1, S1 = 1;
    if (G <= 42) {
      rows0 = rows1 = base1 = (G + 1) / 2;
      S0 = S1 = kWave / rows0;
      nc = 2;
    } else if (G <= 53) {
      nc = 1;
      tail = true;
      rows0 = base1 = 32;
      S0 = 2;
      rows1 = G - 32;
      S1 = kWave / rows1;
    } else if (G <= 64) {
      nc = 1;
      rows0 = rows1 = kWave;
      base1 = 0;
    } else if (G <= 96) {
      nc = 1;
      tail = true;
      rows0 = base1 = kWave;
      rows1 = G - kWave;
      S1 = kWave / rows1;
    } else {
      nc = 2;
      rows0 = rows1 = base1 = kWave;
    }
    sh0.setup(S0, l / rows0);
    sh1.setup(S1, l / rows1);
    on0 = sh0.s < S0;
    on1 = sh1.s < S1;
  }
  // the particle (index within the group, clamped to it) of slot k
  __device__ inline uint32_t particle(int k, int lane, uint32_t G) const {
    const uint32_t i = (k ? base1 : 0u) + static_cast<uint32_t>(lane) % (k ? rows1 : rows0);
    return i < G ? i : G - 1;
  }
  template <int NC, int K0>
  __device__ inline void pp_slots(const V4* ring, const Share& sh, uint32_t n) {
    int q, j0;
    bool more;
    sh.of(n, &q, &j0, &more);
    Real bx[NC], by[NC], bz[NC];
    for (;;) {
      const int c = q < kBatch<Real> ? q : kBatch<Real>;
#pragma unroll
      for (int k = 0; k < NC; ++k) bx[k] = by[k] = bz[k] = 0;
      eval_pp<Real, kMask, NC>(ring + j0, c, gx + K0, gy + K0, gz + K0, eps2, bx, by, bz);
      q -= c;
      j0 += c;
      if (q == 0) break;
#pragma unroll
      for (int k = 0; k < NC; ++k) acc[K0 + k].add(bx[k], by[k], bz[k]);
    }
    if (more) {
      const V4 e = ring[j0];
#pragma unroll
      for (int k = 0; k < NC; ++k)
        pp_term<Real, kMask>(e, gx[K0 + k], gy[K0 + k], gz[K0 + k], eps2, bx[k], by[k], bz[k]);
    }
#pragma unroll
    for (int k = 0; k < NC; ++k) acc[K0 + k].add(bx[k], by[k], bz[k]);
  }
  template <int NC, int K0>
  __device__ inline void pc_slots(const PcRing<Real>& r, const Share& sh, uint32_t n) {
    int q, j0;
    bool more;
    sh.of(n, &q, &j0, &more);
    Real bx[NC], by[NC], bz[NC];
    for (;;) {
      const int c = q < kBatch<Real> ? q : kBatch<Real>;
#pragma unroll
      for (int k = 0; k < NC; ++k) bx[k] = by[k] = bz[k] = 0;
      eval_pc<Real, NC>(r, j0, c, gx + K0, gy + K0, gz + K0, eps2, bx, by, bz);
      q -= c;
      j0 += c;
      if (q == 0) break;
#pragma unroll
      for (int k = 0; k < NC; ++k) acc[K0 + k].add(bx[k], by[k], bz[k]);
    }
    if (more) {
      const auto e0 = r.a[j0];
      const auto e1 = r.b[j0];
      const auto e2 = r.c[j0];
#pragma unroll
      for (int k = 0; k < NC; ++k)
        p2c_term(e0, e1, e2, gx[K0 + k], gy[K0 + k], gz[K0 + k], eps2, bx[k], by[k], bz[k]);
    }
#pragma unroll
    for (int k = 0; k < NC; ++k) acc[K0 + k].add(bx[k], by[k], bz[k]);
  }
  __device__ inline void pp(const V4* ring, uint32_t n) {
    if (nc == 2) {
      if (on0) pp_slots<2, 0>(ring, sh0, n);
    } else {
      if (on0) pp_slots<1, 0>(ring, sh0, n);
      if (tail && on1) pp_slots<1, 1>(ring, sh1, n);
    }
  }
  __device__ inline void pc(const PcRing<Real>& r, uint32_t n) {
    if (nc == 2) {
      if (on0) pc_slots<2, 0>(r, sh0, n);
    } else {
      if (on0) pc_slots<1, 0>(r, sh0, n);
      if (tail && on1) pc_slots<1, 1>(r, sh1, n);
    }
  }
};

// The depth-first walk of one box (a target's or a group's particles) over
// the node ranges `start` (global, packed (first << 3) | (count - 1)), or
// from the system's root when start is null. Accepted nodes and the
// particles of opened leaves are staged in the rings relative to (cx, cy,
// cz) and handed to ev in batches of kBatch to kBuf - 1 entries (fewer at the
// end).
//
// kGroup: a group's walk (grouped_ttg.h:259-276 at the group node): a node
// that is neither accepted nor rejected for every box inside
// (theta^2 * far2 > edge^2) is deferred: appended to dl, for its targets.
// Returns false when more than kDefer nodes would be deferred.
template <typename Real, bool kMask, bool kGroup, typename Eval, typename Lds>
__device__ bool traverse(const WalkArgs& a, Lds& L, uint32_t* gfr, const Box6& box, double cx, double cy, double cz,
                         uint32_t sys_id, const uint32_t* start, uint32_t n_start, bool use_quad, double theta2,
                         Eval& ev, uint32_t& n_pp, uint32_t& n_pc, uint32_t* dl, uint32_t& n_def) {
  constexpr int F = Lds::kFrames;
  constexpr int kStack = Lds::kDeepFrames ? kLevels : F;
  const int lane = __lane_id();
  const uint32_t last_node = a.n_nodes - 1, last_part = a.n_parts - 1;
  const double blo0 = uniform_d(box.v[0]), blo1 = uniform_d(box.v[1]), blo2 = uniform_d(box.v[2]);
  const double bhi0 = uniform_d(box.v[3]), bhi1 = uniform_d(box.v[4]), bhi2 = uniform_d(box.v[5]);
  cx = uniform_d(cx);
  cy = uniform_d(cy);
  cz = uniform_d(cz);
  theta2 = uniform_d(theta2);
  uint32_t pp_cnt = 0, pc_cnt = 0;
  bool ok = true;

  // Evaluate the first n staged entries and move the rest (fewer than
  // kBatch) to the front.
  auto flush_pp = [&](uint32_t n) {
    __builtin_amdgcn_wave_barrier();
    ev.pp(L.pp, n);
    pp_cnt -= n;
    if (!Eval::kTakesAll && pp_cnt) {
      typename Vec4T<Real>::T v;
      if (static_cast<uint32_t>(lane) < pp_cnt) v = L.pp[n + lane];
      __builtin_amdgcn_wave_barrier();
      if (static_cast<uint32_t>(lane) < pp_cnt) L.pp[lane] = v;
    }
    __builtin_amdgcn_wave_barrier();
  };
  auto flush_pc = [&](uint32_t n) {
    __builtin_amdgcn_wave_barrier();
    ev.pc(L.pc, n);
    pc_cnt -= n;
    if (!Eval::kTakesAll && pc_cnt) {
      typename Vec4T<Real>::T v0, v1;
      typename Vec2T<Real>::T v2;
      if (static_cast<uint32_t>(lane) < pc_cnt) {
        v0 = L.pc.a[n + lane];
        v1 = L.pc.b[n + lane];
        v2 = L.pc.c[n + lane];
      }
      __builtin_amdgcn_wave_barrier();
      if (static_cast<uint32_t>(lane) < pc_cnt) {
        L.pc.a[lane] = v0;
        L.pc.b[lane] = v1;
        L.pc.c[lane] = v2;
      }
    }
    __builtin_amdgcn_wave_barrier();
  };

  // lane d: ranges of frame d, and the next of them to pop
  uint32_t fr_n = start ? n_start : 1u, fr_cur = 0;
  if (lane == 0) L.fr[0][0] = sys_id << 3;  // the system's root: node sys_id, one node
  __builtin_amdgcn_wave_barrier();
  int depth = 0;
  while (depth >= 0) {
    const uint32_t nr = __builtin_amdgcn_readlane(fr_n, depth);
    const uint32_t cur = __builtin_amdgcn_readlane(fr_cur, depth);
    if (cur >= nr) {
      --depth;
      continue;
    }
    // Pop whole child ranges, up to 64 nodes. Range j covers slots
    // [excl_j, excl_j + count_j) and flags its first slot, so a slot's range
    // is the number of flags up to it less one: node = first_j + (slot -
    // excl_j). (The ranges themselves need not be ascending: children of
    // deferred nodes come in walk order.)
    const uint32_t rr = cur + lane;
    const bool rv = rr < nr;
    uint32_t node, total;
    if (depth == 0 && start) {
      // a deferred list: single nodes in walk order, one per lane
      node = rv ? (start[rr] >> 3) : 0u;
      total = nr - cur < kWave ? nr - cur : kWave;
      if (lane == 0) fr_cur = cur + total;
    } else {
      uint32_t packed = 0u;
      if constexpr (Lds::kDeepFrames) {
        if (rv) packed = depth < F ? L.fr[depth][rr] : gfr[(depth - F) * kWave + rr];
      } else {
        if (rv) packed = L.fr[depth][rr];
      }
      const uint32_t rcnt = rv ? (packed & 7u) + 1u : 0u;
      const uint32_t rfirst = packed >> 3;
      const uint32_t incl = wave_incl_add(rcnt);
      const bool taken = rv && incl <= kWave;
      const int k = __popcll(ballot(taken));
      total = uniform(__builtin_amdgcn_readlane(incl, k - 1));
      const uint32_t excl = incl - rcnt;
      // the other lanes flag slot 0, where range 0 starts
      const int own = __builtin_amdgcn_ds_permute(taken ? static_cast<int>(excl << 2) : 0, 1);
      if (lane == depth) fr_cur = cur + k;
      const int j = static_cast<int>(rank_of(ballot(own != 0))) + own - 1;
      node = static_cast<uint32_t>(__shfl(static_cast<int>(rfirst - excl), j)) + static_cast<uint32_t>(lane);
    }
    const bool nv = static_cast<uint32_t>(lane) < total;
    // MAC in FP64, reference operation order (multipole.h:130-160). Every
    // lane loads and tests a record (lanes past `total` lane 0's, a line
    // already being fetched) and the flags below drop the extra lanes: no
    // divergent branch.
    // The record's second half, {first, count, m, Qxx} and {Qyy, Qxy, Qxz,
    // Qyz}, comes with the MAC data, so accepted cells are staged from
    // registers without a second round trip to memory.
    const uint32_t node0 = uniform(node);
    const uint32_t nd = nv ? (node < last_node ? node : last_node) : (node0 < last_node ? node0 : last_node);
    const NodeRec* rp = &a.rec[nd];
    const uint4* rw = reinterpret_cast<const uint4*>(rp);
    const uint4 rw2 = rw[2];
    uint4 rw3 = make_uint4(0, 0, 0, 0);
    if constexpr (sizeof(Real) == 4) rw3 = rw[3];
    const double4 mac = make_double4(rp->cx, rp->cy, rp->cz, rp->edge2);
    bool defer = false;
    const double dx0 = fmax(fmax(blo0 - mac.x, mac.x - bhi0), 0.0);
    const double dx1 = fmax(fmax(blo1 - mac.y, mac.y - bhi1), 0.0);
    const double dx2 = fmax(fmax(blo2 - mac.z, mac.z - bhi2), 0.0);
    const double near2 = dx0 * dx0 + dx1 * dx1 + dx2 * dx2;
    const bool accept = theta2 * near2 > mac.w;
    if constexpr (kGroup) {
      // no deferred list (a target's walk through this evaluator): accept or open
      if (!accept && dl != nullptr) {
        const double fx0 = fmax(mac.x - blo0, bhi0 - mac.x);
        const double fx1 = fmax(mac.y - blo1, bhi1 - mac.y);
        const double fx2 = fmax(mac.z - blo2, bhi2 - mac.z);
        const double far2 = fx0 * fx0 + fx1 * fx1 + fx2 * fx2;
        defer = !(theta2 * far2 <= mac.w);
      }
    }
    const bool isleaf = (rw2.y >> 31) != 0;
    const uint32_t lfirst = rw2.x;
    const uint32_t lcnt = rw2.y & 0x7fffffffu;
    const bool cellf = nv && accept;
    const bool deff = nv && defer;
    const bool leaff = nv && !accept && !defer && isleaf;
    // An interior node to open needs a child and a free stack frame. The
    // launch sizes the stack for the tree's depth, so neither check fails on
    // a well-formed tree; if one does, the node is not opened and the step
    // reports an incomplete walk (the reference's missing > 0,
    // integrate_ttg.h:104-106).
    const bool openable = !isleaf && lcnt != 0u && depth + 1 < kStack && static_cast<uint32_t>(depth) + 1 < a.stack_limit;
    const bool openf = nv && !accept && !defer && !isleaf && openable;
    if (ballot(nv && !accept && !defer && !isleaf && !openable)) {
      if (lane == 0) atomicOr(&a.misc[kMiscIncomplete], 1u);
    }
    if constexpr (kGroup) {
      const uint64_t dm = ballot(deff);
      if (dm) {
        const uint32_t nd_new = __popcll(dm);
        if (n_def + nd_new > kDefer) {
          ok = false;
          break;
        }
        if (deff) dl[n_def + rank_of(dm)] = nd << 3;
        n_def += nd_new;
      }
    }
    // children of opened interior nodes -> frame depth + 1
    const uint64_t om = ballot(openf);
    if (om) {
      const uint32_t pos = rank_of(om);
      if constexpr (Lds::kDeepFrames) {
        if (depth + 1 < F) {
          if (openf) L.fr[depth + 1][pos] = (lfirst << 3) | (lcnt - 1u);
        } else {
          if (openf) gfr[(depth + 1 - F) * kWave + pos] = (lfirst << 3) | (lcnt - 1u);
          __threadfence_block();  // read back by other lanes
        }
      } else {
        if (openf) L.fr[depth + 1][pos] = (lfirst << 3) | (lcnt - 1u);
      }
      if (lane == depth + 1) {
        fr_n = __popcll(om);
        fr_cur = 0;
      }
    }
    // accepted nodes
    const uint64_t cm = ballot(cellf);
    if (cm) {
      const uint32_t nc = __popcll(cm);
      const uint32_t pos = rank_of(cm);
      if (use_quad) {
        if (cellf) {
          const uint32_t slot = pc_cnt + pos;
          if constexpr (sizeof(Real) == 4) {
            const float qxx = __uint_as_float(rw2.w), qyy = __uint_as_float(rw3.x);
            L.pc.a[slot] = make_entry<Real>(mac.x - cx, mac.y - cy, mac.z - cz, __uint_as_float(rw2.z));
            L.pc.b[slot] = make_float4(qxx, qyy, -(qxx + qyy), __uint_as_float(rw3.y));
            L.pc.c[slot] = make_float2(__uint_as_float(rw3.z), __uint_as_float(rw3.w));
          } else {
            const double* q = &a.q64[8 * nd];
            L.pc.a[slot] = make_entry<Real>(mac.x - cx, mac.y - cy, mac.z - cz, q[0]);
            L.pc.b[slot] = make_double4(q[1], q[2], q[3], q[4]);
            L.pc.c[slot] = make_double2(q[5], q[6]);
          }
        }
        pc_cnt += nc;
        n_pc += nc;
        if (pc_cnt >= kBatch<Real>) flush_pc(Eval::take(pc_cnt));
      } else {
        if (cellf) {
          const double m = sizeof(Real) == 4 ? static_cast<double>(__uint_as_float(rw2.z)) : a.q64[8 * nd];
          L.pp[pp_cnt + pos] = make_entry<Real>(mac.x - cx, mac.y - cy, mac.z - cz, m);
        }
        pp_cnt += nc;
        n_pp += nc;
        if (pp_cnt >= kBatch<Real>) flush_pp(Eval::take(pp_cnt));
      }
    }
    // particles of opened leaves, mapped to slots like the nodes: the leaves'
    // offsets move to the first lanes, where a slot's count of flags finds them
    const uint64_t lm = ballot(leaff);
    if (lm) {
      const uint32_t lc = leaff ? lcnt : 0u;
      const uint32_t lincl = wave_incl_add(lc);
      const uint32_t lexcl = lincl - lc;
      const uint32_t ltot = uniform(__builtin_amdgcn_readlane(lincl, 63));
      // (lanes without a leaf write the last lane, which then holds none)
      const int from = __builtin_amdgcn_ds_permute(static_cast<int>((leaff ? rank_of(lm) : 63u) << 2),
                                                   static_cast<int>(lfirst - lexcl));
      for (uint32_t b = 0; b < ltot; b += kWave) {
        // leaves that start at or before slot b
        const int before = __popcll(ballot(leaff && lexcl <= b));
        const uint32_t e = b + lane;
        // each leaf that starts later in this chunk flags its first slot; the
        // other lanes clear slot 0
        const bool here = leaff && lexcl > b && lexcl < b + kWave;
        const int own = __builtin_amdgcn_ds_permute(here ? static_cast<int>((lexcl - b) << 2) : 0, here ? 1 : 0);
        const int jj = before - 1 + static_cast<int>(rank_of(ballot(own != 0))) + own;
        uint32_t q = static_cast<uint32_t>(__shfl(from, jj)) + e;
        q = q < last_part ? q : last_part;
        const uint32_t chunk = ltot - b < kWave ? ltot - b : kWave;
        if (e < ltot) {
          const double4 sp = a.posm[q];
          L.pp[pp_cnt + lane] = make_entry<Real>(sp.x - cx, sp.y - cy, sp.z - cz, sp.w);
        }
        pp_cnt += chunk;
        n_pp += chunk;
        if (pp_cnt >= kBatch<Real>) flush_pp(Eval::take(pp_cnt));
      }
    }
    __builtin_amdgcn_wave_barrier();
    if (om) ++depth;
  }
  if (!ok) return false;
  // the last, smaller batches
  if (pp_cnt) flush_pp(pp_cnt);
  if (pc_cnt) flush_pc(pc_cnt);
  __builtin_amdgcn_wave_barrier();
  return true;
}

__device__ inline double wave_min(double v) {
  for (int o = 32; o > 0; o >>= 1) v = fmin(v, __shfl_xor(v, o));
  return v;
}
__device__ inline double wave_max(double v) {
  for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o));
  return v;
}

// FP64 bounding box of particles [b, b + n) (multipole.h:115-128).
__device__ inline Box6 particle_box(const WalkArgs& a, uint32_t b, uint32_t n) {
  const double inf = __builtin_huge_val();
  double lo0 = inf, lo1 = inf, lo2 = inf, hi0 = -inf, hi1 = -inf, hi2 = -inf;
  for (uint32_t p = __lane_id(); p < n; p += kWave) {
    const double4 q = a.posm[b + p];
    lo0 = fmin(lo0, q.x);
    lo1 = fmin(lo1, q.y);
    lo2 = fmin(lo2, q.z);
    hi0 = fmax(hi0, q.x);
    hi1 = fmax(hi1, q.y);
    hi2 = fmax(hi2, q.z);
  }
  Box6 box;
  box.v[0] = uniform_d(wave_min(lo0));
  box.v[1] = uniform_d(wave_min(lo1));
  box.v[2] = uniform_d(wave_min(lo2));
  box.v[3] = uniform_d(wave_max(hi0));
  box.v[4] = uniform_d(wave_max(hi1));
  box.v[5] = uniform_d(wave_max(hi2));
  return box;
}

// A node's particle box as computed by the upward pass.
__device__ __forceinline__ Box6 node_box(uint32_t node) {
  const double* p = late_args().nbox + 6 * uint64_t(node);
  Box6 box;
#pragma unroll
  for (int k = 0; k < 6; ++k) box.v[k] = p[k];
  return box;
}

// The end of one target particle's walk: its FP64 sums plus the group's
// share (gacc, when given), times G, to the outputs (grouped_ttg.h:63-66,
// the update callback) and the fused kick/drift.
__device__ __forceinline__ void finish_particle(uint32_t k3, double ax, double ay, double az,
                                       const double* gacc, double sys_G, double kick_dt, double drift_dt,
                                       uint32_t n_pp, uint32_t n_pc) {
  const LateArgs& a = late_args();
  if (gacc) {
    ax += gacc[3 * uint64_t(k3) + 0];
    ay += gacc[3 * uint64_t(k3) + 1];
    az += gacc[3 * uint64_t(k3) + 2];
  }
  const double gx = sys_G * ax, gy = sys_G * ay, gz = sys_G * az;
  if (a.acc) {
    a.acc[3 * uint64_t(k3) + 0] = gx;
    a.acc[3 * uint64_t(k3) + 1] = gy;
    a.acc[3 * uint64_t(k3) + 2] = gz;
  }
  if (a.n_pp) a.n_pp[k3] = n_pp;
  if (a.n_pc) a.n_pc[k3] = n_pc;
  if (a.parts) {
    // kick_one / drift_one (integrate.h:15-16): v += a*dt; x += v*dt. The
    // particle comes from the unsorted input (src at perm) when given: the
    // whole Morton-ordered record is written here, not by the sort's gather.
    bh_particle pt = a.src ? a.src[a.perm[k3]] : a.parts[k3];
    const double vx = pt.vel[0] + gx * kick_dt;
    const double vy = pt.vel[1] + gy * kick_dt;
    const double vz = pt.vel[2] + gz * kick_dt;
    pt.vel[0] = vx;
    pt.vel[1] = vy;
    pt.vel[2] = vz;
    if (drift_dt != 0.0) {
      pt.pos[0] = pt.pos[0] + vx * drift_dt;
      pt.pos[1] = pt.pos[1] + vy * drift_dt;
      pt.pos[2] = pt.pos[2] + vz * drift_dt;
    }
    a.parts[k3] = pt;
    if (a.carry) {
      // the next step's build reads these instead of the records (x, y, z
      // and m in blocks of n_parts)
      const uint64_t np = a.n_parts;
      a.carry[k3] = pt.pos[0];
      a.carry[np + k3] = pt.pos[1];
      a.carry[2 * np + k3] = pt.pos[2];
      a.carry[3 * np + k3] = pt.mass;
      if (!(isfinite(pt.pos[0]) && isfinite(pt.pos[1]) && isfinite(pt.pos[2]) && isfinite(vx) && isfinite(vy) &&
            isfinite(vz) && isfinite(pt.mass)))
        atomicOr(a.carry_bad, 1u);
    }
  }
}

// Targets of at least kWideMin particles use the group evaluator (its
// layouts cover 33 to kGroupCap particles, two slots per lane); smaller ones
// use lane = (particle, slice).
constexpr uint32_t kWideMin = 33;

// Particles [tb, tb + T) of a target (node tnode; the whole of it or a piece,
// at most 32 particles) with the target evaluator: the walk over `start` (the
// group's deferred nodes) or from the root with the target's box, then the
// slices' sums, plus the group's share (gacc, counts g_pp / g_pc) when given.
template <typename Real, bool kMask, typename Lds>
__device__ __forceinline__ void walk_target(const WalkArgs& a, Lds& L, uint32_t* gfr, uint32_t tnode, uint32_t tb, uint32_t T,
                            const uint32_t* start, uint32_t n_start, const double* gacc, uint32_t g_pp, uint32_t g_pc,
                            unsigned long long& tot_pp, unsigned long long& tot_pc) {
  const int lane = __lane_id();
  const LateArgs& la = late_args();
  const uint32_t sys_id = uniform(la.sid[tb]);
  const SysDev& sp = la.sys[sys_id];
  const bool use_quad = sp.use_quad != 0;
  const double4 tcv = la.ctr[tnode];
  const double tcx = tcv.x, tcy = tcv.y, tcz = tcv.z;
  const Box6 box = node_box(tnode);

  const int S = kWave / static_cast<int>(T);
  TargetEval<Real, kMask> ev;
  ev.sh.setup(static_cast<uint32_t>(S), static_cast<uint32_t>(lane) / T);
  ev.active = lane < static_cast<int>(T) * S;
  ev.eps2 = static_cast<Real>(sp.eps2);
  {
    const double4 q = a.posm[tb + lane % static_cast<int>(T)];
    ev.tx = static_cast<Real>(q.x - tcx);
    ev.ty = static_cast<Real>(q.y - tcy);
    ev.tz = static_cast<Real>(q.z - tcz);
  }
  uint32_t n_pp = 0, n_pc = 0, n_def = 0;
  traverse<Real, kMask, false>(a, L, gfr, box, tcx, tcy, tcz, sys_id, start, n_start, use_quad, sp.theta2, ev, n_pp,
                               n_pc, nullptr, n_def);
  n_pp += g_pp;
  n_pc += g_pc;
  ev.fold();
  // combine slices in FP64 (the P2C ring is free now)
  double* red = reinterpret_cast<double*>(L.pc.a);  // 3 x 64 doubles
  if (ev.active) {
    red[3 * lane + 0] = ev.acc.sx();
    red[3 * lane + 1] = ev.acc.sy();
    red[3 * lane + 2] = ev.acc.sz();
  }
  __builtin_amdgcn_wave_barrier();
  if (lane < static_cast<int>(T)) {
    double ax = 0.0, ay = 0.0, az = 0.0;
    for (int k2 = 0; k2 < S; ++k2) {
      const int src = k2 * static_cast<int>(T) + lane;
      ax += red[3 * src + 0];
      ay += red[3 * src + 1];
      az += red[3 * src + 2];
    }
    finish_particle(tb + lane, ax, ay, az, gacc, sp.G, sp.kick_dt, sp.drift_dt, n_pp, n_pc);
  }
  tot_pp += static_cast<unsigned long long>(n_pp) * T;
  tot_pc += static_cast<unsigned long long>(n_pc) * T;
  __builtin_amdgcn_wave_barrier();
}

// The target that holds particle p of a unit that starts at particle gb: the
// last mark at or before p (a unit of several targets spans at most kGroupCap
// particles).
__device__ __forceinline__ uint32_t covering_target(uint32_t gb, uint32_t p) {
  for (uint32_t back = 0;; back += kWave) {
    const uint32_t d = back + __lane_id();
    const uint32_t m = d <= p - gb ? late_args().tmark[p - d] : 0u;
    const uint64_t have = ballot(m != 0);
    if (have) return uniform(__builtin_amdgcn_readlane(m, __ffsll(static_cast<long long>(have)) - 1)) - 1u;
    if (back + kWave > p - gb) return 0u;  // not reached: a unit's first particle begins a target
  }
}

// Where the cut at particle p of such a unit lies.
__device__ __forceinline__ uint32_t cut_place(uint32_t gb, uint32_t p, uint32_t target_piece) {
  const uint32_t node = covering_target(gb, p);
  const uint32_t b = uniform(late_args().begin[node]), n = uniform(late_args().count[node]);
  return b == p || n > target_piece ? p : b + n;
}

// One walk unit starting at node g: a walk group (topmost node with leaf ||
// count <= max(tsm, 128)) or a run of sibling single-target groups packed
// into one unit (unit_n). A group that is itself a target walks as one.
// Otherwise the wave walks the tree once for the unit's box - the decisions
// every target inside shares - evaluating the shared list for all the
// unit's particles and keeping the deferred nodes; then each target of the
// unit walks only those.
//
// A unit of more particles than its kind's piece is walked in pieces, one
// wavefront each (p0: this piece's place). A piece does the unit's walks, with
// the unit's box and centre or the target's, for its own particles: every
// pair is computed from the same rounded coordinates however a unit is cut.
// A cut that falls inside a target of at most target_piece particles moves
// to its end.
//
// The unit's work is a sequence of jobs: the group's shared walk (if any),
// then its targets in particle order; a unit that is one target, or a piece
// of one, is one job. The group's walk and
// targets of 33 particles or more use the group evaluator (its layouts keep
// the lanes busy for those sizes, and a target of 65-128 particles walks
// once, not once per 64) through one call of its traversal; smaller targets
// use the target evaluator. Deferral is off for target jobs (no deferred
// list): their decisions are accept or open.
template <typename Real, bool kMask, typename Lds>
__device__ __forceinline__ void walk_group(const WalkArgs& a, Lds& L, uint32_t slot, uint32_t g, uint32_t p0) {
  const int lane = __lane_id();
  const uint32_t gb = uniform(late_args().begin[g]);
  // a unit packed from sibling single-target groups spans several nodes
  const uint32_t un = late_args().unit_n ? uniform(late_args().unit_n[g]) : 0u;
  const bool packed = (un >> 31) != 0;
  const uint32_t G = packed ? un & 0x7fffffffu : uniform(late_args().count[g]);
  const uint32_t sys_id = uniform(late_args().sid[gb]);
  const SysDev& sp = late_args().sys[sys_id];
  const bool gleaf = (a.rec[g].count >> 31) != 0;
  uint32_t* gfr = Lds::kDeepFrames ? late_args().deep_frames + uint64_t(slot) * (kLevels - Lds::kFrames) * kWave : nullptr;
  const bool single = !packed && (gleaf || G <= sp.tsm || G > kGroupCap);
  uint32_t* dl = late_args().defer + uint64_t(slot) * kDefer;
  uint32_t g_pp = 0, g_pc = 0, n_def = 0;
  bool ok = false;  // the group's shared walk kept all its deferred nodes
  unsigned long long tot_pp = 0, tot_pc = 0;
  // this piece's particles [r0, r1)
  uint32_t r0 = p0, r1;
  {
    const uint32_t len = piece_size(G, single ? sp.target_piece : sp.unit_piece), left = gb + G - p0;
    r1 = p0 + (len < left ? len : left);
    if (!single) {
      if (r0 > gb) r0 = cut_place(gb, r0, sp.target_piece);
      if (r1 < gb + G) r1 = cut_place(gb, r1, sp.target_piece);
      if (r0 >= r1) return;
    }
  }
  bool group_job = !single;
  uint32_t b0 = r0;   // first particle of the next target job
  uint32_t c = r0;    // next 64-particle chunk of the piece to scan for targets
  uint64_t bits = 0;  // targets of the scanned chunk not yet walked
  uint32_t m = 0;     // this lane's mark in the scanned chunk
  for (;;) {
    // the next job: the group's walk, the unit's one target or a target node
    // (the piece's first may have begun before it)
    bool is_group = false;
    uint32_t tnode = g, jb = r0, size = r1 - r0;
    if (group_job) {
      is_group = true;
      group_job = false;
    } else if (b0 >= r1) {
      break;
    } else if (single) {
      b0 = r1;
    } else {
      if (b0 == r0) {
        tnode = covering_target(gb, r0);
        c = r0 + 1;
      } else {
        while (!bits && c < r1) {
          const uint32_t i = c + lane;
          m = i < r1 ? late_args().tmark[i] : 0u;
          bits = ballot(m != 0);
          c += kWave;
        }
        if (!bits) break;  // not reached: targets fill the unit
        const int j = __ffsll(static_cast<long long>(bits)) - 1;
        bits &= bits - 1;
        tnode = uniform(__builtin_amdgcn_readlane(m, j)) - 1u;
      }
      jb = b0;
      const uint32_t e = uniform(late_args().begin[tnode]) + uniform(late_args().count[tnode]);
      b0 = e < r1 ? e : r1;
      size = b0 - jb;
    }
    const uint32_t* start = ok ? dl : nullptr;
    const uint32_t n_start = ok ? n_def : 0u;
    const double* gacc = ok ? late_args().gacc : nullptr;
    const uint32_t jpp = ok ? g_pp : 0u, jpc = ok ? g_pc : 0u;
    if (!is_group && size < kWideMin) {
      walk_target<Real, kMask>(a, L, gfr, tnode, jb, size, start, n_start, gacc, jpp, jpc, tot_pp, tot_pc);
      continue;
    }
    // group evaluator: the group's shared walk or 33-128 particles of a target
    // a packed unit's box and the origin of its relative coordinates (the
    // box centre); a group's or target's: its node box and centre
    const bool pbox = is_group && packed;
    const Box6 box = pbox ? particle_box(a, gb, G) : node_box(tnode);
    const double4 ccv = pbox ? make_double4(0.5 * (box.v[0] + box.v[3]), 0.5 * (box.v[1] + box.v[4]),
                                            0.5 * (box.v[2] + box.v[5]), 0.0)
                             : late_args().ctr[tnode];
    GroupEval<Real, kMask> ev;
    ev.setup(size, lane);
    ev.eps2 = static_cast<Real>(sp.eps2);
#pragma unroll
    for (int k = 0; k < kGroupChunks; ++k) {
      const double4 q = a.posm[jb + ev.particle(k, lane, size)];
      ev.gx[k] = static_cast<Real>(q.x - ccv.x);
      ev.gy[k] = static_cast<Real>(q.y - ccv.y);
      ev.gz[k] = static_cast<Real>(q.z - ccv.z);
    }
    uint32_t n_pp = 0, n_pc = 0, j_def = 0;
    const bool walked = traverse<Real, kMask, true>(a, L, gfr, box, ccv.x, ccv.y, ccv.z, sys_id,
                                                    is_group ? nullptr : start, is_group ? 0u : n_start,
                                                    sp.use_quad != 0, sp.theta2, ev, n_pp, n_pc,
                                                    is_group ? dl : nullptr, j_def);
    if (is_group) {
      ok = walked;
      g_pp = n_pp;
      g_pc = n_pc;
      n_def = j_def;
      if (!ok) continue;  // the targets walk from the root
    } else {
      n_pp += jpp;
      n_pc += jpc;
    }
    // per-particle sums: each slot's slices added in FP64 through LDS (the
    // P2C ring is free after the walk); the group's are stored for its
    // targets, a target's finish its particles
    double* red = reinterpret_cast<double*>(L.pc.a);  // 3 x 64 doubles
    const int used = ev.nc == 2 || ev.tail ? 2 : 1;
#pragma unroll
    for (int k = 0; k < kGroupChunks; ++k) {
      if (k < used) {
        const uint32_t P = k ? ev.rows1 : ev.rows0, S = k ? ev.sh1.slices : ev.sh0.slices;
        red[3 * lane + 0] = ev.acc[k].sx();
        red[3 * lane + 1] = ev.acc[k].sy();
        red[3 * lane + 2] = ev.acc[k].sz();
        __builtin_amdgcn_wave_barrier();
        const uint32_t i = (k ? ev.base1 : 0u) + static_cast<uint32_t>(lane);
        if (static_cast<uint32_t>(lane) < P && i < size) {
          double ax = 0.0, ay = 0.0, az = 0.0;
          for (uint32_t s2 = 0; s2 < S; ++s2) {
            const uint32_t src = s2 * P + static_cast<uint32_t>(lane);
            ax += red[3 * src + 0];
            ay += red[3 * src + 1];
            az += red[3 * src + 2];
          }
          if (is_group) {
            late_args().gacc[3 * uint64_t(jb + i) + 0] = ax;
            late_args().gacc[3 * uint64_t(jb + i) + 1] = ay;
            late_args().gacc[3 * uint64_t(jb + i) + 2] = az;
          } else {
            finish_particle(jb + i, ax, ay, az, gacc, sp.G, sp.kick_dt, sp.drift_dt, n_pp, n_pc);
          }
        }
        __builtin_amdgcn_wave_barrier();
      }
    }
    if (is_group) {
      // the deferred list and the group sums are read back by other lanes
      __threadfence_block();
    } else {
      tot_pp += static_cast<unsigned long long>(n_pp) * size;
      tot_pc += static_cast<unsigned long long>(n_pc) * size;
    }
  }
  if (lane == 0) {
    L.tot[0] += tot_pp;
    L.tot[1] += tot_pc;
  }
}

// A fixed grid of workgroups (one wavefront each) takes the walk units from
// eight queues. Workgroup b runs on XCD b % 8 and takes units from queue
// b % 8, which holds the eighth [x U / 8, (x + 1) U / 8) of the U units
// (Morton order): each XCD walks a contiguous run, so neighbouring units
// share its L2, and within an XCD the units go to whichever wavefront is
// free. A wavefront whose queue is past its end goes on with the queue that
// has most units left, and leaves once none has any; a head only grows, so
// every wavefront exits. Equal shares of the units are not equal shares of the
// work: of 64 systems of different sizes the XCDs needed 16 to 39 ms, now all
// 26.4; 16M 38.7 -> 38.2, 4M 10.2 -> 10.0. The heads lie a cache line apart and
// are looked at before a claim: next to each other, and claimed to find out
// that a queue is empty, they took 0.3 ms more at 1M. The unit count and the
// heads are on the device (counted and cleared by the step), so the launch
// needs no host read.
//
// Device-scope atomics on one address from many wavefronts queue up behind
// each other (measured inside this kernel at 65,536 particles: a claim 27,000
// cycles while all wavefronts start, the unit's two total counters 44,000 to
// 115,000 cycles when a few thousand small units end in a row, a unit itself
// 160,000). So a wavefront's first unit is its own place in the queue (the
// head counts the units after those), and its interaction totals are summed
// in LDS and added once, when it leaves. Many small systems gain most: 2,000
// of 1,000 particles in 16-particle units, walk 4.14 -> 2.00 ms.
template <typename Real, int kWaves, bool kMask, bool kDeep>
__global__ __launch_bounds__(kWaves * 64) __attribute__((amdgpu_waves_per_eu(4))) void k_walk(WalkArgs a) {
  __shared__ WaveLds<Real, kShallowFrames, kDeep> lds[kWaves];
  static_assert(kWaves == 1, "one wavefront per workgroup: the queues hand out units per workgroup");
  stamp(a.misc, kStampWalk);
  if (a.misc[kMiscNonfinite] | a.misc[kMiscAbort]) return;
  const uint32_t units = a.misc[kMiscGroups];
  auto& L = lds[0];
  if (__lane_id() == 0) L.tot[0] = L.tot[1] = 0ull;
  __builtin_amdgcn_wave_barrier();
  const uint32_t first = gridDim.x >> 3;
  // queue q's units: [lo, lo + len)
  uint32_t q = blockIdx.x & 7u, lo, len;
  const auto part = [&](uint32_t p) { return static_cast<uint32_t>(uint64_t(units) * p / 8); };
  lo = part(q);
  len = part(q + 1) - lo;
  // Every lane takes part in the claim (adding 1 for lane 0, 0 for the
  // others) and the unit is read from lane 0's result: no branch on the
  // lane id inside the loop, so all 64 lanes stay together in it (a
  // lane-0-only claim lets the compiler keep the other lanes looping on
  // their own, with a stale claim).
  const auto claim = [&]() __attribute__((always_inline)) {
    const uint32_t mine = atomicAdd(&late_args().queue[kQueueStride * q], __lane_id() == 0 ? 1u : 0u);
    return first + uniform(__builtin_amdgcn_readlane(mine, 0));
  };
  uint32_t k = blockIdx.x >> 3;
  for (;;) {
    while (k >= len) {
      // the queue with most units left, if any is: lane p looks at queue p
      const uint32_t p = __lane_id() & 7u, n = part(p + 1) - part(p);
      uint32_t left = 0;
      if (n > first) {
        const uint32_t h = __hip_atomic_load(&late_args().queue[kQueueStride * p], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        left = h < n - first ? n - first - h : 0u;
      }
      uint32_t most = left << 3 | p;
      for (int o = 4; o > 0; o >>= 1) most = max(most, static_cast<uint32_t>(__shfl_xor(static_cast<int>(most), o)));
      most = uniform(most);
      if (most < 8u) break;
      q = most & 7u;
      lo = part(q);
      len = part(q + 1) - lo;
      k = claim();
    }
    if (k >= len) break;
    const uint2 u = late_args().units[lo + k];
    walk_group<Real, kMask>(a, L, blockIdx.x, uniform(u.x), uniform(u.y));
    k = claim();
  }
  if (__lane_id() == 0 && (L.tot[0] | L.tot[1]) != 0ull) {
    atomicAdd(&late_args().totals[0], L.tot[0]);
    atomicAdd(&late_args().totals[1], L.tot[1]);
  }
}

static_assert(std::is_same<decltype(&k_walk<float, 1, false, false>), void (*)(WalkArgs)>::value,
              "late_args() reads the kernel's first argument");

__global__ __launch_bounds__(256) void k_points(const bh_particle* __restrict__ p, uint32_t n, double4* __restrict__ dst) {
  const uint32_t i = blockIdx.x * 256 + threadIdx.x;
  if (i < n) dst[i] = make_double4(p[i].pos[0], p[i].pos[1], p[i].pos[2], p[i].mass);
}

// One source's pull on a target, in FP64: G is applied at the end.
// The general form, for any operands.
__device__ __forceinline__ void direct_term(const double4& t, const double4& q, double eps2, double (&a)[3]) {
  const double dx = q.x - t.x, dy = q.y - t.y, dz = q.z - t.z;
  const double d2 = dx * dx + dy * dy + dz * dz;
  const double ds2 = d2 + eps2;
  const double ds = sqrt(ds2);
  const double sc = q.w * (1.0 / (ds2 * ds));
  a[0] += dx * sc;
  a[1] += dy * sc;
  a[2] += dz * sc;
}

// The same for a softened distance that cannot overflow or underflow: the square root and
// the division take two thirds of the general form's time, and x^(-3/2) =
// y^3 (1 - r)^(-3/2), y the hardware reciprocal square root and r = 1 - x y^2,
// needs eight instructions. The series to r^2 leaves a relative error of order
// r^3, far below rounding for the hardware estimate's r. It rounds no more
// often than the general form: against long double the accelerations of 64
// particles are off by 2.5e-16 (general: 2.6e-16) rms, of 700 by 4.1e-16 (4.1e-16).
__device__ __forceinline__ void direct_term_tame(const double4& t, const double4& q, double eps2, double (&a)[3]) {
  const double dx = q.x - t.x, dy = q.y - t.y, dz = q.z - t.z;
  const double x = __builtin_fma(dz, dz, __builtin_fma(dy, dy, __builtin_fma(dx, dx, eps2)));
  const double y = __builtin_amdgcn_rsq(x);
  const double y2 = y * y;
  const double r = __builtin_fma(-x, y2, 1.0);
  // as a factor of its own, so that an infinite product stays infinite
  const double p = __builtin_fma(r, __builtin_fma(r, 1.875, 1.5), 1.0);
  const double sc = q.w * (y2 * y) * p;
  a[0] = __builtin_fma(dx, sc, a[0]);
  a[1] = __builtin_fma(dy, sc, a[1]);
  a[2] = __builtin_fma(dz, sc, a[2]);
}

// Coordinates whose squared distances stay finite and do not underflow either,
// where the series would make not a number of an infinite pull: of two numbers
// of 1e-137 or more (or zero) the difference is zero or at least 1e-153. False
// for NaN.
__device__ __forceinline__ bool tame(double c) {
  const double m = fabs(c);
  return m < 1e150 && (m >= 1e-137 || m == 0.0);
}
__device__ __forceinline__ bool tame(const double4& q) { return tame(q.x) && tame(q.y) && tame(q.z); }

// brute_force_accel (brute_force.h:15-28) for targets tidx[0..m) over a
// slice of the sources; partial sums per slice, reduced in slice order.
// Bound by FP64 issue: 106 cycles per wavefront and source, of which 16 FP64
// operations and the reciprocal square root take 85-95 (131,072 particles:
// 27.5 ms with the general form only -> 11.9; 4,096 targets of 1M: 7.8 -> 3.2).
// The sources are [s0, s1) of all, cut into the launch's splits; with more, the
// sums go on from those of the sources before. tgt: the targets themselves, or
// null for those at their indices in src.
// A target leaves its own source out; only the tiles that hold a source of
// the wavefront's targets check for it. Eight wavefronts per SIMD hold the
// whole grid of a small target set at once.
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(8))) void k_direct(const double4* __restrict__ src, uint32_t s0, uint32_t s1,
                                                const double4* __restrict__ tgt, const uint32_t* __restrict__ tidx,
                                                uint32_t m, double eps2, double* __restrict__ partial, uint32_t splits,
                                                bool more) {
  __shared__ double4 s_src[256];
  const uint32_t k = blockIdx.x * 256 + threadIdx.x;
  const uint32_t split = blockIdx.y;
  const uint32_t lo = s0 + static_cast<uint32_t>(uint64_t(s1 - s0) * split / splits);
  const uint32_t hi = s0 + static_cast<uint32_t>(uint64_t(s1 - s0) * (split + 1) / splits);
  const bool ok = k < m;
  double* o = &partial[(uint64_t(split) * m + k) * 3];
  const uint32_t i = ok ? (tidx ? tidx[k] : k) : 0xffffffffu;
  double4 t = make_double4(0, 0, 0, 0);
  if (ok) t = tgt ? tgt[k] : src[i];
  double a[3] = {0.0, 0.0, 0.0};
  if (more && ok)
    for (int c = 0; c < 3; ++c) a[c] = o[c];
  const bool calm = tame(t) && fabs(eps2) < 1e300;
  for (uint32_t b = lo; b < hi; b += 256) {
    const uint32_t e = hi - b < 256 ? hi - b : 256;
    bool all = calm;
    __syncthreads();
    if (threadIdx.x < e) {
      const double4 q = src[b + threadIdx.x];
      s_src[threadIdx.x] = q;
      all = all && tame(q);
    }
    all = __syncthreads_and(all);
    const bool own = __any(i - b < e);
    if (all && !own) {
#pragma unroll 4
      for (uint32_t jj = 0; jj < e; ++jj) direct_term_tame(t, s_src[jj], eps2, a);
    } else if (all) {
      for (uint32_t jj = 0; jj < e; ++jj)
        if (b + jj != i) direct_term_tame(t, s_src[jj], eps2, a);
    } else {
      for (uint32_t jj = 0; jj < e; ++jj)
        if (b + jj != i) direct_term(t, s_src[jj], eps2, a);
    }
  }
  if (ok) {
    o[0] = a[0];
    o[1] = a[1];
    o[2] = a[2];
  }
}

__global__ __launch_bounds__(256) void k_direct_reduce(const double* __restrict__ partial, uint32_t m, uint32_t splits,
                                                       double G, double* __restrict__ acc) {
  const uint32_t k = blockIdx.x * 256 + threadIdx.x;
  if (k >= m) return;
  double a0 = 0.0, a1 = 0.0, a2 = 0.0;
#pragma unroll 16
  for (uint32_t s = 0; s < splits; ++s) {
    const double* o = &partial[(uint64_t(s) * m + k) * 3];
    a0 += o[0];
    a1 += o[1];
    a2 += o[2];
  }
  acc[3 * uint64_t(k) + 0] = G * a0;
  acc[3 * uint64_t(k) + 1] = G * a1;
  acc[3 * uint64_t(k) + 2] = G * a2;
}

// e + q.w / |t - q| in FP64. The hardware reciprocal square root is refined
// by the second-order step y (1 + r/2 + 3r^2/8), r = 1 - x y^2 (the Taylor
// series of (1 - r)^(-1/2)), which leaves a relative error of order r^3: far
// below FP64 rounding for the hardware estimate's r.
__device__ __forceinline__ double pot_term(const double4& t, const double4& q, double e) {
  const double dx = t.x - q.x, dy = t.y - q.y, dz = t.z - q.z;
  const double x = __builtin_fma(dz, dz, __builtin_fma(dy, dy, dx * dx));
  const double y = __builtin_amdgcn_rsq(x);
  const double r = __builtin_fma(-(x * y), y, 1.0);
  const double p = __builtin_fma(r, __builtin_fma(r, 0.375, 0.5), 1.0);
  return __builtin_fma(q.w * y, p, e);
}

// potential_energy (integrate.h:35-43) over unordered pairs: particle i
// adds m_j / r_ij for the partners j = i + d (mod n), d = 1 .. floor(n / 2),
// which counts every pair once (in an even-sized set the pair n / 2 apart is
// counted from its lower index only) and gives every thread the same work.
// Split s of the grid's second dimension takes the offsets
// [1 + h s / splits, 1 + h (s + 1) / splits), h = floor(n / 2); a block
// walks the window of partners its 256 particles share in tiles of 256.
// partial[s * blocks + b] = sum over the block's i of m_i sum_j m_j / r_ij.
__global__ __launch_bounds__(256) void k_potential(const double4* __restrict__ src, uint32_t n,
                                                   double* __restrict__ partial, uint32_t splits) {
  __shared__ double4 s_src[256];
  __shared__ double s_red[4];
  const uint32_t i0 = blockIdx.x * 256;
  const uint32_t i = i0 + threadIdx.x;
  const uint32_t split = blockIdx.y;
  const uint64_t h = n / 2;
  const uint64_t d_lo = 1 + h * split / splits, d_hi = 1 + h * (split + 1) / splits;
  const bool ok = i < n;
  // this thread's partner offsets [d_lo, my_hi)
  uint64_t my_hi = d_hi;
  if (n % 2 == 0 && d_hi == h + 1 && i >= h) my_hi = h;
  double4 t = make_double4(0, 0, 0, 0);
  if (ok) t = src[i];
  double e = 0.0;
  // partners of the block: positions i0 + d_lo .. i0 + 255 + d_hi - 1
  // (unwrapped). Every lane reads the same partner at the same time (an LDS
  // broadcast); a tile where some lane's window starts or ends is masked
  // per lane, the tiles in between (nearly all) are not.
  const uint64_t w_lo = uint64_t(i0) + d_lo, w_hi = uint64_t(i0) + 255 + d_hi;
  for (uint64_t jb = w_lo; jb < w_hi; jb += 256) {
    __syncthreads();
    {
      const uint64_t j = jb + threadIdx.x;
      if (j < w_hi) s_src[threadIdx.x] = src[j % n];
    }
    __syncthreads();
    const int cnt = static_cast<int>(w_hi - jb < 256 ? w_hi - jb : 256);
    // this lane's partners in the tile: [lo, hi) (unwrapped partner position
    // of offset d is i + d)
    const int64_t k_lo = static_cast<int64_t>(uint64_t(i) + d_lo) - static_cast<int64_t>(jb);
    const int64_t k_hi = static_cast<int64_t>(uint64_t(i) + my_hi) - static_cast<int64_t>(jb);
    const int lo = ok ? static_cast<int>(k_lo < 0 ? 0 : (k_lo > 256 ? 256 : k_lo)) : 0;
    const int hi = ok ? static_cast<int>(k_hi < 0 ? 0 : (k_hi > 256 ? 256 : k_hi)) : 0;
    const bool whole = __syncthreads_and(lo == 0 && hi >= cnt);
    if (whole) {
#pragma unroll 4
      for (int k = 0; k < cnt; ++k) e = pot_term(t, s_src[k], e);
    } else {
      for (int k = 0; k < cnt; ++k) {
        const double with = pot_term(t, s_src[k], e);
        e = (k >= lo && k < hi) ? with : e;
      }
    }
  }
  double v = ok ? t.w * e : 0.0;
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
  if (__lane_id() == 0) s_red[threadIdx.x >> 6] = v;
  __syncthreads();
  if (threadIdx.x == 0) partial[uint64_t(split) * gridDim.x + blockIdx.x] = s_red[0] + s_red[1] + s_red[2] + s_red[3];
}

// Masking r = 0 is needed only without softening (grouped_ttg.h:119-123); it
// never triggers when eps2 > 0, so one masked launch serves mixed batches.
template <typename Real, int kWaves>
hipError_t launch_walk_t(const WalkArgs& a, uint32_t slots, bool deep, bool any_unsoftened, hipStream_t s) {
  // every XCD gets the same number of workgroups
  const uint32_t blocks = (slots + 7) / 8 * 8;
  // The stack needs one frame per level below a walk's start. The first
  // kShallowFrames frames are in LDS (4 waves per SIMD); trees with more
  // levels (any system of a batch) also use the global deep frames.
  if (!any_unsoftened) {
    if (!deep)
      hipLaunchKernelGGL((k_walk<Real, kWaves, false, false>), dim3(blocks), dim3(kWaves * 64), 0, s, a);
    else
      hipLaunchKernelGGL((k_walk<Real, kWaves, false, true>), dim3(blocks), dim3(kWaves * 64), 0, s, a);
  } else {
    if (!deep)
      hipLaunchKernelGGL((k_walk<Real, kWaves, true, false>), dim3(blocks), dim3(kWaves * 64), 0, s, a);
    else
      hipLaunchKernelGGL((k_walk<Real, kWaves, true, true>), dim3(blocks), dim3(kWaves * 64), 0, s, a);
  }
  return hipGetLastError();
}

}  // namespace

hipError_t launch_walk(const WalkArgs& a, uint32_t slots, bool deep, int fp64, bool any_unsoftened, hipStream_t s) {
  if (slots == 0 || slots % 8 != 0 || slots > kWalkSlots) return hipErrorInvalidValue;
  // One wavefront per workgroup: walk units differ widely in work, and a
  // workgroup's LDS is released only when all its waves are done (2 waves
  // per workgroup: 49.7 ms at 16M, 4: 53.9, 8: 64.8; 1: 47.0).
  return fp64 ? launch_walk_t<double, 1>(a, slots, deep, any_unsoftened, s)
              : launch_walk_t<float, 1>(a, slots, deep, any_unsoftened, s);
}

hipError_t launch_points(const bh_particle* p, uint32_t n, double4* dst, hipStream_t s) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_points, dim3((n + 255) / 256), dim3(256), 0, s, p, n, dst);
  return hipGetLastError();
}

hipError_t launch_potential(const double4* src, uint32_t n, double* partial, uint32_t splits, hipStream_t s) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_potential, dim3((n + 255) / 256, splits), dim3(256), 0, s, src, n, partial, splits);
  return hipGetLastError();
}

uint32_t pair_splits(uint64_t blocks, uint64_t partners, uint64_t least, uint32_t ragged) {
  uint64_t best = std::min<uint64_t>(std::max<uint64_t>(2048 / blocks, 1), 512);
  while (best > 1 && partners / best < (blocks * best > 256 ? least : least / 4)) best >>= 1;
  uint64_t cost = ~0ull;
  const uint64_t most = blocks * best < 1024 ? best : std::max(best, std::min(8 * best, partners / 4096));
  for (uint64_t s = best; s <= most; ++s) {
    const uint64_t c = (blocks * s + 255) / 256 * ((partners + s - 1) / s + ragged);
    if (c + c / 64 < cost) best = s, cost = c;
  }
  return static_cast<uint32_t>(best);
}

hipError_t launch_direct(const double4* src, uint32_t s0, uint32_t s1, const double4* tgt, const uint32_t* tidx,
                         uint32_t m, double eps2, double* partial, uint32_t splits, bool more, hipStream_t s) {
  if (m == 0) return hipSuccess;
  hipLaunchKernelGGL(k_direct, dim3((m + 255) / 256, splits), dim3(256), 0, s, src, s0, s1, tgt, tidx, m, eps2, partial,
                     splits, more);
  return hipGetLastError();
}

hipError_t launch_direct_reduce(const double* partial, uint32_t m, uint32_t splits, double G, double* acc,
                                hipStream_t s) {
  if (m == 0) return hipSuccess;
  hipLaunchKernelGGL(k_direct_reduce, dim3((m + 255) / 256), dim3(256), 0, s, partial, m, splits, G, acc);
  return hipGetLastError();
}

}  // namespace bhk
