// Internal interfaces between the host orchestration (bh_api.cpp) and the
// CDNA4 kernels (bh_sort.hip, bh_tree.hip, bh_walk.hip). Not part of the ABI.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/bh_gpu.h"

namespace bhk {

constexpr int kWave = 64;
constexpr int kDepthCap = 21;           // flat_tree.h:102 (21 octal digits)
constexpr int kLevels = kDepthCap + 1;  // depths 0..21
constexpr uint32_t kMaxLeafCap = 1024;  // halo of the tree-build tile
constexpr uint32_t kSortTile = 4096;    // keys per onesweep workgroup, at most
constexpr uint32_t kTreeTile = 4096;    // particles per tree-build workgroup
constexpr int kTreeCols = 24;           // per tile: 22 level counts, leaf count, pad

// Flag/value word of the decoupled look-back (30-bit counts).
constexpr uint32_t kLbAgg = 1u << 30;
constexpr uint32_t kLbPre = 2u << 30;
constexpr uint32_t kLbVal = (1u << 30) - 1;

// One system of a batch: its particles are [off, off + n) of the batch
// arrays, both in input and in sorted order (systems stay contiguous).
struct SysDev {
  double theta2;
  double eps2;
  double G;
  double kick_dt;
  double drift_dt;
  uint32_t off;
  uint32_t n;
  uint32_t max_leaf;
  uint32_t tsm;      // min(target_size, group_size)
  uint16_t use_quad;
  uint16_t tile;         // walk tile: particles a unit of several targets holds (kMinTile..kGroupCap)
  uint16_t unit_piece;   // particles of a piece of a unit of several targets
  uint16_t target_piece; // particles of a piece of a unit that is one target
};
static_assert(sizeof(SysDev) == 64, "SysDev layout");

constexpr uint32_t kChunk = 4096;    // particles per bounds block, at most
constexpr uint32_t kMaxSystems = 65535;
constexpr uint64_t kMaxN = (1ull << 30) - 1;  // particles per step (all systems)
constexpr uint32_t kGroupCap = 128;  // largest walk tile: a walk unit's particles fill at most two slots per lane
constexpr uint32_t kMinTile = 16;    // smallest walk tile
constexpr uint32_t kDefer = 512;     // deferred nodes a group may hand its targets
constexpr uint32_t kShallowFrames = 12;  // walk stack of trees with at most this many levels
constexpr uint32_t kQueueStride = 32;    // words from one walk-unit queue head to the next: a cache line
constexpr uint32_t kQueueWords = 8 * kQueueStride;
constexpr uint32_t kWalkSlots = 4096;    // walk workgroups at most: 256 CUs x 4 SIMDs x 4 waves

// The step's flag and count words (`misc`), cleared when a step starts and
// read back once when it ends. Kernels after the tree's node count test the
// abort word and return at once when it is set, so a step whose tree did not
// fit the planned arrays or levels leaves its output untouched and is run
// again with larger ones.
constexpr int kMiscNonfinite = 0;   // some position, velocity or mass is NaN or infinite
constexpr int kMiscAbort = 1;       // kAbortNodes | kAbortDepth
constexpr int kMiscIncomplete = 2;  // the walk met an interior node it could not open
constexpr int kMiscMaxDepth = 3;    // deepest level of the tree
constexpr int kMiscLevels = 8;      // [8, 8 + kLevels): nodes per level; [8 + kLevels]: leaves
constexpr int kMiscTargets = 40;    // walk targets
constexpr int kMiscGroups = 41;     // walk units
constexpr int kMiscWords = 64;
// Behind them the two 64-bit interaction totals and the times (of the GPU's
// constant-rate clock) at which the step's phases began: start, tree, targets,
// walk, and the report that ends the step.
constexpr int kMiscTotals = kMiscWords;
constexpr int kMiscStamps = kMiscTotals + 4;
constexpr int kStamps = 5;
enum Stamp { kStampStart, kStampTree, kStampTargets, kStampWalk, kStampEnd };
constexpr int kReportWords = kMiscStamps + 2 * kStamps;
constexpr uint32_t kAbortNodes = 1;  // more nodes or leaves than the node arrays hold
constexpr uint32_t kAbortDepth = 2;  // deeper than the levels the upward pass launched
constexpr uint32_t kAbortSort = 4;   // too many keys share the sort's leading bits

// The device a context was created on.
int ctx_device(const bh_ctx* ctx);

// What the walk reads of a node, in one 64-byte record: the MAC data (FP64
// com and squared edge), the link (leaf: first particle and count | 1 << 31;
// interior: first child and child count) and the FP32 mass and traceless
// quadrupole (Qzz = -(Qxx + Qyy)).
struct alignas(64) NodeRec {
  double cx, cy, cz, edge2;
  uint32_t first, count;
  float m, qxx, qyy, qxy, qxz, qyz;
};
static_assert(sizeof(NodeRec) == 64, "NodeRec layout");

// Device view of one tree (level-order BFS numbering).
struct TreeDev {
  uint32_t* begin;       // [M] first particle (Morton position)
  uint32_t* count;       // [M] particles
  uint8_t* depth;        // [M]
  uint8_t* leaf;         // [M]
  uint32_t* cs;          // [M] child start: level-order index of the first child slot
  uint32_t* first_child; // [M] (0 for leaves)
  uint8_t* nchild;       // [M]
  uint32_t* parent;      // [M] (UINT32_MAX for the root)
  uint32_t* leaf_idx;    // [M] index into the leaf list (leaves only)
  double4* ctr;          // [M] geometric centre xyz, half width
  double* mass;          // [M]
  double* com;           // [3M]
  double* iab;           // [6M] xx,yy,zz,xy,xz,yz about the com
  NodeRec* rec;          // [M] the walk's node record
  double* q64;           // [8M] mass, Qxx, Qyy, Qzz, Qxy, Qxz, Qyz, 0
  double* nbox;          // [6M] FP64 box of the node's particles: lo x, y, z, hi x, y, z
  uint32_t* leaf_node;   // [leaves] node of each leaf, Morton order
  uint32_t* leaf_first;  // [leaves] first particle of each leaf
  uint32_t* level_off;   // [kLevels + 2] level start offsets, then total, total
  uint32_t* misc;        // [kMiscWords] the step's flags and counts
  uint32_t cap;          // node (and leaf) capacity of the arrays above
};

struct WalkArgs {
  const NodeRec* rec;
  const double* q64;
  const double4* ctr;
  const uint32_t* begin;
  const uint32_t* count;
  const double4* posm;     // x, y, z, m in Morton order
  const uint2* units;      // walk units, Morton order: {node, first particle} of each piece
  const uint32_t* unit_n;  // [n_nodes] particles | 1 << 31 of a packed unit at its first node, else 0 (nullable)
  const uint32_t* tmark;   // [n] target node + 1 at each target's first particle, else 0
  const uint16_t* sid;     // system of each particle
  const SysDev* sys;       // system table; the root of system s is node s
  const double* nbox;      // [6 n_nodes] FP64 particle box of every node (lo xyz, hi xyz)
  double* gacc;            // [3n] scratch: a group's shared-list sums per particle
  uint32_t* defer;         // [slots * kDefer] scratch: deferred nodes, per walk workgroup
  uint32_t* deep_frames;   // [slots * (kLevels - kShallowFrames) * 64] stack frames below the LDS ones
  uint32_t* misc;          // the step's flags and the unit count
  uint32_t* queue;         // [kQueueWords] walk-unit queue heads, one per XCD and cache line, zero at the start
  uint32_t n_nodes;        // index clamps (the node capacity): a node or particle
  uint32_t n_parts;        // index never leaves its array, whatever the tree holds
  uint32_t stack_limit;    // frames the walk may use (kLevels; lower only to test the incomplete-walk report)
  bh_particle* parts;      // Morton-order particles to kick/drift (nullable)
  const bh_particle* src;  // with parts: the unsorted input, read at perm (else parts is read in place)
  const uint32_t* perm;    // [n] Morton position -> input index (with src)
  double* carry;           // with parts: [4 n] the new x, y, z and m (blocks of n) for the next step's build (nullable)
  uint32_t* carry_bad;     // with carry: set when a new position, velocity or mass is not finite
  double* acc;             // [3n] G * acceleration (nullable)
  uint32_t* n_pp;          // [n] (nullable)
  uint32_t* n_pc;          // [n] (nullable)
  unsigned long long* totals;  // [2]
};

// ---- bh_sort.hip
// Up to kMax device ranges of 32-bit words to zero (unused: n = 0).
struct ZeroRanges {
  static constexpr int kMax = 6;
  uint32_t* p[kMax] = {};
  uint64_t n[kMax] = {};
};
hipError_t launch_zero(const ZeroRanges& r, hipStream_t s);
__device__ inline void zero_ranges(const ZeroRanges& r, uint64_t t, uint64_t threads) {
#pragma unroll
  for (int k = 0; k < ZeroRanges::kMax; ++k) {
    // 16 bytes at a time where the range allows it
    uint32_t* p = r.p[k];
    const uint64_t quads = (reinterpret_cast<uintptr_t>(p) & 15u) ? 0 : r.n[k] / 4;
    for (uint64_t i = t; i < quads; i += threads) reinterpret_cast<uint4*>(p)[i] = make_uint4(0u, 0u, 0u, 0u);
    for (uint64_t i = 4 * quads + t; i < r.n[k]; i += threads) p[i] = 0u;
  }
}
// The time at which a phase's first workgroup begins, into the report.
__device__ inline void stamp(uint32_t* misc, Stamp which) {
  if (blockIdx.x == 0 && threadIdx.x == 0)
    reinterpret_cast<unsigned long long*>(misc + kMiscStamps)[which] = wall_clock64();
}

// The step's first launches: the system table read from the host, everything
// that a step needs zeroed, every particle's system, and the bounds.
struct StartArgs {
  const uint4* host_table;   // pinned host memory: the system table ...
  uint4* table;              // ... and where the device keeps it
  uint32_t table_quads;
  const uint4* host_hist;    // pinned: digit counts of the system ids (null: one system)
  uint4* hist;
  ZeroRanges zero;
  const uint4* host_chunks;  // [n_chunks] in the host's table: {system, begin, end, 0}, particles of one system
  const uint32_t* chunk_first;  // [n_sys + 1] in the device's table: first chunk of each system, then n_chunks
  uint32_t n_chunks, n_sys;
  uint32_t n, chunk;         // one system: chunk c is [c * chunk, min(n, (c + 1) * chunk)), not read from the host
  uint16_t* sid;             // [n]
  double* partial;           // [6 n_chunks]
  double* lohi;              // [6 n_sys]
  uint32_t* misc;
};
hipError_t launch_start(const bh_particle* p, const StartArgs& a, hipStream_t s);
// One system of at most kSmallSort particles: all of that (a.zero's range 0 is
// misc), its keys, their sort and (posm not null) the walk copy in one launch or,
// above 1,024 particles, two, with bkeys and bperm between; a.hist, the chunks
// and a.partial are not used. It orders whole keys, so there is nothing to give
// up.
constexpr uint32_t kSmallSort = 12288;
hipError_t launch_small_sort(const bh_particle* p, const StartArgs& a, uint64_t* keys, uint32_t* perm, uint64_t* bkeys,
                             uint32_t* bperm, double4* posm, hipStream_t s);
// The step's last: the report (misc, totals, stamps) to pinned host memory.
hipError_t launch_report(uint32_t* misc, uint32_t* host, hipStream_t s);
// Keys, and the histograms of their `passes` leading 8-bit digits.
hipError_t launch_keys_hist(const bh_particle* p, uint32_t n, int passes, const uint16_t* sid, const double* lohi,
                            uint64_t* keys, uint32_t* hist, hipStream_t s);
// The same from the compact copy a resident step's walk wrote for its
// output (the next step's input): blocks of n x, y, z and m, of which these
// read x, y, z (24 of the records' 64 bytes). carried_bad: that walk's
// non-finite flag, added to misc[kMiscNonfinite].
hipError_t launch_start(const double* pos, const uint32_t* carried_bad, const StartArgs& a, hipStream_t s);
hipError_t launch_small_sort(const double* pos, const uint32_t* carried_bad, const StartArgs& a, uint64_t* keys,
                             uint32_t* perm, uint64_t* bkeys, uint32_t* bperm, double4* posm, hipStream_t s);
hipError_t launch_keys_hist(const double* pos, uint32_t n, int passes, const uint16_t* sid, const double* lohi,
                            uint64_t* keys, uint32_t* hist, hipStream_t s);
// key_passes passes over the keys' leading bits, sid_passes (0-2) over the
// system id taken from sid[index], and the runs of equal leading bits (none
// with 8 passes) ordered by the bits below: a stable sort of each system's
// (key, index) pairs in place. hist: 10 x 256 digit counts (8-9: the
// systems). abort: gets kAbortSort when such a run is too long.
hipError_t launch_radix_sort(uint64_t* keys_a, uint32_t* vals_a, uint64_t* keys_b, uint32_t* vals_b, uint32_t n,
                             uint32_t tile, int key_passes, int sid_passes, const uint16_t* sid, const uint32_t* hist,
                             uint32_t* lookback, uint32_t* abort, uint64_t** keys_out, uint32_t** vals_out,
                             hipStream_t s);
// The FP64 walk copy (x, y, z, m) in Morton order; with out, also the
// Morton-ordered particles (a step's walk writes those itself).
hipError_t launch_gather(const bh_particle* in, bh_particle* out, const uint32_t* perm, double4* posm, uint32_t n,
                         hipStream_t s);
// The same walk copy from a carried compact copy (blocks of n x, y, z and
// m) in the order perm indexes.
hipError_t launch_gather(const double* pos, const uint32_t* perm, double4* posm, uint32_t n, hipStream_t s);
// A pass's workgroups take `tile` keys, kSortTile or half of it: with few tiles a
// pass is a chain of latencies, and half the keys shorten it, with many it is
// bound by memory and a tile's 256 look-back words are overhead (sort phase,
// 4,096 -> 2,048 keys: 65,536 particles 75.5 -> 67.7 us, 131,072 82 -> 75, 262,144
// 94 -> 90, 400,000 equal, 1M 171 -> 193).
inline uint32_t sort_tile(uint32_t n) { return n <= 64 * kSortTile ? kSortTile / 2 : kSortTile; }
// Tile counters (10 of 64 words, so that rows of look-back words stay aligned),
// then up to 10 passes' look-back words.
constexpr uint32_t kSortCounters = 64;
inline uint64_t radix_lookback_words(uint32_t n, uint32_t tile, int passes) {
  return kSortCounters + uint64_t(passes) * ((uint64_t(n) + tile - 1) / tile) * 256;
}

// ---- bh_tree.hip
hipError_t launch_tree_count(const uint64_t* keys, uint32_t n, const uint16_t* sid, const SysDev* sys,
                             uint32_t max_leaf_max, uint8_t* L, uint8_t* H, uint32_t* tile_counts, uint32_t* misc,
                             hipStream_t s);
// Numbers the nodes and writes their topology; when the tree has more nodes
// or leaves than t.cap it writes nothing and sets kAbortNodes, when it is
// deeper than depth_plan it sets kAbortDepth.
// The levels' and the leaves' totals go to misc.
hipError_t launch_tree_emit(const uint8_t* L, const uint8_t* H, uint32_t n, const uint32_t* tile_counts,
                            uint32_t* tile_prefix, TreeDev t, uint32_t depth_plan, hipStream_t s);
// Links, geometry and the upward pass: every leaf in one launch, then the
// interior nodes of levels depth_plan - 1..0 (one launch per level, each
// grid-striding over the level's range read on the device; n_sys systems
// bound a level's node count by n_sys * 8^d; a single system's upper levels in
// one launch, all of them for a small one). The first also zeroes `zero`.
hipError_t launch_tree_finish(const uint64_t* keys, const double4* posm, uint32_t n, const uint16_t* sid, uint32_t n_sys,
                              const double* lohi, uint32_t depth_plan, const ZeroRanges& zero, TreeDev t, hipStream_t s);
// Marks the walk targets (node + 1 at the first particle in tmark; their
// number is added to misc[kMiscTargets]) and lists the walk units (their
// number to misc[kMiscGroups]). Targets: topmost nodes with leaf || count <=
// tsm. Units: with grouped, topmost nodes with leaf || count <= max(tsm,
// tile), runs of sibling ones that are single targets packed up to tile
// particles (unit_n per node: particles | 1 << 31 at a packed unit's first
// node, else 0); otherwise the targets. A unit of more particles than its
// kind's piece is listed once per piece. tmark, gmark, the two counts and
// the unit_list_words() look-back words must be zero.
hipError_t launch_units(TreeDev t, uint32_t n, const uint16_t* sid, const SysDev* sys, bool grouped, uint32_t* tmark,
                        uint32_t* gmark, uint32_t* unit_n, uint32_t* lookback, uint2* units, hipStream_t s);
inline uint64_t unit_list_words(uint64_t n) { return (n + kTreeTile - 1) / kTreeTile + 1; }

// What a piece of a unit of cnt particles holds (the last one the rest): equal
// pieces of at most `piece`.
__host__ __device__ inline uint32_t piece_size(uint32_t cnt, uint32_t piece) {
  const uint32_t k = (cnt + piece - 1) / piece;
  return k > 1 ? (cnt + k - 1) / k : cnt;
}

// ---- bh_walk.hip
// slots workgroups (a multiple of 8, at most kWalkSlots) take the units from
// per-XCD queues; deep selects the variant whose stack also uses deep_frames
// (trees of more than kShallowFrames levels).
hipError_t launch_walk(const WalkArgs& a, uint32_t slots, bool deep, int fp64, bool any_unsoftened, hipStream_t s);
// dst[i] = (x, y, z, m) of record i
hipError_t launch_points(const bh_particle* p, uint32_t n, double4* dst, hipStream_t s);
// partial[splits * m]: per split sums over the sources [s0, s1) of src, with more
// added to what is there. Targets tgt[k], or src[tidx[k]] (src[k]) without tgt;
// tidx[k] (k) is the source that target k leaves out.
hipError_t launch_direct(const double4* src, uint32_t s0, uint32_t s1, const double4* tgt, const uint32_t* tidx,
                         uint32_t m, double eps2, double* partial, uint32_t splits, bool more, hipStream_t s);
// acc[m] = G times the splits' sums
hipError_t launch_direct_reduce(const double* partial, uint32_t m, uint32_t splits, double G, double* acc,
                                hipStream_t s);
// Into how many windows the partners that each of `blocks` workgroups goes over
// are split, in the grids of pair sums: up to the 2,048 workgroups that fill the
// chip's wavefronts, with at least `least` partners a window (a quarter of that
// while no compute unit has two workgroups). Long windows are split further, up
// to eight times, where that leaves less work on the compute unit with most (256
// share the workgroups; `ragged` partners' time goes with a window's ends; it has
// to save 1/64, as each split has sums of its own): only filling the chip left
// some units a third more than others at sizes just over a multiple. ms:
//   pairs of (k_potential)   1,000 0.088 -> 0.079   200,000 13.2 -> 11.4   300,001 28.4 -> 24.5
//                            400,003 49.5 -> 42.5   600,000 100.7 -> 93.4  131,072 equal
//   all targets (k_direct)   1,000 0.122 -> 0.086   100,003 7.9 -> 7.2     300,000 69.9 -> 59.6
// (Windows picked that way at 5,000 to 20,000 particles, too, were up to 10%
// slower: there the ends and the wavefronts a unit has count as much.)
uint32_t pair_splits(uint64_t blocks, uint64_t partners, uint64_t least, uint32_t ragged);
// partial[splits * ceil(n/256)]: per (slice, block) sums of m_i * m_j / r_ij over
// unordered pairs {i, j} (each counted once, from the i of the block)
hipError_t launch_potential(const double4* src, uint32_t n, double* partial, uint32_t splits, hipStream_t s);

}  // namespace bhk
