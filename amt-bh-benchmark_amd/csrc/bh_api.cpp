// Host side of the C ABI (include/bh_gpu.h): the context, its grow-only
// device buffers, and the per-step orchestration of the kernels.
//
// One step (step_particles, integrate_ttg.h:88-107, grouped branch):
//   start (system table, zeroing, chunk bounds) -> bounds -> keys + digit
//   histograms -> onesweep radix passes over the leading bits -> runs of equal
//   ones -> gather of the FP64 walk copy (one system of at most kSmallSort
//   particles: one or two launches for all of these) ->
//   tree counts -> node emit -> links/centres -> upward pass (leaves, levels) ->
//   targets and walk units -> walk with fused kick/drift -> report.
// Everything is ordered on the context's stream and nothing in between
// needs the host: the kernels read the node, level and unit counts on the
// device. The host waits once, at the end; the last kernel has by then written
// the flags, counts and phase times to pinned host memory. The node arrays and the number of upward levels are
// planned from what the context has seen (and from n); a tree that turns out
// larger or deeper sets an abort word, every kernel after the node count
// returns at once, and the step runs again with the arrays grown (its input
// is never written, so running it again is exact). Because a step makes no
// host decision midway, the whole launch sequence can be captured once into
// a HIP graph and replayed (bh_set_graph_mode).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <limits>
#include <memory>
#include <mutex>
#include <new>
#include <string>
#include <vector>

#include "bh_internal.h"

using namespace bhk;

static_assert(kGroupCap == BH_MAX_WALK_TILE && kMinTile == BH_MIN_WALK_TILE, "walk tile limits");

namespace {

// The allocation-free entry point's working memory: one fixed array per GPU
// (every call on that GPU shares it), reached through the address that
// hipGetSymbolAddress returns for the current device.
constexpr size_t kNoAllocBytes = size_t(BH_NOALLOC_SCRATCH_MIB) << 20;
constexpr uint32_t kNoAllocSlots = 512;  // walk workgroups of the allocation-free step
static __device__ __align__(256) unsigned char scratch[kNoAllocBytes];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_ptr[kMaxDevices] = {};

// The device address of `scratch` on `device` (which must be current),
// looked up once per device.
hipError_t scratch_address(int device, void** out) {
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (device < 0 || device >= kMaxDevices) return hipErrorInvalidDevice;
  if (!g_scratch_ptr[device]) {
    void* ptr = nullptr;
    const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return e;
    g_scratch_ptr[device] = ptr;
  }
  *out = g_scratch_ptr[device];
  return hipSuccess;
}

template <typename T>
struct DevBuf {
  T* p = nullptr;
  size_t cap = 0;
};

// Every array a step uses besides the particles in and out.
struct Scratch {
  uint64_t *keys_a = nullptr, *keys_b = nullptr;
  uint32_t *vals_a = nullptr, *vals_b = nullptr;
  uint32_t *hist = nullptr, *lookback = nullptr;
  double *lohi = nullptr, *partial = nullptr;
  uint32_t* misc = nullptr;              // kMiscWords
  unsigned long long* totals = nullptr;  // [2] interaction totals
  double4* posm = nullptr;
  uint8_t *L = nullptr, *H = nullptr;
  uint32_t *tcounts = nullptr, *tprefix = nullptr;
  uint16_t* sid = nullptr;
  uint8_t* tables = nullptr;
  TreeDev t{};
  uint32_t *mark = nullptr, *gmark = nullptr, *unit_n = nullptr, *unit_lb = nullptr;
  uint2* units = nullptr;
  uint32_t *defer = nullptr, *deep_frames = nullptr;
  double* gacc = nullptr;
};

// The walk's queue heads lie over the sort's look-back words (at least 2,560),
// which are free by then.
uint32_t* walk_queue(const Scratch& b) { return b.lookback; }

// What the host decides before a step is enqueued.
struct Plan {
  uint32_t n = 0;         // particles of all systems
  uint32_t S = 0;         // non-empty systems
  uint32_t n_chunks = 0;  // bounds blocks ...
  uint32_t chunk = kChunk;  // ... of at most this many particles
  uint32_t sort_tile = kSortTile;  // keys of a radix workgroup
  uint32_t mlx = 0;       // largest max_leaf
  int sid_passes = 0;     // radix passes over the system id
  int key_passes = 8;     // radix passes over the keys' leading bits (8: all of them)
  uint64_t largest = 0;   // particles of the largest system
  bool unsoftened = false;
  size_t table_bytes = 0, off_chunks = 0, off_first = 0, off_hist = 0;
  uint64_t node_estimate = 0;
  uint32_t cap_nodes = 0;  // node array capacity the kernels may use
  uint32_t depth_plan = kDepthCap;
  bool deep = true;        // walk stack frames beyond LDS
  uint32_t slots = 0;      // walk workgroups
  bool walk = true;        // false: tree build only
  bool carry_out = false;  // the walk writes the compact positions of its output (resident steps)
  bool carried_in = false; // the input is the last resident step's output: build from its compact positions
};

// A few workgroups sort the system, one up to 1,024 particles.
bool small(const Plan& p) { return p.S == 1 && p.n <= kSmallSort; }

// One captured step, keyed by everything its launches depend on.
struct GraphKey {
  const void* in;
  const void* out;
  uint64_t gen;
  uint32_t n, S, n_chunks, mlx, cap_nodes, depth_plan, slots;
  uint32_t table_bytes;
  uint8_t deep, unsoftened, precision, mode, carry_out, carried_in, key_passes, pad;
  bool operator==(const GraphKey& o) const { return std::memcmp(this, &o, sizeof *this) == 0; }
};
struct GraphEntry {
  GraphKey key;
  hipGraphExec_t exec;
  uint64_t used;
};
constexpr size_t kGraphCache = 256;

constexpr uint64_t kFewPoints = 1024;  // records that load_points packs on the host

// After a step whose keys shared too many leading bits, so many sort by whole
// keys before the leading bits are tried again, as a system may lose its far
// particle and the next one need not have any. A trial that fails costs its
// sort and tree counts (at 20,000 particles half a step): each doubles the span.
constexpr uint32_t kFullSteps = 64, kFullStepsMost = 4096;

struct Ctx {
  int device = 0;
  hipStream_t stream = nullptr;
  double clock_khz = 0.0;   // rate of the GPU's constant clock
  unsigned long long stamps[kStamps] = {};  // when the last step's phases began
  bool have_stats = false;
  bool last_graph = false;  // the last step ran as a graph: only its total time is known
  uint32_t reruns = 0;      // times the last step ran again with larger arrays
  std::string err;
  int precision = BH_FP32;
  int walk_mode = BH_WALK_GROUPED;
  int graph_mode = BH_GRAPH_OFF;
  uint32_t walk_tile = kGroupCap;
  uint32_t stack_limit = kLevels;  // lowered only by bh_debug_walk_stack_limit
  void* arena = nullptr;  // this device's allocation-free scratch

  DevBuf<bh_particle> pa, pb;    // particle ping-pong of the resident state
  int cur = 0;                   // which of pa/pb holds the resident state
  uint64_t state_n = 0;
  // {x, y, z, m} of the last resident step's output and its non-finite flag,
  // valid (carried_ok) until anything else runs or the state is exposed
  DevBuf<double> carry;
  DevBuf<uint32_t> carry_flag;
  bool carried_ok = false;
  const void* carried_out = nullptr;
  uint64_t carried_n = 0;
  DevBuf<bh_particle> tmp_in, tmp_out;  // host-path staging (bh_step, bh_step_batch_host, bh_build_tree)
  DevBuf<uint64_t> keys_a, keys_b;
  DevBuf<uint32_t> vals_a, vals_b;
  DevBuf<uint32_t> hist, lookback;
  DevBuf<double> lohi, partial;
  DevBuf<uint32_t> misc;
  DevBuf<double4> posm;
  DevBuf<uint8_t> L, H;
  DevBuf<uint32_t> tcounts, tprefix;
  DevBuf<uint32_t> mark, gmark, unit_n, unit_lb, defer, deep_frames;
  DevBuf<uint2> units;
  DevBuf<double> gacc, nbox;
  DevBuf<uint32_t> begin, count, cs, first_child, parent, leaf_idx, leaf_node, leaf_first, level_off;
  DevBuf<uint8_t> depth, leaf, nchild;
  DevBuf<double4> ctr;
  DevBuf<NodeRec> rec;
  DevBuf<double> mass, com, iab, q64;
  DevBuf<uint8_t> tables;
  DevBuf<uint16_t> sid;
  // direct sum and energies
  DevBuf<bh_particle> drec;  // a piece of the records on their way into dsrc
  DevBuf<double4> dsrc;
  double4 few[kFewPoints];   // few of them, on the host
  DevBuf<double4> dtgt;      // a direct sum's targets when it begins before all records are there
  // Copies beside kernels (made by the first call that needs them): the kernels'
  // stream and the copies' stream, one after the other so that they get hardware
  // queues of their own (in one queue nothing overlaps: 5.1 ms instead of 3.55),
  hipStream_t side[2] = {};
  hipEvent_t landed[2] = {};   // the end of the copy into each half of drec
  hipEvent_t picked[2] = {};   // and of the kernel that reads it
  DevBuf<uint32_t> didx, dcnt;
  DevBuf<double> dpart, dacc;

  uint32_t* host_misc = nullptr;  // pinned: the last step's report (kReportWords)
  uint8_t* host_tables = nullptr; // pinned system table staging
  size_t host_tables_cap = 0;
  uint64_t gen = 1;               // bumped whenever a buffer a graph may hold moves

  // plans learnt from earlier steps
  uint32_t cap_nodes = 0;        // node capacity asked for (grow-only)
  bool depth_known = false;
  uint32_t full_sort = 0;        // steps left that sort by whole keys, as one's shared too many leading bits
  uint32_t full_span = kFullSteps;  // how many, when the next such step is met
  uint32_t depth_hint = kDepthCap;

  std::vector<GraphEntry> graphs;
  uint64_t graph_clock = 0;

  // last tree (for export and bh_accel) and last step's report
  bool has_tree = false;
  Plan plan{};
  Scratch sc{};
  uint32_t n = 0, n_nodes = 0, n_leaves = 0, max_depth = 0, n_targets = 0, n_groups = 0;
  uint32_t max_leaf = 0, group_size = 0;
  unsigned long long last_totals[2] = {0, 0};
  bh_particle* sorted = nullptr;    // device: Morton-ordered particles of the last tree
  uint64_t* keys_sorted = nullptr;  // device: sorted keys of the last tree
  uint32_t* perm_sorted = nullptr;  // device: sorted position -> input index
};

// One system of a batch as the host sees it.
struct HostSys {
  uint64_t n;
  bh_force_params fp;
  uint32_t max_leaf, group_size, target_size;
  double kick_dt, drift_dt;
  uint32_t tile;  // 0: the context's
};

bool set_err(Ctx* c, const char* fmt, ...) {
  char buf[512];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(buf, sizeof buf, fmt, ap);
  va_end(ap);
  c->err = buf;
  return false;
}

#define HIP_OK(c, expr)                                                                         \
  do {                                                                                          \
    hipError_t e_ = (expr);                                                                     \
    if (e_ != hipSuccess) {                                                                     \
      set_err((c), "%s failed: %s (%s:%d)", #expr, hipGetErrorString(e_), __FILE__, __LINE__); \
      return BH_ERR_HIP;                                                                        \
    }                                                                                           \
  } while (0)

#define TRY(expr)                 \
  do {                            \
    int rc_ = (expr);             \
    if (rc_ != BH_OK) return rc_; \
  } while (0)

void drop_graphs(Ctx* c) {
  for (auto& g : c->graphs) (void)hipGraphExecDestroy(g.exec);
  c->graphs.clear();
}

template <typename T>
int ensure(Ctx* c, DevBuf<T>& b, size_t n, const char* what) {
  if (n == 0) n = 1;
  if (b.cap >= n) return BH_OK;
  // a graph may still refer to the old buffer: forget every graph first
  drop_graphs(c);
  ++c->gen;
  if (b.p) {
    (void)hipStreamSynchronize(c->stream);
    (void)hipFree(b.p);
  }
  b.p = nullptr;
  b.cap = 0;
  const size_t want = n + n / 8;
  hipError_t e = hipMalloc(reinterpret_cast<void**>(&b.p), want * sizeof(T));
  if (e != hipSuccess) {
    (void)hipGetLastError();
    b.p = nullptr;
    set_err(c, "device allocation of %zu bytes for %s failed: %s", want * sizeof(T), what, hipGetErrorString(e));
    return BH_ERR_OOM;
  }
  b.cap = want;
  return BH_OK;
}

template <typename T>
void release(DevBuf<T>& b) {
  if (b.p) (void)hipFree(b.p);
  b.p = nullptr;
  b.cap = 0;
}

int check_args(Ctx* c, uint64_t n, const bh_force_params* fp, uint32_t max_leaf, uint32_t group_size) {
  if (n > kMaxN) {
    set_err(c, "n = %llu exceeds the supported %llu particles", (unsigned long long)n, (unsigned long long)kMaxN);
    return BH_ERR_TOO_LARGE;
  }
  if (max_leaf > kMaxLeafCap) {
    set_err(c, "max_leaf = %u exceeds the supported %u", max_leaf, kMaxLeafCap);
    return BH_ERR_TOO_LARGE;
  }
  if (group_size == 0) {
    set_err(c, "group_size 0 selects the per-node pass, which this library does not provide");
    return BH_ERR_INVALID;
  }
  if (fp && (!(fp->theta >= 0.0) || !(fp->eps2 >= 0.0) || !std::isfinite(fp->G) || !std::isfinite(fp->theta) ||
             !std::isfinite(fp->eps2))) {
    set_err(c, "invalid force parameters (theta %g, eps2 %g, G %g)", fp->theta, fp->eps2, fp->G);
    return BH_ERR_INVALID;
  }
  return BH_OK;
}

// What one wavefront walks of a system of n particles with targets of up to
// tsm: at most `unit` particles of a unit of several targets, `target` of one
// target. Larger pieces share more of a walk; smaller ones give a system that
// cannot fill the GPU more wavefronts and shorter last ones. A piece computes
// its particles from the same rounded coordinates as the whole unit would, and
// the rule knows the system alone, not what is stepped with it, so a batch
// gives each system the bytes of a step alone. The lines lie where a system
// alone gains most while large batches of such systems, which fill the GPU
// anyway, take no more than 2% longer than before (walk ms, leaf / target
// size in brackets, one system in whole units -> here; then a batch as it was
// before the walk's other changes -> here):
//   1,000 (16/32)    0.294 -> 0.076     2,000 systems 1.94 -> 1.94
//   4,096 (16/32)    0.430 -> 0.129       512 systems 3.17 -> 2.97
//   16,384 (16/32)   0.507 -> 0.191       200 systems 6.44 -> 6.50
//   16,384 (32/96)   0.536 -> 0.326       200 systems 5.56 -> 5.53
//   65,536 (16/32)   0.732 -> 0.329        64 systems 9.40 -> 9.22
//   65,536 (32/96)   0.668 -> 0.456        64 systems 8.48 -> 8.45
//   131,072 (32/96)  0.750 -> 0.591        32 systems 8.76 -> 8.67
//   250,007 (32/64)  1.229 -> 0.837        16 systems 9.33 -> 9.09
//   270,000 (32/64)  1.20 -> 0.93          16 systems 9.63 -> 9.51
//   400,003 (32/64)  1.35 -> 1.21          12 systems 10.59 -> 10.50
//   500,000 (32/64)  1.58 -> 1.47          16 systems 17.04 -> 17.37
//   500,000 (16/32)  1.665 -> 1.429        16 systems 18.75 -> 17.62
//   500,000 (32/96)  1.531 -> 1.466        16 systems 9.39 -> 9.31
//   1M (32/96) 3.06 -> 2.87; 1M uniform (8/32) 1.43 -> 1.33
// Above 2M whole units are the fastest (4M: 10.25 against 10.50 at 64). With
// the next class's {64, 64} the three rows of target size 64 would be 1.02, 1.30
// and 1.56 alone, but 9.29, 10.17 and 16.8 in the batches.
struct Pieces {
  uint16_t unit, target;
};
Pieces walk_pieces(uint64_t n, uint32_t tsm) {
  const bool narrow = tsm <= 32;
  if (n <= 4096) return narrow ? Pieces{16, 32} : Pieces{24, 32};
  if (n <= 16384) return narrow ? Pieces{16, 32} : Pieces{32, 48};
  if (n <= 65536) return narrow ? Pieces{24, 32} : Pieces{32, 48};
  if (n <= (256u << 10)) return Pieces{32, 64};
  if (n <= (512u << 10) && !narrow && tsm <= 64) return Pieces{32, 64};
  if (n <= (2u << 20)) return Pieces{64, 64};
  return Pieces{kGroupCap, kGroupCap};
}

// Pinned staging of the system table; with no_grow (the allocation-free
// step) it must already be large enough.
int host_table_room(Ctx* c, size_t bytes, bool no_grow) {
  if (c->host_tables_cap >= bytes) return BH_OK;
  if (no_grow) {
    set_err(c, "the system table needs %zu bytes of pinned staging, %zu were set up", bytes, c->host_tables_cap);
    return BH_ERR_TOO_LARGE;
  }
  drop_graphs(c);  // graphs copy the table from this buffer
  ++c->gen;
  if (c->host_tables) {
    (void)hipStreamSynchronize(c->stream);
    (void)hipHostFree(c->host_tables);
  }
  c->host_tables = nullptr;
  c->host_tables_cap = 0;
  const size_t want = bytes + bytes / 2;
  if (hipHostMalloc(reinterpret_cast<void**>(&c->host_tables), want, hipHostMallocDefault) != hipSuccess) {
    (void)hipGetLastError();
    set_err(c, "pinned host allocation of %zu bytes failed", want);
    return BH_ERR_OOM;
  }
  c->host_tables_cap = want;
  return BH_OK;
}

// The batch's system table: per-system parameters, chunks of <= kChunk
// particles for the per-system bounds, and the system-id digit counts of the
// sort's last passes, written to the pinned staging (the step's first kernel
// reads it there). Empty systems take no part: the device table lists the
// others, in order, and a particle's system id indexes that list.
int plan_systems(Ctx* c, const HostSys* sys, uint32_t S, bool no_grow, Plan* p) {
  if (S == 0 || S > kMaxSystems) {
    set_err(c, "a batch holds 1..%u systems, %u given", kMaxSystems, S);
    return BH_ERR_INVALID;
  }
  uint64_t n = 0, chunks = 0, largest = 0;
  uint32_t mlx = 0, live = 0;
  bool unsoftened = false;
  double nodes = 0.0;
  for (uint32_t k = 0; k < S; ++k) {
    TRY(check_args(c, sys[k].n, &sys[k].fp, sys[k].max_leaf, sys[k].group_size));
    if (sys[k].tile && (sys[k].tile < kMinTile || sys[k].tile > kGroupCap)) {
      set_err(c, "walk tile %u outside %u..%u", sys[k].tile, kMinTile, kGroupCap);
      return BH_ERR_INVALID;
    }
    if (sys[k].n == 0) continue;
    ++live;
    n += sys[k].n;
    mlx = std::max(mlx, sys[k].max_leaf);
    largest = std::max(largest, sys[k].n);
    unsoftened |= static_cast<float>(sys[k].fp.eps2) == 0.0f;  // zero in the FP32 walk too
    // nodes per particle of Plummer, Hernquist and uniform trees: at most
    // min(1.6, 4 / max_leaf), with a quarter to spare
    nodes += 1.25 * static_cast<double>(sys[k].n) * std::min(1.6, 4.0 / std::max(1u, sys[k].max_leaf)) + 64.0;
  }
  if (n > kMaxN) {
    set_err(c, "batch of %llu particles exceeds the supported %llu", (unsigned long long)n, (unsigned long long)kMaxN);
    return BH_ERR_TOO_LARGE;
  }
  // up to 256 chunks of a quarter, so that a small system's bounds reach
  // more CUs; the allocation-free step's table has room for full ones
  const uint32_t chunk = !no_grow && n <= 64 * kChunk ? kChunk / 4 : kChunk;
  for (uint32_t k = 0; k < S; ++k) chunks += (sys[k].n + chunk - 1) / chunk;
  *p = Plan{};
  p->n = static_cast<uint32_t>(n);
  p->chunk = chunk;
  // (the allocation-free step's scratch has room for the larger tiles' words)
  if (!no_grow) p->sort_tile = sort_tile(p->n);
  p->largest = largest;
  if (n == 0) return BH_OK;
  p->S = live;
  p->n_chunks = static_cast<uint32_t>(chunks);
  p->mlx = mlx;
  p->sid_passes = live == 1 ? 0 : (live <= 256 ? 1 : 2);
  p->unsoftened = unsoftened;
  p->node_estimate = static_cast<uint64_t>(nodes);
  p->off_chunks = sizeof(SysDev) * live;
  p->off_first = p->off_chunks + sizeof(uint4) * chunks;
  p->off_hist = (p->off_first + 4 * (live + 1) + 15) / 16 * 16;
  p->table_bytes = p->off_hist + 2 * 256 * 4;
  TRY(host_table_room(c, p->table_bytes, no_grow));
  std::memset(c->host_tables, 0, p->table_bytes);
  SysDev* sd = reinterpret_cast<SysDev*>(c->host_tables);
  uint4* ch = reinterpret_cast<uint4*>(c->host_tables + p->off_chunks);
  uint32_t* first = reinterpret_cast<uint32_t*>(c->host_tables + p->off_first);
  uint32_t* hist = reinterpret_cast<uint32_t*>(c->host_tables + p->off_hist);
  uint64_t off = 0, ci = 0;
  for (uint32_t k = 0, src = 0; k < live; ++k, ++src) {
    while (sys[src].n == 0) ++src;
    const HostSys& h = sys[src];
    sd[k].theta2 = h.fp.theta * h.fp.theta;
    sd[k].eps2 = h.fp.eps2;
    sd[k].G = h.fp.G;
    sd[k].kick_dt = h.kick_dt;
    sd[k].drift_dt = h.drift_dt;
    sd[k].off = static_cast<uint32_t>(off);
    sd[k].n = static_cast<uint32_t>(h.n);
    sd[k].max_leaf = h.max_leaf;
    sd[k].tsm = std::min(h.target_size, h.group_size);
    sd[k].use_quad = h.fp.use_quadrupole != 0;
    sd[k].tile = static_cast<uint16_t>(h.tile ? h.tile : c->walk_tile);
    const Pieces pieces = walk_pieces(h.n, sd[k].tsm);
    sd[k].unit_piece = pieces.unit;
    sd[k].target_piece = pieces.target;
    first[k] = static_cast<uint32_t>(ci);
    for (uint64_t b = 0; b < h.n; b += chunk)
      ch[ci++] = make_uint4(k, static_cast<uint32_t>(off + b), static_cast<uint32_t>(off + std::min<uint64_t>(h.n, b + chunk)), 0);
    hist[k & 255] += static_cast<uint32_t>(h.n);
    hist[256 + (k >> 8)] += static_cast<uint32_t>(h.n);
    off += h.n;
  }
  first[live] = static_cast<uint32_t>(ci);
  // single-system queries (export, accel) read the first system's shape
  for (uint32_t k = 0; k < S; ++k) {
    if (sys[k].n == 0) continue;
    c->max_leaf = sys[k].max_leaf;
    c->group_size = sys[k].group_size;
    break;
  }
  return BH_OK;
}

// Walk workgroups: enough to fill the GPU (4 waves on every SIMD), fewer for
// small inputs; always a multiple of 8 (one share per XCD).
uint32_t walk_slots(uint32_t n, uint32_t limit) {
  uint32_t s = (n + 7) / 8;
  s = std::min(s, limit);
  s = std::max(s, 8u);
  return (s + 7) / 8 * 8;
}

// Radix passes over the leading key bits of systems of up to n particles.
// 8 p bits are 10, 13 or 16 octree levels (p = 4, 5, 6); the runs of particles
// that share them are ordered by one more pass, so the cells of that level
// should hold few: the centre of a Hernquist sphere (density 1 / r, radius up
// to 20), the most clustered of the initial conditions, has 5 particles in
// such a cell at 32,768, 8 at 2M, 1 at 16M. A pass is 6 to 8 us up to 64
// tiles, 20 at 1M and 134 at 16M.
int sort_passes(uint64_t n) { return n <= 32768 ? 4 : n <= (2u << 20) ? 5 : 6; }

// The plan's sizes that depend on what the context has learnt.
void plan_shape(Ctx* c, Plan* p, bool walk, bool full_sort) {
  p->walk = walk;
  p->key_passes = full_sort ? 8 : sort_passes(p->largest);
  const uint64_t want = std::max<uint64_t>(p->node_estimate, c->cap_nodes);
  p->cap_nodes = static_cast<uint32_t>(std::min<uint64_t>(want, 1ull << 30));
  p->depth_plan = c->depth_known ? c->depth_hint : static_cast<uint32_t>(kDepthCap);
  p->deep = p->depth_plan + 1 > kShallowFrames;
  p->slots = walk_slots(p->n, kWalkSlots);
}

// Grows the context's buffers to the plan and points `b` at them.
int provision(Ctx* c, const Plan& p, Scratch* b) {
  const uint32_t n = p.n, m = p.cap_nodes;
  const uint32_t tiles = (n + kTreeTile - 1) / kTreeTile;
  TRY(ensure(c, c->keys_a, n, "keys"));
  TRY(ensure(c, c->keys_b, n, "keys"));
  TRY(ensure(c, c->vals_a, n, "indices"));
  TRY(ensure(c, c->vals_b, n, "indices"));
  TRY(ensure(c, c->hist, 10 * 256, "histograms"));
  TRY(ensure(c, c->lookback, radix_lookback_words(n, p.sort_tile, 10), "look-back"));
  TRY(ensure(c, c->lohi, 6ull * p.S, "bounds"));
  TRY(ensure(c, c->partial, 6ull * p.n_chunks, "bounds"));
  TRY(ensure(c, c->misc, kReportWords, "flags"));
  TRY(ensure(c, c->posm, n, "walk copy"));
  TRY(ensure(c, c->L, n, "tree build"));
  TRY(ensure(c, c->H, n, "tree build"));
  TRY(ensure(c, c->tcounts, uint64_t(tiles) * kTreeCols, "tree build"));
  TRY(ensure(c, c->tprefix, uint64_t(tiles) * kTreeCols, "tree build"));
  TRY(ensure(c, c->level_off, kLevels + 2, "tree levels"));
  TRY(ensure(c, c->sid, n, "system ids"));
  TRY(ensure(c, c->tables, p.table_bytes, "system table"));
  TRY(ensure(c, c->begin, m, "nodes"));
  TRY(ensure(c, c->count, m, "nodes"));
  TRY(ensure(c, c->cs, m, "nodes"));
  TRY(ensure(c, c->first_child, m, "nodes"));
  TRY(ensure(c, c->parent, m, "nodes"));
  TRY(ensure(c, c->leaf_idx, m, "nodes"));
  TRY(ensure(c, c->depth, m, "nodes"));
  TRY(ensure(c, c->leaf, m, "nodes"));
  TRY(ensure(c, c->nchild, m, "nodes"));
  TRY(ensure(c, c->ctr, m, "nodes"));
  TRY(ensure(c, c->rec, m, "nodes"));
  TRY(ensure(c, c->mass, m, "nodes"));
  TRY(ensure(c, c->com, 3ull * m, "nodes"));
  TRY(ensure(c, c->iab, 6ull * m, "nodes"));
  TRY(ensure(c, c->q64, 8ull * m, "nodes"));
  TRY(ensure(c, c->nbox, 6ull * m, "nodes"));
  TRY(ensure(c, c->leaf_node, m, "leaves"));
  TRY(ensure(c, c->leaf_first, m, "leaves"));
  if (p.carry_out || p.carried_in) {
    TRY(ensure(c, c->carry, 4ull * n, "carried positions"));
    TRY(ensure(c, c->carry_flag, 1, "carried positions"));
  }
  if (p.walk) {
    TRY(ensure(c, c->mark, n, "targets"));
    TRY(ensure(c, c->gmark, n, "walk units"));
    TRY(ensure(c, c->units, n, "walk units"));
    TRY(ensure(c, c->unit_lb, unit_list_words(n), "walk units"));
    TRY(ensure(c, c->unit_n, m, "walk units"));
    TRY(ensure(c, c->gacc, 3ull * n, "group sums"));
    TRY(ensure(c, c->defer, uint64_t(p.slots) * kDefer, "deferred nodes"));
    if (p.deep) TRY(ensure(c, c->deep_frames, uint64_t(p.slots) * (kLevels - kShallowFrames) * kWave, "walk stack"));
  }
  Scratch& s = *b;
  s = Scratch{};
  s.keys_a = c->keys_a.p;
  s.keys_b = c->keys_b.p;
  s.vals_a = c->vals_a.p;
  s.vals_b = c->vals_b.p;
  s.hist = c->hist.p;
  s.lookback = c->lookback.p;
  s.lohi = c->lohi.p;
  s.partial = c->partial.p;
  s.misc = c->misc.p;
  s.totals = reinterpret_cast<unsigned long long*>(s.misc + kMiscTotals);
  s.posm = c->posm.p;
  s.L = c->L.p;
  s.H = c->H.p;
  s.tcounts = c->tcounts.p;
  s.tprefix = c->tprefix.p;
  s.sid = c->sid.p;
  s.tables = c->tables.p;
  TreeDev& t = s.t;
  t.begin = c->begin.p;
  t.count = c->count.p;
  t.depth = c->depth.p;
  t.leaf = c->leaf.p;
  t.cs = c->cs.p;
  t.first_child = c->first_child.p;
  t.nchild = c->nchild.p;
  t.parent = c->parent.p;
  t.leaf_idx = c->leaf_idx.p;
  t.ctr = c->ctr.p;
  t.mass = c->mass.p;
  t.com = c->com.p;
  t.iab = c->iab.p;
  t.rec = c->rec.p;
  t.q64 = c->q64.p;
  t.nbox = c->nbox.p;
  t.leaf_node = c->leaf_node.p;
  t.leaf_first = c->leaf_first.p;
  t.level_off = c->level_off.p;
  t.misc = c->misc.p;
  t.cap = m;
  if (p.walk) {
    s.mark = c->mark.p;
    s.gmark = c->gmark.p;
    s.units = c->units.p;
    s.unit_lb = c->unit_lb.p;
    s.unit_n = c->unit_n.p;
    s.gacc = c->gacc.p;
    s.defer = c->defer.p;
    s.deep_frames = p.deep ? c->deep_frames.p : nullptr;
  }
  return BH_OK;
}

// Cuts the plan's arrays out of a fixed block of device memory, in the
// order and sizes of provision(), with the node capacity set to whatever is
// left. Fails (returns false) when the per-particle arrays do not fit.
bool carve(uint8_t* base, size_t bytes, Plan* p, Scratch* b) {
  size_t off = 0;
  bool ok = true;
  auto take = [&](size_t sz) -> uint8_t* {
    off = (off + 255) / 256 * 256;
    uint8_t* q = base + off;
    if (off + sz > bytes) ok = false;
    off += sz;
    return q;
  };
  const uint32_t n = p->n;
  const uint32_t tiles = (n + kTreeTile - 1) / kTreeTile;
  Scratch& s = *b;
  s = Scratch{};
  s.keys_a = reinterpret_cast<uint64_t*>(take(8ull * n));
  s.keys_b = reinterpret_cast<uint64_t*>(take(8ull * n));
  s.vals_a = reinterpret_cast<uint32_t*>(take(4ull * n));
  s.vals_b = reinterpret_cast<uint32_t*>(take(4ull * n));
  s.hist = reinterpret_cast<uint32_t*>(take(4 * 10 * 256));
  s.lookback = reinterpret_cast<uint32_t*>(take(4 * radix_lookback_words(n, p->sort_tile, 10)));
  s.lohi = reinterpret_cast<double*>(take(48ull * p->S));
  s.partial = reinterpret_cast<double*>(take(48ull * p->n_chunks));
  s.misc = reinterpret_cast<uint32_t*>(take(4 * kReportWords));
  s.totals = reinterpret_cast<unsigned long long*>(s.misc + kMiscTotals);
  s.posm = reinterpret_cast<double4*>(take(32ull * n));
  s.L = take(n);
  s.H = take(n);
  s.tcounts = reinterpret_cast<uint32_t*>(take(4ull * tiles * kTreeCols));
  s.tprefix = reinterpret_cast<uint32_t*>(take(4ull * tiles * kTreeCols));
  s.sid = reinterpret_cast<uint16_t*>(take(2ull * n));
  s.tables = take(p->table_bytes);
  s.mark = reinterpret_cast<uint32_t*>(take(4ull * n));
  s.gmark = reinterpret_cast<uint32_t*>(take(4ull * n));
  s.units = reinterpret_cast<uint2*>(take(8ull * n));
  s.unit_lb = s.tcounts;  // the tree's tile counts are free by then
  s.gacc = reinterpret_cast<double*>(take(24ull * n));
  s.defer = reinterpret_cast<uint32_t*>(take(4ull * p->slots * kDefer));
  s.deep_frames = reinterpret_cast<uint32_t*>(take(4ull * p->slots * (kLevels - kShallowFrames) * kWave));
  TreeDev& t = s.t;
  t.level_off = reinterpret_cast<uint32_t*>(take(4 * (kLevels + 2)));
  t.misc = s.misc;
  if (!ok) return false;
  // node arrays: 327 bytes per node, plus alignment of the 19 arrays
  const size_t per_node = 4 * 6 + 3 + 32 + 64 + 8 + 24 + 48 + 64 + 48 + 4 * 3;
  off = (off + 255) / 256 * 256;
  const size_t left = bytes > off + 19 * 256 ? bytes - off - 19 * 256 : 0;
  const uint64_t m = std::min<uint64_t>(left / per_node, 1ull << 30);
  if (m < 64) return false;
  t.begin = reinterpret_cast<uint32_t*>(take(4 * m));
  t.count = reinterpret_cast<uint32_t*>(take(4 * m));
  t.cs = reinterpret_cast<uint32_t*>(take(4 * m));
  t.first_child = reinterpret_cast<uint32_t*>(take(4 * m));
  t.parent = reinterpret_cast<uint32_t*>(take(4 * m));
  t.leaf_idx = reinterpret_cast<uint32_t*>(take(4 * m));
  t.depth = take(m);
  t.leaf = take(m);
  t.nchild = take(m);
  t.ctr = reinterpret_cast<double4*>(take(32 * m));
  t.rec = reinterpret_cast<NodeRec*>(take(64 * m));
  t.mass = reinterpret_cast<double*>(take(8 * m));
  t.com = reinterpret_cast<double*>(take(24 * m));
  t.iab = reinterpret_cast<double*>(take(48 * m));
  t.q64 = reinterpret_cast<double*>(take(64 * m));
  t.nbox = reinterpret_cast<double*>(take(48 * m));
  t.leaf_node = reinterpret_cast<uint32_t*>(take(4 * m));
  t.leaf_first = reinterpret_cast<uint32_t*>(take(4 * m));
  s.unit_n = reinterpret_cast<uint32_t*>(take(4 * m));
  t.cap = static_cast<uint32_t>(m);
  p->cap_nodes = t.cap;
  return ok;
}

struct Sorted {
  uint64_t* keys = nullptr;
  uint32_t* perm = nullptr;
};

// build_flat_tree (flat_build_ttg.h:276-281) of every system of the plan,
// d_in[0..n) into the scratch; the Morton-ordered particles (each system in
// its own range) go to d_out, here or (walk_writes_out) by the step's walk,
// which reads them from d_in.
int enqueue_build(Ctx* c, const Plan& p, const Scratch& b, const bh_particle* d_in, bh_particle* d_out, Sorted* out,
                  bool walk_writes_out) {
  hipStream_t s = c->stream;
  const uint32_t n = p.n;
  const SysDev* sys = reinterpret_cast<const SysDev*>(b.tables);
  StartArgs a{};
  a.host_table = reinterpret_cast<const uint4*>(c->host_tables);
  a.table = reinterpret_cast<uint4*>(b.tables);
  a.table_quads = static_cast<uint32_t>(p.off_hist / sizeof(uint4));
  if (p.sid_passes) a.host_hist = reinterpret_cast<const uint4*>(c->host_tables + p.off_hist);
  a.hist = reinterpret_cast<uint4*>(b.hist + 8 * 256);
  // the step's flag words and totals, key digit histograms and look-back
  // words, and the walk's marks
  a.zero.p[0] = b.misc;
  a.zero.n[0] = kMiscStamps;
  if (p.walk) {
    a.zero.p[1] = b.mark;
    a.zero.n[1] = n;
    a.zero.p[2] = b.gmark;
    a.zero.n[2] = n;
  }
  if (!small(p)) {
    a.zero.p[3] = b.hist;
    a.zero.n[3] = 8 * 256;
    a.zero.p[4] = b.lookback;
    a.zero.n[4] = radix_lookback_words(n, p.sort_tile, p.key_passes + p.sid_passes);
  }
  a.host_chunks = reinterpret_cast<const uint4*>(c->host_tables + p.off_chunks);
  a.chunk_first = reinterpret_cast<const uint32_t*>(b.tables + p.off_first);
  a.n_chunks = p.n_chunks;
  a.n_sys = p.S;
  a.n = n;
  a.chunk = p.chunk;
  a.sid = b.sid;
  a.partial = b.partial;
  a.lohi = b.lohi;
  a.misc = b.misc;
  if (small(p)) {
    out->keys = b.keys_a;
    out->perm = b.vals_a;
    double4* posm = walk_writes_out ? b.posm : nullptr;
    if (p.carried_in)
      HIP_OK(c, launch_small_sort(c->carry.p, c->carry_flag.p, a, out->keys, out->perm, b.keys_b, b.vals_b, posm, s));
    else
      HIP_OK(c, launch_small_sort(d_in, a, out->keys, out->perm, b.keys_b, b.vals_b, posm, s));
    if (!walk_writes_out) HIP_OK(c, launch_gather(d_in, d_out, out->perm, b.posm, n, s));
  } else {
    if (p.carried_in) {
      HIP_OK(c, launch_start(c->carry.p, c->carry_flag.p, a, s));
      HIP_OK(c, launch_keys_hist(c->carry.p, n, p.key_passes, b.sid, b.lohi, b.keys_a, b.hist, s));
    } else {
      HIP_OK(c, launch_start(d_in, a, s));
      HIP_OK(c, launch_keys_hist(d_in, n, p.key_passes, b.sid, b.lohi, b.keys_a, b.hist, s));
    }
    HIP_OK(c, launch_radix_sort(b.keys_a, b.vals_a, b.keys_b, b.vals_b, n, p.sort_tile, p.key_passes, p.sid_passes, b.sid,
                                b.hist, b.lookback, b.misc + kMiscAbort, &out->keys, &out->perm, s));
    if (p.carried_in && walk_writes_out)
      HIP_OK(c, launch_gather(c->carry.p, out->perm, b.posm, n, s));
    else
      HIP_OK(c, launch_gather(d_in, walk_writes_out ? nullptr : d_out, out->perm, b.posm, n, s));
  }
  HIP_OK(c, launch_tree_count(out->keys, n, b.sid, sys, p.mlx, b.L, b.H, b.tcounts, b.misc, s));
  HIP_OK(c, launch_tree_emit(b.L, b.H, n, b.tcounts, b.tprefix, b.t, p.depth_plan, s));
  // what the walk needs zeroed and could not be before: unit_lb may lie over
  // tcounts, the queue heads over the look-back words, and the carried flag
  // has been read
  ZeroRanges z;
  if (p.walk) {
    z.p[0] = b.unit_lb;
    z.n[0] = unit_list_words(n);
    z.p[1] = walk_queue(b);
    z.n[1] = kQueueWords;
  }
  if (p.walk && p.carry_out) {
    z.p[2] = c->carry_flag.p;
    z.n[2] = 1;
  }
  HIP_OK(c, launch_tree_finish(out->keys, b.posm, n, b.sid, p.S, b.lohi, p.depth_plan, z, b.t, s));
  return BH_OK;
}

// run_grouped_pass (grouped_ttg.h:297-323) over every system of the tree in
// the scratch, with each system's parameters from the system table. The build
// zeroed what it and the unit list need zero.
int enqueue_walk(Ctx* c, const Plan& p, const Scratch& b, bh_particle* parts, double* d_acc, uint32_t* d_npp,
                 uint32_t* d_npc, const bh_particle* src = nullptr, const uint32_t* perm = nullptr) {
  hipStream_t s = c->stream;
  const uint32_t n = p.n;
  const SysDev* sys = reinterpret_cast<const SysDev*>(b.tables);
  const bool grouped = c->walk_mode == BH_WALK_GROUPED;
  // per-target mode: the walk units are the targets themselves
  HIP_OK(c, launch_units(b.t, n, b.sid, sys, grouped, b.mark, b.gmark, b.unit_n, b.unit_lb, b.units, s));
  WalkArgs a;
  a.rec = b.t.rec;
  a.q64 = b.t.q64;
  a.ctr = b.t.ctr;
  a.begin = b.t.begin;
  a.count = b.t.count;
  a.posm = b.posm;
  a.units = b.units;
  a.unit_n = grouped ? b.unit_n : nullptr;
  a.tmark = b.mark;
  a.sid = b.sid;
  a.sys = sys;
  a.gacc = b.gacc;
  a.nbox = b.t.nbox;
  a.defer = b.defer;
  a.deep_frames = p.deep ? b.deep_frames : nullptr;
  a.misc = b.misc;
  a.queue = walk_queue(b);
  a.n_nodes = p.cap_nodes;
  a.n_parts = n;
  a.stack_limit = c->stack_limit;
  a.parts = parts;
  a.src = src;
  a.perm = perm;
  a.carry = nullptr;
  a.carry_bad = nullptr;
  if (parts && p.carry_out) {
    a.carry = c->carry.p;
    a.carry_bad = c->carry_flag.p;
  }
  a.acc = d_acc;
  a.n_pp = d_npp;
  a.n_pc = d_npc;
  a.totals = b.totals;
  HIP_OK(c, launch_walk(a, p.slots, p.deep, c->precision == BH_FP64, p.unsoftened, s));
  return BH_OK;
}

int enqueue_report(Ctx* c, const Scratch& b) {
  HIP_OK(c, launch_report(b.misc, c->host_misc, c->stream));
  return BH_OK;
}

// Waits for the stream, whose last kernel wrote the report: the step's only
// synchronisation.
int finish(Ctx* c) {
  HIP_OK(c, hipStreamSynchronize(c->stream));
  std::memcpy(c->stamps, c->host_misc + kMiscStamps, sizeof c->stamps);
  return BH_OK;
}

// Milliseconds from the beginning of one phase of the last step to another's.
double phase_ms(const Ctx* c, Stamp from, Stamp to) {
  return static_cast<double>(c->stamps[to] - c->stamps[from]) / c->clock_khz;
}

GraphKey graph_key(const Ctx* c, const Plan& p, const void* in, const void* out) {
  GraphKey k;
  std::memset(&k, 0, sizeof k);
  k.in = in;
  k.out = out;
  k.gen = c->gen;
  k.n = p.n;
  k.S = p.S;
  k.n_chunks = p.n_chunks;
  k.mlx = p.mlx;
  k.cap_nodes = p.cap_nodes;
  k.depth_plan = p.depth_plan;
  k.slots = p.slots;
  k.table_bytes = static_cast<uint32_t>(p.table_bytes);
  k.deep = p.deep;
  k.unsoftened = p.unsoftened;
  k.precision = static_cast<uint8_t>(c->precision);
  k.mode = static_cast<uint8_t>(c->walk_mode);
  k.carry_out = p.carry_out ? 1 : 0;
  k.carried_in = p.carried_in ? 1 : 0;
  k.key_passes = static_cast<uint8_t>(p.key_passes);
  return k;
}

// The step as one graph launch: replays the graph captured for the same
// launches, or captures and instantiates it first (the least recently used
// of kGraphCache graphs makes room).
int launch_graph(Ctx* c, const Plan& p, const Scratch& b, const bh_particle* d_in, bh_particle* d_out, Sorted* sorted) {
  const GraphKey key = graph_key(c, p, d_in, d_out);
  GraphEntry* hit = nullptr;
  for (auto& g : c->graphs)
    if (g.key == key) hit = &g;
  // the sort's output buffers follow from the pass count alone
  const int passes = small(p) ? 0 : p.key_passes + p.sid_passes;
  sorted->keys = (passes % 2 == 0) ? b.keys_a : b.keys_b;
  sorted->perm = (passes % 2 == 0) ? b.vals_a : b.vals_b;
  if (!hit) {
    HIP_OK(c, hipStreamBeginCapture(c->stream, hipStreamCaptureModeRelaxed));
    Sorted sd;
    int rc = enqueue_build(c, p, b, d_in, d_out, &sd, true);
    if (rc == BH_OK) rc = enqueue_walk(c, p, b, d_out, nullptr, nullptr, nullptr, d_in, sd.perm);
    if (rc == BH_OK) rc = enqueue_report(c, b);
    hipGraph_t graph = nullptr;
    const hipError_t ec = hipStreamEndCapture(c->stream, &graph);
    if (rc != BH_OK) {
      if (graph) (void)hipGraphDestroy(graph);
      return rc;
    }
    HIP_OK(c, ec);
    hipGraphExec_t exec = nullptr;
    const hipError_t ei = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
    (void)hipGraphDestroy(graph);
    HIP_OK(c, ei);
    if (sd.keys != sorted->keys || sd.perm != sorted->perm) {
      (void)hipGraphExecDestroy(exec);
      set_err(c, "radix sort output buffers differ from the pass-count rule");
      return BH_ERR_HIP;
    }
    if (c->graphs.size() >= kGraphCache) {
      auto lru = std::min_element(c->graphs.begin(), c->graphs.end(),
                                  [](const GraphEntry& x, const GraphEntry& y) { return x.used < y.used; });
      (void)hipGraphExecDestroy(lru->exec);
      c->graphs.erase(lru);
    }
    c->graphs.push_back(GraphEntry{key, exec, 0});
    hit = &c->graphs.back();
  }
  hit->used = ++c->graph_clock;
  HIP_OK(c, hipGraphLaunch(hit->exec, c->stream));
  return BH_OK;
}

// Keeps the report of a finished step or build.
void take_report(Ctx* c, const Plan& p, const Scratch& b, const Sorted& sd, bh_particle* d_out, bool walked) {
  const uint32_t* m = c->host_misc;
  uint64_t nodes = 0;
  for (int d = 0; d < kLevels; ++d) nodes += m[kMiscLevels + d];
  c->n = p.n;
  c->n_nodes = static_cast<uint32_t>(nodes);
  c->n_leaves = m[kMiscLevels + kLevels];
  c->max_depth = m[kMiscMaxDepth];
  if (walked) {
    c->n_targets = m[kMiscTargets];
    c->n_groups = m[kMiscGroups];
    std::memcpy(c->last_totals, m + kMiscWords, sizeof c->last_totals);
  }
  c->plan = p;
  c->sc = b;
  c->sorted = d_out;
  c->keys_sorted = sd.keys;
  c->perm_sorted = sd.perm;
}

// A step (walk = true) or tree build of the systems planned in the pinned
// table, on the context's buffers: eagerly or as a graph, then the report.
// A tree that outgrew the plan is built again with room for it.
int run(Ctx* c, Plan p, const bh_particle* d_in, bh_particle* d_out, bool walk, bh_step_timing* timing) {
  c->have_stats = false;
  c->has_tree = false;
  c->carried_ok = false;
  bool full_sort = c->full_sort > 0 && !small(p);
  if (full_sort) --c->full_sort;
  for (int attempt = 0;; ++attempt) {
    c->reruns = static_cast<uint32_t>(attempt);
    plan_shape(c, &p, walk, full_sort);
    Scratch b;
    TRY(provision(c, p, &b));
    Sorted sd;
    const bool graph = walk && c->graph_mode == BH_GRAPH_ON;
    if (graph) {
      TRY(launch_graph(c, p, b, d_in, d_out, &sd));
    } else {
      TRY(enqueue_build(c, p, b, d_in, d_out, &sd, walk));
      if (walk) TRY(enqueue_walk(c, p, b, d_out, nullptr, nullptr, nullptr, d_in, sd.perm));
      TRY(enqueue_report(c, b));
    }
    TRY(finish(c));
    const uint32_t* m = c->host_misc;
    if (m[kMiscNonfinite]) {
      set_err(c, "non-finite position, velocity or mass in the input");
      return BH_ERR_NONFINITE;
    }
    const uint32_t abort = m[kMiscAbort];
    if (abort) {
      if (attempt >= 3) {
        set_err(c, "the tree outgrew its planned arrays on every attempt (abort word %u)", abort);
        return BH_ERR_HIP;
      }
      if (abort & kAbortSort) {
        // the tree was counted on keys that are not in order: many times the
        // nodes (1M particles and a far one: 2.9M for 0.2M) and too many levels
        full_sort = true;
        c->full_sort = c->full_span;
        c->full_span = std::min(2 * c->full_span, kFullStepsMost);
        continue;
      }
      if (abort & kAbortNodes) {
        uint64_t need = m[kMiscLevels + kLevels];
        uint64_t nodes = 0;
        for (int d = 0; d < kLevels; ++d) nodes += m[kMiscLevels + d];
        need = std::max(need, nodes);
        c->cap_nodes = static_cast<uint32_t>(std::min<uint64_t>(need + need / 8 + 64, 1ull << 30));
      }
      if (abort & kAbortDepth) {
        c->depth_hint = std::max(c->depth_known ? c->depth_hint : 0u, m[kMiscMaxDepth]);
        c->depth_known = true;
      }
      continue;
    }
    if (!full_sort && !small(p)) c->full_span = kFullSteps;
    // later steps plan for the deepest tree seen
    c->depth_hint = c->depth_known ? std::max(c->depth_hint, m[kMiscMaxDepth]) : m[kMiscMaxDepth];
    c->depth_known = true;
    take_report(c, p, b, sd, d_out, walk);
    c->has_tree = true;
    c->have_stats = walk;
    c->last_graph = graph;
    if (timing) {
      if (graph) {
        timing->tree_build_ms = 0.0;
        timing->traversal_ms = phase_ms(c, kStampStart, kStampEnd);  // of a graph the whole step is reported
      } else {
        timing->tree_build_ms = phase_ms(c, kStampStart, walk ? kStampTargets : kStampEnd);
        timing->traversal_ms = walk ? phase_ms(c, kStampTargets, kStampEnd) : 0.0;
      }
      timing->exchange_ms = 0.0;
    }
    if (walk && m[kMiscIncomplete]) {
      set_err(c, "incomplete tree: the walk met an interior node it could not open");
      return BH_ERR_INCOMPLETE;
    }
    if (walk && p.carry_out) {
      c->carried_ok = true;
      c->carried_out = d_out;
      c->carried_n = p.n;
    }
    return BH_OK;
  }
}

// One step of a batch: systems sys[0..S) own consecutive ranges of d_in.
// resident: a step of the resident state; its walk keeps the output's
// compact positions, which the next resident step builds from when its input
// is that output and nothing else ran in between.
int step_batch(Ctx* c, const bh_particle* d_in, bh_particle* d_out, const HostSys* sys, uint32_t S, bh_step_timing* timing,
               bool resident = false) {
  if (timing) *timing = bh_step_timing{0.0, 0.0, 0.0};
  HIP_OK(c, hipSetDevice(c->device));
  Plan p;
  TRY(plan_systems(c, sys, S, false, &p));
  if (p.n == 0) return BH_OK;
  p.carry_out = resident;
  p.carried_in = resident && c->carried_ok && c->carried_out == d_in && c->carried_n == p.n;
  return run(c, p, d_in, d_out, true, timing);
}

int step_device(Ctx* c, const bh_particle* d_in, bh_particle* d_out, uint64_t n, const bh_force_params* fp,
                uint32_t max_leaf, uint32_t group_size, uint32_t target_size, double kick_dt, double drift_dt,
                bh_step_timing* timing, bool resident = false) {
  TRY(check_args(c, n, fp, max_leaf, group_size));
  if (n == 0) {
    if (timing) *timing = bh_step_timing{0.0, 0.0, 0.0};
    return BH_OK;
  }
  const HostSys one{n, *fp, max_leaf, group_size, target_size, kick_dt, drift_dt, 0};
  return step_batch(c, d_in, d_out, &one, 1, timing, resident);
}

std::vector<HostSys> host_systems(const bh_system* systems, uint32_t S) {
  std::vector<HostSys> v(S);
  for (uint32_t k = 0; k < S; ++k)
    v[k] = HostSys{systems[k].n,         systems[k].fp,      systems[k].max_leaf,
                   systems[k].group_size, systems[k].target_size, systems[k].kick_dt,
                   systems[k].drift_dt, systems[k].walk_tile};
  return v;
}

bool overlap(const bh_particle* a, const bh_particle* b, uint64_t n) { return n && a + n > b && b + n > a; }

Ctx* as(bh_ctx* c) { return reinterpret_cast<Ctx*>(c); }

}  // namespace

int bhk::ctx_device(const bh_ctx* c) { return c ? reinterpret_cast<const Ctx*>(c)->device : 0; }

namespace {

// Reference node numbering (flat_build_ttg.h:194-273): BFS backbone down to
// subtree roots (count <= 4096 or leaf), then each subtree's other nodes BFS
// in subtree-root order; group roots in push order (flat_tree.h:190-225).
void reference_order(const std::vector<uint32_t>& count, const std::vector<uint8_t>& leaf,
                     const std::vector<uint32_t>& first_child, const std::vector<uint8_t>& nchild, uint32_t group_size,
                     std::vector<uint32_t>& ref_of, std::vector<uint32_t>& groups) {
  const size_t m = count.size();
  ref_of.assign(m, 0);
  groups.clear();
  auto group_root = [&](uint32_t u, uint32_t parent_count) {
    return (leaf[u] || count[u] <= group_size) && parent_count > group_size;
  };
  std::vector<uint32_t> bb{0};
  ref_of[0] = 0;
  if (group_root(0, std::numeric_limits<uint32_t>::max())) groups.push_back(0);
  std::vector<uint32_t> sroots;
  for (size_t i = 0; i < bb.size(); ++i) {
    const uint32_t u = bb[i];
    if (count[u] <= 4096 || leaf[u]) {
      sroots.push_back(u);
      continue;
    }
    for (uint32_t k = 0; k < nchild[u]; ++k) {
      const uint32_t ch = first_child[u] + k;
      ref_of[ch] = static_cast<uint32_t>(bb.size());
      bb.push_back(ch);
      if (group_root(ch, count[u])) groups.push_back(ch);
    }
  }
  uint32_t next = static_cast<uint32_t>(bb.size());
  std::vector<uint32_t> sub;
  for (uint32_t r : sroots) {
    sub.clear();
    sub.push_back(r);
    for (size_t k = 0; k < sub.size(); ++k) {
      const uint32_t u = sub[k];
      if (leaf[u]) continue;
      for (uint32_t q = 0; q < nchild[u]; ++q) {
        const uint32_t ch = first_child[u] + q;
        ref_of[ch] = next++;
        sub.push_back(ch);
        if (group_root(ch, count[u])) groups.push_back(ch);
      }
    }
  }
}

// Positions and masses of n host records in c->dsrc. The records go over as
// they are, a bounded piece at a time, and the GPU picks the fields: packing
// them on the host took 9 ns a particle, 7 of 9 ms at 1M. Up to kFewPoints
// they are packed all the same, which saves a launch and takes no longer
// (energies of 2 particles 43.1 -> 40.7 us, 100 47.8 -> 45.5, 1,024 52.9 -> 50.5).
constexpr uint64_t kLoadPiece = 1u << 20;
// A copy of more than 1 MiB from pageable memory takes another path in the
// runtime, which costs 20 us more than it saves up to 1.5 MiB: two copies there
// (energies of 17,000 particles 0.280 -> 0.267 ms, 20,000 0.300 -> 0.292; direct
// sum of 256 over 20,000 0.126 -> 0.112; three copies for 30,000: 0.162 -> 0.186).
constexpr uint64_t kOneCopy = (1u << 20) / sizeof(bh_particle);
constexpr uint64_t kTwoCopies = kOneCopy * 3 / 2;

int load_points(Ctx* c, const bh_particle* host, uint64_t n, const char* what) {
  TRY(ensure(c, c->dsrc, n, what));
  if (n <= kFewPoints) {
    for (uint64_t i = 0; i < n; ++i)
      c->few[i] = make_double4(host[i].pos[0], host[i].pos[1], host[i].pos[2], host[i].mass);
    HIP_OK(c, hipMemcpyAsync(c->dsrc.p, c->few, n * sizeof(double4), hipMemcpyHostToDevice, c->stream));
    return BH_OK;
  }
  TRY(ensure(c, c->drec, std::min(n, kLoadPiece), what));
  for (uint64_t i = 0; i < n; i += kLoadPiece) {
    const uint64_t k = std::min(n - i, kLoadPiece);
    const uint64_t part = k > kOneCopy && k <= kTwoCopies ? (k + 1) / 2 : k;
    for (uint64_t j = 0; j < k; j += part)
      HIP_OK(c, hipMemcpyAsync(c->drec.p + j, host + i + j, std::min(k - j, part) * sizeof(bh_particle),
                               hipMemcpyHostToDevice, c->stream));
    HIP_OK(c, launch_points(c->drec.p, static_cast<uint32_t>(k), c->dsrc.p + i, c->stream));
  }
  return BH_OK;
}

void drop_side_streams(Ctx* c) {
  for (int h = 0; h < 2; ++h) {
    if (c->landed[h]) (void)hipEventDestroy(c->landed[h]);
    if (c->picked[h]) (void)hipEventDestroy(c->picked[h]);
    if (c->side[h]) (void)hipStreamDestroy(c->side[h]);
    c->landed[h] = c->picked[h] = nullptr;
    c->side[h] = nullptr;
  }
}

// False when the streams and events cannot be had.
bool side_streams(Ctx* c) {
  if (c->side[0]) return true;
  bool ok = true;
  for (int h = 0; h < 2 && ok; ++h) ok = hipStreamCreateWithFlags(&c->side[h], hipStreamNonBlocking) == hipSuccess;
  for (int h = 0; h < 2 && ok; ++h)
    ok = hipEventCreateWithFlags(&c->landed[h], hipEventDisableTiming) == hipSuccess &&
         hipEventCreateWithFlags(&c->picked[h], hipEventDisableTiming) == hipSuccess;
  if (!ok) {
    (void)hipGetLastError();
    drop_side_streams(c);
  }
  return ok;
}

// A direct sum over few targets and many sources takes as long to get the
// records over the host link as to sum them, so it sums each piece of the
// sources while the next one is copied: the pieces go through the two halves
// of drec, and the targets (xt, picked on the host: there are few) go first.
// Call in ms, all sources first -> in pieces:
//   targets of sources    2^18          pieces of 2^17, 2^19
//   4,096 of 1M           5.7 -> 3.55   3.4, 4.6
//   8,192 of 1M           8.9 -> 6.6    6.3, 7.8
//   1,000 of 1M           3.2 -> 2.75   2.95, 3.15
//   64 of 1M              2.65 -> 2.6   2.85, 2.75
//   1,000 of 600,000      1.82 -> 1.6   1.69, 1.8
//   4,096 of 4M           22.8 -> 12.1  12.0, 12.9
// Picking more than n / 128 targets on the host would take as long as it saves
// (a target's record is a cache miss, a source's copy 1.7 ns); with fewer than
// two pieces there is nothing to overlap.
constexpr uint64_t kDirectPiece = 1u << 18;

bool direct_in_pieces(const uint32_t* idx, uint64_t n, uint64_t m) {
  return idx && n >= 2 * kDirectPiece && m <= n / 128;
}

int enqueue_direct_pieces(Ctx* c, const bh_particle* host, uint64_t n, const double4* xt, uint64_t m, double eps2,
                          uint32_t splits) {
  const hipStream_t run = c->side[0], copy = c->side[1];
  TRY(ensure(c, c->dsrc, n, "direct sum"));
  TRY(ensure(c, c->dtgt, m, "direct sum"));
  TRY(ensure(c, c->drec, 2 * kDirectPiece, "direct sum"));
  HIP_OK(c, hipMemcpyAsync(c->dtgt.p, xt, m * sizeof(double4), hipMemcpyHostToDevice, run));
  for (int h = 0; h < 2; ++h) HIP_OK(c, hipEventRecord(c->picked[h], run));
  int h = 0;
  for (uint64_t i = 0; i < n; i += kDirectPiece, h ^= 1) {
    const uint64_t k = std::min(n - i, kDirectPiece);
    bh_particle* rec = c->drec.p + h * kDirectPiece;
    HIP_OK(c, hipStreamWaitEvent(copy, c->picked[h], 0));
    HIP_OK(c, hipMemcpyAsync(rec, host + i, k * sizeof(bh_particle), hipMemcpyHostToDevice, copy));
    HIP_OK(c, hipEventRecord(c->landed[h], copy));
    HIP_OK(c, hipStreamWaitEvent(run, c->landed[h], 0));
    HIP_OK(c, launch_points(rec, static_cast<uint32_t>(k), c->dsrc.p + i, run));
    HIP_OK(c, hipEventRecord(c->picked[h], run));
    HIP_OK(c, launch_direct(c->dsrc.p, static_cast<uint32_t>(i), static_cast<uint32_t>(i + k), c->dtgt.p, c->didx.p,
                            static_cast<uint32_t>(m), eps2, c->dpart.p, splits, i > 0, run));
  }
  return BH_OK;
}

int enqueue_potential(Ctx* c, const bh_particle* host, uint64_t n, uint32_t blocks, uint32_t splits) {
  HIP_OK(c, hipSetDevice(c->device));
  TRY(ensure(c, c->dpart, uint64_t(blocks) * splits, "energies"));
  TRY(load_points(c, host, n, "energies"));
  HIP_OK(c, launch_potential(c->dsrc.p, static_cast<uint32_t>(n), c->dpart.p, splits, c->stream));
  return BH_OK;
}

}  // namespace

extern "C" {

uint64_t bh_max_particles(void) { return kMaxN; }

int bh_ctx_create(bh_ctx** out, int device) {
  if (!out) return BH_ERR_INVALID;
  *out = nullptr;
  Ctx* c = new Ctx();
  c->device = device;
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || device < 0 || device >= ndev || device >= kMaxDevices) {
    (void)hipGetLastError();
    delete c;
    return BH_ERR_HIP;
  }
  // pinned staging sized so that a one-system table of the allocation-free
  // step never has to grow
  const size_t table0 = 64 << 10;
  int khz = 0;
  if (hipSetDevice(device) != hipSuccess || hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking) != hipSuccess ||
      hipHostMalloc(reinterpret_cast<void**>(&c->host_misc), kReportWords * sizeof(uint32_t), hipHostMallocDefault) !=
          hipSuccess ||
      hipHostMalloc(reinterpret_cast<void**>(&c->host_tables), table0, hipHostMallocDefault) != hipSuccess ||
      scratch_address(device, &c->arena) != hipSuccess ||
      hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, device) != hipSuccess || khz <= 0) {
    (void)hipGetLastError();
    if (c->host_tables) (void)hipHostFree(c->host_tables);
    if (c->host_misc) (void)hipHostFree(c->host_misc);
    if (c->stream) (void)hipStreamDestroy(c->stream);
    delete c;
    return BH_ERR_HIP;
  }
  c->host_tables_cap = table0;
  c->clock_khz = khz;
  *out = reinterpret_cast<bh_ctx*>(c);
  return BH_OK;
}

void bh_ctx_destroy(bh_ctx* h) {
  Ctx* c = as(h);
  if (!c) return;
  (void)hipSetDevice(c->device);
  if (c->stream) (void)hipStreamSynchronize(c->stream);
  drop_graphs(c);
  release(c->pa);
  release(c->carry);
  release(c->carry_flag);
  release(c->pb);
  release(c->tmp_in);
  release(c->tmp_out);
  release(c->keys_a);
  release(c->keys_b);
  release(c->vals_a);
  release(c->vals_b);
  release(c->hist);
  release(c->lookback);
  release(c->lohi);
  release(c->partial);
  release(c->misc);
  release(c->posm);
  release(c->L);
  release(c->H);
  release(c->tcounts);
  release(c->tprefix);
  release(c->mark);
  release(c->gmark);
  release(c->units);
  release(c->unit_lb);
  release(c->unit_n);
  release(c->defer);
  release(c->deep_frames);
  release(c->gacc);
  release(c->nbox);
  release(c->begin);
  release(c->count);
  release(c->cs);
  release(c->first_child);
  release(c->parent);
  release(c->leaf_idx);
  release(c->leaf_node);
  release(c->leaf_first);
  release(c->level_off);
  release(c->depth);
  release(c->leaf);
  release(c->nchild);
  release(c->ctr);
  release(c->rec);
  release(c->mass);
  release(c->com);
  release(c->iab);
  release(c->q64);
  release(c->tables);
  release(c->sid);
  release(c->drec);
  release(c->dsrc);
  release(c->dtgt);
  release(c->didx);
  release(c->dcnt);
  release(c->dpart);
  release(c->dacc);
  drop_side_streams(c);
  if (c->host_tables) (void)hipHostFree(c->host_tables);
  if (c->host_misc) (void)hipHostFree(c->host_misc);
  if (c->stream) (void)hipStreamDestroy(c->stream);
  delete c;
}

const char* bh_last_error(const bh_ctx* h) {
  const Ctx* c = reinterpret_cast<const Ctx*>(h);
  return c ? c->err.c_str() : "null context";
}

int bh_set_precision(bh_ctx* h, int precision) {
  Ctx* c = as(h);
  if (!c) return BH_ERR_INVALID;
  if (precision != BH_FP32 && precision != BH_FP64) {
    set_err(c, "unknown precision %d", precision);
    return BH_ERR_INVALID;
  }
  c->precision = precision;
  return BH_OK;
}

int bh_set_walk_mode(bh_ctx* h, int mode) {
  Ctx* c = as(h);
  if (!c) return BH_ERR_INVALID;
  if (mode != BH_WALK_GROUPED && mode != BH_WALK_PER_TARGET) {
    set_err(c, "unknown walk mode %d", mode);
    return BH_ERR_INVALID;
  }
  c->walk_mode = mode;
  return BH_OK;
}

int bh_set_graph_mode(bh_ctx* h, int mode) {
  Ctx* c = as(h);
  if (!c) return BH_ERR_INVALID;
  if (mode != BH_GRAPH_OFF && mode != BH_GRAPH_ON) {
    set_err(c, "unknown graph mode %d", mode);
    return BH_ERR_INVALID;
  }
  if (mode == BH_GRAPH_OFF) {
    (void)hipSetDevice(c->device);
    drop_graphs(c);
  }
  c->graph_mode = mode;
  return BH_OK;
}

int bh_set_walk_tile(bh_ctx* h, uint32_t tile) {
  Ctx* c = as(h);
  if (!c) return BH_ERR_INVALID;
  if (tile < kMinTile || tile > kGroupCap) {
    set_err(c, "walk tile %u outside %u..%u", tile, kMinTile, kGroupCap);
    return BH_ERR_INVALID;
  }
  c->walk_tile = tile;
  return BH_OK;
}

int bh_debug_walk_stack_limit(bh_ctx* h, uint32_t levels) {
  Ctx* c = as(h);
  if (!c) return BH_ERR_INVALID;
  if (levels == 0 || levels > static_cast<uint32_t>(kLevels)) {
    set_err(c, "walk stack limit %u outside 1..%d", levels, kLevels);
    return BH_ERR_INVALID;
  }
  drop_graphs(c);  // the limit is a launch argument
  c->stack_limit = levels;
  return BH_OK;
}

int bh_graph_count(bh_ctx* h, uint32_t* count) {
  Ctx* c = as(h);
  if (!c || !count) return BH_ERR_INVALID;
  *count = static_cast<uint32_t>(c->graphs.size());
  return BH_OK;
}

int bh_step_device(bh_ctx* h, const bh_particle* d_in, bh_particle* d_out, uint64_t n, const bh_force_params* fp,
                   uint32_t max_leaf, uint32_t group_size, uint32_t target_size, double kick_dt, double drift_dt,
                   bh_step_timing* timing) {
  Ctx* c = as(h);
  if (!c || !fp || (n && (!d_in || !d_out))) return c ? (set_err(c, "null argument"), BH_ERR_INVALID) : BH_ERR_INVALID;
  if (overlap(d_in, d_out, n)) {
    set_err(c, "d_in and d_out overlap");
    return BH_ERR_INVALID;
  }
  return step_device(c, d_in, d_out, n, fp, max_leaf, group_size, target_size, kick_dt, drift_dt, timing);
}

int bh_step_device_noalloc(bh_ctx* h, const bh_particle* d_in, bh_particle* d_out, uint64_t n, const bh_force_params* fp,
                           uint32_t max_leaf, uint32_t group_size, uint32_t target_size, double kick_dt,
                           double drift_dt, bh_step_timing* timing) {
  Ctx* c = as(h);
  if (!c || !fp || (n && (!d_in || !d_out))) return c ? (set_err(c, "null argument"), BH_ERR_INVALID) : BH_ERR_INVALID;
  if (timing) *timing = bh_step_timing{0.0, 0.0, 0.0};
  if (n > BH_NOALLOC_MAX_N) {
    set_err(c, "n = %llu exceeds the allocation-free step's limit of %u particles", (unsigned long long)n,
            BH_NOALLOC_MAX_N);
    return BH_ERR_TOO_LARGE;
  }
  if (overlap(d_in, d_out, n)) {
    set_err(c, "d_in and d_out overlap");
    return BH_ERR_INVALID;
  }
  TRY(check_args(c, n, fp, max_leaf, group_size));
  if (n == 0) return BH_OK;
  HIP_OK(c, hipSetDevice(c->device));
  const HostSys one{n, *fp, max_leaf, group_size, target_size, kick_dt, drift_dt, 0};
  Plan p;
  TRY(plan_systems(c, &one, 1, true, &p));
  // every level and the deep stack are planned from the start: the only
  // thing that can outgrow the fixed scratch is the node count
  p.walk = true;
  p.depth_plan = kDepthCap;
  p.deep = true;
  p.slots = walk_slots(p.n, kNoAllocSlots);
  Scratch b;
  if (!carve(static_cast<uint8_t*>(c->arena), kNoAllocBytes, &p, &b)) {
    set_err(c, "n = %llu does not fit the allocation-free step's %zu-byte scratch", (unsigned long long)n, kNoAllocBytes);
    return BH_ERR_TOO_LARGE;
  }
  // the tree lives in the shared scratch: it is not this context's to export
  c->has_tree = false;
  c->have_stats = false;
  c->reruns = 0;
  Sorted sd;
  TRY(enqueue_build(c, p, b, d_in, d_out, &sd, true));
  TRY(enqueue_walk(c, p, b, d_out, nullptr, nullptr, nullptr, d_in, sd.perm));
  TRY(enqueue_report(c, b));
  TRY(finish(c));
  const uint32_t* m = c->host_misc;
  if (m[kMiscNonfinite]) {
    set_err(c, "non-finite position, velocity or mass in the input");
    return BH_ERR_NONFINITE;
  }
  if (m[kMiscAbort]) {
    uint64_t nodes = 0;
    for (int d = 0; d < kLevels; ++d) nodes += m[kMiscLevels + d];
    set_err(c, "the tree needs %llu nodes and %u leaves; the allocation-free scratch holds %u",
            (unsigned long long)nodes, m[kMiscLevels + kLevels], p.cap_nodes);
    return BH_ERR_TOO_LARGE;
  }
  c->n_targets = m[kMiscTargets];
  c->n_groups = m[kMiscGroups];
  std::memcpy(c->last_totals, m + kMiscWords, sizeof c->last_totals);
  uint64_t nodes = 0;
  for (int d = 0; d < kLevels; ++d) nodes += m[kMiscLevels + d];
  c->n_nodes = static_cast<uint32_t>(nodes);
  c->n_leaves = m[kMiscLevels + kLevels];
  c->have_stats = true;
  c->last_graph = false;
  if (timing) {
    timing->tree_build_ms = phase_ms(c, kStampStart, kStampTargets);
    timing->traversal_ms = phase_ms(c, kStampTargets, kStampEnd);
  }
  if (m[kMiscIncomplete]) {
    set_err(c, "incomplete tree: the walk met an interior node it could not open");
    return BH_ERR_INCOMPLETE;
  }
  return BH_OK;
}

int bh_step(bh_ctx* h, bh_particle* particles, uint64_t n, const bh_force_params* fp, uint32_t max_leaf,
            uint32_t group_size, uint32_t target_size, double kick_dt, double drift_dt, bh_step_timing* timing) {
  Ctx* c = as(h);
  if (!c || !fp || (n && !particles)) return c ? (set_err(c, "null argument"), BH_ERR_INVALID) : BH_ERR_INVALID;
  TRY(check_args(c, n, fp, max_leaf, group_size));
  if (n == 0) {
    if (timing) *timing = bh_step_timing{0.0, 0.0, 0.0};
    return BH_OK;
  }
  HIP_OK(c, hipSetDevice(c->device));
  TRY(ensure(c, c->tmp_in, n, "particles"));
  TRY(ensure(c, c->tmp_out, n, "particles"));
  HIP_OK(c, hipMemcpyAsync(c->tmp_in.p, particles, n * sizeof(bh_particle), hipMemcpyHostToDevice, c->stream));
  TRY(step_device(c, c->tmp_in.p, c->tmp_out.p, n, fp, max_leaf, group_size, target_size, kick_dt, drift_dt, timing));
  HIP_OK(c, hipMemcpyAsync(particles, c->tmp_out.p, n * sizeof(bh_particle), hipMemcpyDeviceToHost, c->stream));
  HIP_OK(c, hipStreamSynchronize(c->stream));
  return BH_OK;
}

int bh_step_batch(bh_ctx* h, const bh_particle* d_in, bh_particle* d_out, const bh_system* systems, uint32_t n_systems,
                  bh_step_timing* timing) {
  Ctx* c = as(h);
  if (!c || !systems || !d_in || !d_out) return c ? (set_err(c, "null argument"), BH_ERR_INVALID) : BH_ERR_INVALID;
  const std::vector<HostSys> v = host_systems(systems, n_systems);
  uint64_t n = 0;
  for (const auto& q : v) n += q.n;
  if (overlap(d_in, d_out, n)) {
    set_err(c, "d_in and d_out overlap");
    return BH_ERR_INVALID;
  }
  return step_batch(c, d_in, d_out, v.data(), n_systems, timing);
}

int bh_step_batch_host(bh_ctx* h, bh_particle* particles, const bh_system* systems, uint32_t n_systems,
                       bh_step_timing* timing) {
  Ctx* c = as(h);
  if (!c || !systems || !particles) return c ? (set_err(c, "null argument"), BH_ERR_INVALID) : BH_ERR_INVALID;
  const std::vector<HostSys> v = host_systems(systems, n_systems);
  uint64_t n = 0;
  for (const auto& q : v) n += q.n;
  if (n > kMaxN) {
    set_err(c, "batch of %llu particles exceeds the supported %llu", (unsigned long long)n, (unsigned long long)kMaxN);
    return BH_ERR_TOO_LARGE;
  }
  HIP_OK(c, hipSetDevice(c->device));
  TRY(ensure(c, c->tmp_in, n, "particles"));
  TRY(ensure(c, c->tmp_out, n, "particles"));
  if (n) HIP_OK(c, hipMemcpyAsync(c->tmp_in.p, particles, n * sizeof(bh_particle), hipMemcpyHostToDevice, c->stream));
  TRY(step_batch(c, c->tmp_in.p, c->tmp_out.p, v.data(), n_systems, timing));
  if (n) HIP_OK(c, hipMemcpyAsync(particles, c->tmp_out.p, n * sizeof(bh_particle), hipMemcpyDeviceToHost, c->stream));
  HIP_OK(c, hipStreamSynchronize(c->stream));
  return BH_OK;
}

int bh_state_upload(bh_ctx* h, const bh_particle* host, uint64_t n) {
  Ctx* c = as(h);
  if (!c || (n && !host)) return BH_ERR_INVALID;
  if (n > kMaxN) {
    set_err(c, "n = %llu exceeds the supported %llu particles", (unsigned long long)n, (unsigned long long)kMaxN);
    return BH_ERR_TOO_LARGE;
  }
  HIP_OK(c, hipSetDevice(c->device));
  TRY(ensure(c, c->pa, n, "particles"));
  TRY(ensure(c, c->pb, n, "particles"));
  c->carried_ok = false;
  if (n) HIP_OK(c, hipMemcpyAsync(c->pa.p, host, n * sizeof(bh_particle), hipMemcpyHostToDevice, c->stream));
  HIP_OK(c, hipStreamSynchronize(c->stream));
  c->cur = 0;
  c->state_n = n;
  return BH_OK;
}

int bh_state_step(bh_ctx* h, const bh_force_params* fp, uint32_t max_leaf, uint32_t group_size, uint32_t target_size,
                  double kick_dt, double drift_dt, bh_step_timing* timing) {
  Ctx* c = as(h);
  if (!c || !fp) return BH_ERR_INVALID;
  if (c->state_n == 0) {
    set_err(c, "no resident state: upload particles with bh_state_upload first");
    return BH_ERR_INVALID;
  }
  bh_particle* in = c->cur == 0 ? c->pa.p : c->pb.p;
  bh_particle* out = c->cur == 0 ? c->pb.p : c->pa.p;
  TRY(step_device(c, in, out, c->state_n, fp, max_leaf, group_size, target_size, kick_dt, drift_dt, timing, true));
  c->cur ^= 1;
  return BH_OK;
}

int bh_state_step_batch(bh_ctx* h, const bh_system* systems, uint32_t n_systems, bh_step_timing* timing) {
  Ctx* c = as(h);
  if (!c || !systems) return c ? (set_err(c, "null argument"), BH_ERR_INVALID) : BH_ERR_INVALID;
  if (c->state_n == 0) {
    set_err(c, "no resident state: upload particles with bh_state_upload first");
    return BH_ERR_INVALID;
  }
  const std::vector<HostSys> v = host_systems(systems, n_systems);
  uint64_t n = 0;
  for (const auto& q : v) n += q.n;
  if (n != c->state_n) {
    set_err(c, "the systems hold %llu particles, the resident state %llu", (unsigned long long)n,
            (unsigned long long)c->state_n);
    return BH_ERR_INVALID;
  }
  bh_particle* in = c->cur == 0 ? c->pa.p : c->pb.p;
  bh_particle* out = c->cur == 0 ? c->pb.p : c->pa.p;
  TRY(step_batch(c, in, out, v.data(), n_systems, timing, true));
  c->cur ^= 1;
  return BH_OK;
}

bh_particle* bh_state_device_ptr(bh_ctx* h) {
  Ctx* c = as(h);
  if (!c) return nullptr;
  // the caller may write the state: the next step reads it afresh
  c->carried_ok = false;
  return c->cur == 0 ? c->pa.p : c->pb.p;
}

int bh_state_download(bh_ctx* h, bh_particle* host, uint64_t n) {
  Ctx* c = as(h);
  if (!c || (n && !host)) return BH_ERR_INVALID;
  if (n != c->state_n) {
    set_err(c, "resident state holds %llu particles, %llu requested", (unsigned long long)c->state_n,
            (unsigned long long)n);
    return BH_ERR_INVALID;
  }
  HIP_OK(c, hipSetDevice(c->device));
  if (n)
    HIP_OK(c, hipMemcpyAsync(host, bh_state_device_ptr(h), n * sizeof(bh_particle), hipMemcpyDeviceToHost, c->stream));
  HIP_OK(c, hipStreamSynchronize(c->stream));
  return BH_OK;
}

int bh_build_tree(bh_ctx* h, const bh_particle* host, uint64_t n, uint32_t max_leaf, uint32_t group_size) {
  Ctx* c = as(h);
  if (!c || (n && !host)) return BH_ERR_INVALID;
  TRY(check_args(c, n, nullptr, max_leaf, group_size));
  c->has_tree = false;
  if (n == 0) {
    set_err(c, "empty input");
    return BH_ERR_INVALID;
  }
  HIP_OK(c, hipSetDevice(c->device));
  TRY(ensure(c, c->tmp_in, n, "particles"));
  TRY(ensure(c, c->tmp_out, n, "particles"));
  HIP_OK(c, hipMemcpyAsync(c->tmp_in.p, host, n * sizeof(bh_particle), hipMemcpyHostToDevice, c->stream));
  const bh_force_params dflt{0.5, 0.0, 1.0, 1, 0};
  const HostSys one{n, dflt, max_leaf, group_size, group_size, 0.0, 0.0, 0};
  Plan p;
  TRY(plan_systems(c, &one, 1, false, &p));
  return run(c, p, c->tmp_in.p, c->tmp_out.p, false, nullptr);
}

int bh_tree_sizes(bh_ctx* h, uint64_t* n_nodes, uint64_t* n_groups, double* dom4) {
  Ctx* c = as(h);
  if (!c) return BH_ERR_INVALID;
  if (!c->has_tree) {
    set_err(c, "no tree built");
    return BH_ERR_NO_TREE;
  }
  HIP_OK(c, hipSetDevice(c->device));
  const TreeDev& t = c->sc.t;
  if (n_nodes) *n_nodes = c->n_nodes;
  if (n_groups) {
    const uint32_t m = c->n_nodes;
    std::vector<uint32_t> count(m), parent(m);
    std::vector<uint8_t> leaf(m);
    HIP_OK(c, hipMemcpy(count.data(), t.count, m * 4ull, hipMemcpyDeviceToHost));
    HIP_OK(c, hipMemcpy(parent.data(), t.parent, m * 4ull, hipMemcpyDeviceToHost));
    HIP_OK(c, hipMemcpy(leaf.data(), t.leaf, m, hipMemcpyDeviceToHost));
    uint64_t g = 0;
    for (uint32_t u = 0; u < m; ++u) {
      const uint32_t pc = u == 0 ? std::numeric_limits<uint32_t>::max() : count[parent[u]];
      if ((leaf[u] || count[u] <= c->group_size) && pc > c->group_size) ++g;
    }
    *n_groups = g;
  }
  if (dom4) {
    double4 r;
    HIP_OK(c, hipMemcpy(&r, t.ctr, sizeof(double4), hipMemcpyDeviceToHost));
    dom4[0] = r.x;
    dom4[1] = r.y;
    dom4[2] = r.z;
    dom4[3] = r.w;
  }
  return BH_OK;
}

int bh_tree_export(bh_ctx* h, int layout, uint64_t* keys, uint32_t* perm, bh_particle* sorted, bh_walk_node* nodes,
                   double* center, double* iab, uint32_t* groups) {
  Ctx* c = as(h);
  if (!c) return BH_ERR_INVALID;
  if (!c->has_tree) {
    set_err(c, "no tree built");
    return BH_ERR_NO_TREE;
  }
  if (layout != BH_LAYOUT_REFERENCE && layout != BH_LAYOUT_BFS) {
    set_err(c, "unknown layout %d", layout);
    return BH_ERR_INVALID;
  }
  if (c->plan.S != 1) {
    set_err(c, "tree export covers single-system trees");
    return BH_ERR_INVALID;
  }
  HIP_OK(c, hipSetDevice(c->device));
  HIP_OK(c, hipStreamSynchronize(c->stream));
  const TreeDev& t = c->sc.t;
  const uint32_t n = c->n, m = c->n_nodes;
  if (keys) HIP_OK(c, hipMemcpy(keys, c->keys_sorted, uint64_t(n) * 8, hipMemcpyDeviceToHost));
  if (perm) HIP_OK(c, hipMemcpy(perm, c->perm_sorted, uint64_t(n) * 4, hipMemcpyDeviceToHost));
  if (sorted) HIP_OK(c, hipMemcpy(sorted, c->sorted, uint64_t(n) * sizeof(bh_particle), hipMemcpyDeviceToHost));
  std::vector<uint32_t> begin(m), count(m), first_child(m), parent(m);
  std::vector<uint8_t> depth(m), leaf(m), nchild(m);
  std::vector<double4> ctr(m);
  std::vector<double> mass(m), com(3ull * m), ib(6ull * m);
  HIP_OK(c, hipMemcpy(begin.data(), t.begin, m * 4ull, hipMemcpyDeviceToHost));
  HIP_OK(c, hipMemcpy(count.data(), t.count, m * 4ull, hipMemcpyDeviceToHost));
  HIP_OK(c, hipMemcpy(first_child.data(), t.first_child, m * 4ull, hipMemcpyDeviceToHost));
  HIP_OK(c, hipMemcpy(parent.data(), t.parent, m * 4ull, hipMemcpyDeviceToHost));
  HIP_OK(c, hipMemcpy(depth.data(), t.depth, m, hipMemcpyDeviceToHost));
  HIP_OK(c, hipMemcpy(leaf.data(), t.leaf, m, hipMemcpyDeviceToHost));
  HIP_OK(c, hipMemcpy(nchild.data(), t.nchild, m, hipMemcpyDeviceToHost));
  HIP_OK(c, hipMemcpy(ctr.data(), t.ctr, m * sizeof(double4), hipMemcpyDeviceToHost));
  HIP_OK(c, hipMemcpy(mass.data(), t.mass, m * 8ull, hipMemcpyDeviceToHost));
  HIP_OK(c, hipMemcpy(com.data(), t.com, m * 24ull, hipMemcpyDeviceToHost));
  HIP_OK(c, hipMemcpy(ib.data(), t.iab, m * 48ull, hipMemcpyDeviceToHost));
  std::vector<uint32_t> ref_of, grp;
  if (layout == BH_LAYOUT_REFERENCE) {
    reference_order(count, leaf, first_child, nchild, c->group_size, ref_of, grp);
  } else {
    ref_of.resize(m);
    for (uint32_t u = 0; u < m; ++u) {
      ref_of[u] = u;
      const uint32_t pc = u == 0 ? std::numeric_limits<uint32_t>::max() : count[parent[u]];
      if ((leaf[u] || count[u] <= c->group_size) && pc > c->group_size) grp.push_back(u);
    }
  }
  for (uint32_t u = 0; u < m; ++u) {
    const uint32_t r = ref_of[u];
    if (nodes) {
      bh_walk_node w;
      std::memset(&w, 0, sizeof w);
      for (int a = 0; a < 3; ++a) w.com[a] = com[3ull * u + a];
      w.mass = mass[u];
      w.half_width = ctr[u].w;
      w.first_child = leaf[u] ? 0u : ref_of[first_child[u]];
      w.particle_begin = begin[u];
      w.particle_count = count[u];
      w.num_children = leaf[u] ? 0 : nchild[u];
      w.leaf = leaf[u];
      w.depth = depth[u];
      nodes[r] = w;
    }
    if (center) {
      center[3ull * r + 0] = ctr[u].x;
      center[3ull * r + 1] = ctr[u].y;
      center[3ull * r + 2] = ctr[u].z;
    }
    if (iab)
      for (int a = 0; a < 6; ++a) iab[6ull * r + a] = ib[6ull * u + a];
  }
  if (groups)
    for (size_t g = 0; g < grp.size(); ++g) groups[g] = ref_of[grp[g]];
  return BH_OK;
}

int bh_accel(bh_ctx* h, const bh_force_params* fp, uint32_t target_size, double* acc, uint32_t* n_pp, uint32_t* n_pc,
             uint64_t* totals) {
  Ctx* c = as(h);
  if (!c || !fp) return BH_ERR_INVALID;
  if (!c->has_tree) {
    set_err(c, "no tree built");
    return BH_ERR_NO_TREE;
  }
  TRY(check_args(c, c->n, fp, c->max_leaf, c->group_size));
  if (c->plan.S != 1) {
    set_err(c, "bh_accel covers single-system trees");
    return BH_ERR_INVALID;
  }
  HIP_OK(c, hipSetDevice(c->device));
  const uint32_t n = c->n;
  TRY(ensure(c, c->dacc, 3ull * n, "accelerations"));
  TRY(ensure(c, c->dcnt, 2ull * n, "interaction counts"));
  // the walk's buffers for the built tree (the build planned none)
  Plan p = c->plan;
  p.walk = true;
  Scratch b;
  TRY(provision(c, p, &b));
  if (b.t.begin != c->sc.t.begin || b.keys_a != c->sc.keys_a || b.misc != c->sc.misc) {
    set_err(c, "the tree's buffers moved since it was built");
    return BH_ERR_NO_TREE;
  }
  // the walk's parameters for the built tree: rewrite its system entry
  HIP_OK(c, hipStreamSynchronize(c->stream));
  SysDev* sd = reinterpret_cast<SysDev*>(c->host_tables);
  sd->theta2 = fp->theta * fp->theta;
  sd->eps2 = fp->eps2;
  sd->G = fp->G;
  sd->kick_dt = 0.0;
  sd->drift_dt = 0.0;
  sd->tsm = std::min(target_size, c->group_size);
  sd->use_quad = fp->use_quadrupole != 0;
  const Pieces pieces = walk_pieces(n, sd->tsm);
  sd->unit_piece = pieces.unit;
  sd->target_piece = pieces.target;
  p.unsoftened = static_cast<float>(fp->eps2) == 0.0f;
  HIP_OK(c, hipMemcpyAsync(b.tables, c->host_tables, sizeof(SysDev), hipMemcpyHostToDevice, c->stream));
  c->have_stats = false;
  c->reruns = 0;
  // what the build, or an earlier walk, left
  ZeroRanges z;
  z.p[0] = b.misc + kMiscIncomplete;
  z.n[0] = 1;
  z.p[1] = b.misc + kMiscTargets;
  z.n[1] = kMiscStamps - kMiscTargets;  // target and unit counts, totals
  z.p[2] = b.mark;
  z.n[2] = n;
  z.p[3] = b.gmark;
  z.n[3] = n;
  z.p[4] = b.unit_lb;
  z.n[4] = unit_list_words(n);
  z.p[5] = walk_queue(b);
  z.n[5] = kQueueWords;
  HIP_OK(c, launch_zero(z, c->stream));
  TRY(enqueue_walk(c, p, b, nullptr, c->dacc.p, c->dcnt.p, c->dcnt.p + n));
  TRY(enqueue_report(c, b));
  TRY(finish(c));
  c->stamps[kStampStart] = c->stamps[kStampTree] = c->stamps[kStampTargets];
  const uint32_t* m = c->host_misc;
  c->n_targets = m[kMiscTargets];
  c->n_groups = m[kMiscGroups];
  std::memcpy(c->last_totals, m + kMiscWords, sizeof c->last_totals);
  c->have_stats = true;
  c->last_graph = false;
  if (acc) HIP_OK(c, hipMemcpy(acc, c->dacc.p, 24ull * n, hipMemcpyDeviceToHost));
  if (n_pp) HIP_OK(c, hipMemcpy(n_pp, c->dcnt.p, 4ull * n, hipMemcpyDeviceToHost));
  if (n_pc) HIP_OK(c, hipMemcpy(n_pc, c->dcnt.p + n, 4ull * n, hipMemcpyDeviceToHost));
  if (totals) {
    totals[0] = c->last_totals[0];
    totals[1] = c->last_totals[1];
  }
  if (m[kMiscIncomplete]) {
    set_err(c, "incomplete tree: the walk met an interior node it could not open");
    return BH_ERR_INCOMPLETE;
  }
  return BH_OK;
}

int bh_last_step_stats(bh_ctx* h, bh_step_stats* st) {
  Ctx* c = as(h);
  if (!c || !st) return BH_ERR_INVALID;
  if (!c->have_stats) {
    set_err(c, "no step or walk has run on this context");
    return BH_ERR_NO_TREE;
  }
  HIP_OK(c, hipSetDevice(c->device));
  if (c->last_graph) {
    st->sort_ms = st->tree_ms = st->targets_ms = st->walk_ms = 0.0;
  } else {
    st->sort_ms = phase_ms(c, kStampStart, kStampTree);
    st->tree_ms = phase_ms(c, kStampTree, kStampTargets);
    st->targets_ms = phase_ms(c, kStampTargets, kStampWalk);
    st->walk_ms = phase_ms(c, kStampWalk, kStampEnd);
  }
  st->step_ms = phase_ms(c, kStampStart, kStampEnd);
  st->n_pp = c->last_totals[0];
  st->n_pc = c->last_totals[1];
  st->n_nodes = c->n_nodes;
  st->n_leaves = c->n_leaves;
  st->n_targets = c->n_targets;
  st->n_units = c->n_groups;
  st->graph = c->last_graph ? 1 : 0;
  st->reruns = c->reruns;
  return BH_OK;
}

int bh_direct_sum(bh_ctx* h, const bh_particle* host, uint64_t n, const uint32_t* idx, uint64_t m, double eps2, double G,
                  double* acc) {
  Ctx* c = as(h);
  if (!c || !host || !acc) return BH_ERR_INVALID;
  if (n > kMaxN || m > kMaxN) {
    set_err(c, "too many particles");
    return BH_ERR_TOO_LARGE;
  }
  if (!idx) m = n;
  if (n == 0 || m == 0) return BH_OK;
  HIP_OK(c, hipSetDevice(c->device));
  if (idx)
    for (uint64_t k = 0; k < m; ++k)
      if (idx[k] >= n) {
        set_err(c, "target index %u out of range", idx[k]);
        return BH_ERR_INVALID;
      }
  std::unique_ptr<double4[]> xt;
  if (direct_in_pieces(idx, n, m) && side_streams(c)) xt.reset(new (std::nothrow) double4[m]);
  const uint32_t splits = pair_splits((m + 255) / 256, xt ? kDirectPiece : n, 256, 64);
  const hipStream_t run = xt ? c->side[0] : c->stream;
  TRY(ensure(c, c->didx, m, "direct sum"));
  TRY(ensure(c, c->dpart, 3ull * m * splits, "direct sum"));
  TRY(ensure(c, c->dacc, 3ull * m, "direct sum"));
  if (idx) HIP_OK(c, hipMemcpyAsync(c->didx.p, idx, m * 4, hipMemcpyHostToDevice, run));
  if (xt) {
    for (uint64_t k = 0; k < m; ++k) {
      const bh_particle& r = host[idx[k]];
      xt[k] = make_double4(r.pos[0], r.pos[1], r.pos[2], r.mass);
    }
    const int rc = enqueue_direct_pieces(c, host, n, xt.get(), m, eps2, splits);
    if (rc != BH_OK) {  // nothing still reads the caller's memory or xt
      for (int h = 0; h < 2; ++h) (void)hipStreamSynchronize(c->side[h]);
      return rc;
    }
  } else {
    TRY(load_points(c, host, n, "direct sum"));
    HIP_OK(c, launch_direct(c->dsrc.p, 0, static_cast<uint32_t>(n), nullptr, idx ? c->didx.p : nullptr,
                            static_cast<uint32_t>(m), eps2, c->dpart.p, splits, false, run));
  }
  HIP_OK(c, launch_direct_reduce(c->dpart.p, static_cast<uint32_t>(m), splits, G, c->dacc.p, run));
  HIP_OK(c, hipMemcpyAsync(acc, c->dacc.p, 24 * m, hipMemcpyDeviceToHost, run));
  HIP_OK(c, hipStreamSynchronize(run));
  return BH_OK;
}

int bh_energies(bh_ctx* h, const bh_particle* host, uint64_t n, double G, double* kinetic, double* potential) {
  Ctx* c = as(h);
  if (!c || (n && !host)) return BH_ERR_INVALID;
  if (n > kMaxN) {
    set_err(c, "too many particles");
    return BH_ERR_TOO_LARGE;
  }
  const uint32_t blocks = static_cast<uint32_t>((n + 255) / 256);
  const uint32_t splits = pair_splits(std::max(blocks, 1u), n / 2, 128, 384);
  if (potential) *potential = 0.0;
  const bool pairs = potential && n >= 2;
  // the GPU sums the pairs while the host sums the kinetic energy
  const int rc = pairs ? enqueue_potential(c, host, n, blocks, splits) : BH_OK;
  if (kinetic) {
    // integrate.h:27-31, summed in particle order on the host (O(n))
    double e = 0.0;
    for (uint64_t i = 0; i < n; ++i) {
      const double v2 = host[i].vel[0] * host[i].vel[0] + host[i].vel[1] * host[i].vel[1] + host[i].vel[2] * host[i].vel[2];
      e += 0.5 * host[i].mass * v2;
    }
    *kinetic = e;
  }
  if (rc != BH_OK) return rc;
  if (!pairs) return BH_OK;
  std::vector<double> part(uint64_t(blocks) * splits);
  HIP_OK(c, hipMemcpyAsync(part.data(), c->dpart.p, part.size() * sizeof(double), hipMemcpyDeviceToHost, c->stream));
  HIP_OK(c, hipStreamSynchronize(c->stream));
  // the kernel counts every unordered pair once
  double sum = 0.0;
  for (double v : part) sum += v;
  *potential = -G * sum;
  return BH_OK;
}

}  // extern "C"
