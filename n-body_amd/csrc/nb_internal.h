// nb_internal.h — device-side state and kernel launchers shared by the
// translation units of libnbody (not installed; the public ABI is nbody.h).
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>
#include <exception>
#include <mutex>
#include <new>
#include <shared_mutex>
#include <string>
#include <vector>

#include <rocprofiler-sdk-roctx/roctx.h>

#include "nbody.h"

// ---- error plumbing -------------------------------------------------------
void nb_set_error(const std::string& msg);
int nb_fail(int code, const std::string& msg);
#define NB_HIP(call)                                                               \
  do {                                                                             \
    hipError_t e_ = (call);                                                        \
    if (e_ != hipSuccess)                                                          \
      return nb_fail(NB_E_HIP, std::string(#call) + ": " + hipGetErrorString(e_)); \
  } while (0)

// Stream capture and the runtime calls that may not overlap it. A graph
// capture (the first nb_step / nb_batch_step of a context) holds this lock
// exclusively; entry points that allocate, free, copy or synchronise hold it
// shared. Different contexts may therefore be used from different threads.
std::shared_mutex& nb_capture_mutex();
#define NB_API_SHARED std::shared_lock<std::shared_mutex> nb_api_guard_(nb_capture_mutex())
#define NB_API_CAPTURE std::unique_lock<std::shared_mutex> nb_capture_guard_(nb_capture_mutex())

// Every int-returning C entry point runs its body inside NB_TRY ... NB_CATCH so
// that no C++ exception (a failed host allocation, a thread that cannot start)
// crosses the C ABI: it becomes a status code and an nb_last_error() message.
#define NB_TRY try {
#define NB_CATCH(fn)                                                                  \
  }                                                                                   \
  catch (const std::bad_alloc&) {                                                     \
    return nb_fail(NB_E_OOM, fn ": host allocation failed");                          \
  }                                                                                   \
  catch (const std::exception& nb_ex_) {                                              \
    return nb_fail(NB_E_HIP, std::string(fn ": ") + nb_ex_.what());                   \
  }                                                                                   \
  catch (...) {                                                                       \
    return nb_fail(NB_E_HIP, fn ": unexpected exception");                            \
  }

// Host trace range over an entry point (roctx): it names the call on a
// `rocprofv3 --marker-trace` timeline and costs a few ns when no tool is attached.
struct nb_trace_range {
  explicit nb_trace_range(const char* name) { roctxRangePushA(name); }
  ~nb_trace_range() { roctxRangePop(); }
  nb_trace_range(const nb_trace_range&) = delete;
  nb_trace_range& operator=(const nb_trace_range&) = delete;
};
#define NB_RANGE(name) nb_trace_range nb_trace_range_(name)

// Padding granule of the FP32 body array: the direct kernel's i-blocks hold
// 64 lanes x up to 4 bodies, and its j-range is split over up to 4 waves in
// multiples of 4 bodies, so every count is a multiple of 256.
constexpr int kPadBodies = 256;

// Largest direct sum that holds all its sources in one workgroup's LDS.
constexpr int kSmallBodies = 8192;

// Octree geometry: 30-bit Morton codes give at most 10 levels below the root.
constexpr int kMaxLevel = 10;

// ---- Barnes-Hut buffer layout --------------------------------------------------
// Every device array of the Barnes-Hut pipeline for n bodies lives in one block:
// a context allocates it once (nb_bh_alloc), and nb_bh_forces_noalloc carves the
// same layout out of a static device array. The Morton-sort buffers come first,
// so a direct-sum context that only reorders (nb_sort_alloc) allocates the
// prefix [0, off[kBhPms]).
constexpr int kBboxBlocks = 256;                      // bbox partial blocks
constexpr int kSortTile = 2048;                       // keys per block in the radix passes
constexpr int kSortGroup = 64;                        // tiles whose digit counts are also added up
constexpr int kTreeTile = 1024;                       // bodies per block in the tree build
constexpr int kLevels = kMaxLevel + 1;                // levels a node can have
constexpr int kCostBuckets = 64;  // half-octaves of estimated record time
// Whether the Barnes-Hut build pairs sibling ranges (and the traversal orders
// its work): by size unless a flag forces it either way.
inline bool nb_bh_pairs(int64_t n, int flags) {
  if (flags & NB_F_BH_SINGLE_RANGES) return false;
  return (flags & NB_F_BH_PAIRS) || n >= NB_BH_PAIR_MIN_BODIES;
}

enum nb_bh_buf {
  kBhBbox, kBhGeom, kBhKey0, kBhKey1, kBhVal0, kBhVal1, kBhCodes, kBhHist, kBhGroupHist,
  kBhPms, kBhPrefix, kBhScanPart, kBhNode, kBhNext, kBhLevel, kBhMarks,
  kBhNodeEnd, kBhLevelCnt, kBhCounters, kBhWaves, kBhInter, kBhFlags,
  kBhRecCost, kBhRecBucket, kBhRecOrder, kBhRecHist, kBhBufCount
};

// Node bound: a level holds at most min(8^l, n) nodes and there are 11 levels.
constexpr int64_t nb_tree_bound(int64_t n) {
  int64_t total = 0, w = 1;
  for (int l = 0; l <= kMaxLevel; ++l) {
    total += w < n ? w : n;
    if (w < n) w *= 8;
  }
  return total;
}

struct nb_bh_layout {
  int64_t off[kBhBufCount + 1] = {};  // byte offsets, 256-aligned; off[kBhBufCount] = total
  int64_t sort_blocks = 0, max_nodes = 0;
};

constexpr nb_bh_layout nb_bh_layout_for(int64_t n) {
  nb_bh_layout L{};
  const int64_t sort_blocks = (n + kSortTile - 1) / kSortTile;
  const int64_t groups = (sort_blocks + kSortGroup - 1) / kSortGroup;
  const int64_t bound = nb_tree_bound(n);
  int64_t bytes[kBhBufCount] = {};
  bytes[kBhBbox] = 4 * 6 * kBboxBlocks;
  bytes[kBhGeom] = 4 * 32;
  bytes[kBhKey0] = bytes[kBhKey1] = bytes[kBhVal0] = bytes[kBhVal1] = bytes[kBhCodes] = 4 * n;
  bytes[kBhHist] = 4 * 256 * sort_blocks;
  bytes[kBhGroupHist] = 4 * 4 * 256 * groups;
  bytes[kBhPms] = 16 * n;
  bytes[kBhPrefix] = 32 * (n + 1);
  bytes[kBhScanPart] = 32 * ((n + kTreeTile - 1) / kTreeTile + 1);
  bytes[kBhNode] = 32 * bound;
  bytes[kBhNext] = 4 * bound;
  bytes[kBhLevel] = 4 * (kMaxLevel + 2);
  bytes[kBhMarks] = n;
  bytes[kBhNodeEnd] = 4 * bound;
  bytes[kBhLevelCnt] = 4 * kLevels * ((n + kTreeTile - 1) / kTreeTile);
  bytes[kBhCounters] = 4 * 16;
  bytes[kBhWaves] = 16 * n;
  bytes[kBhInter] = 8 * 2;
  bytes[kBhFlags] = 4 * 4;
  bytes[kBhRecCost] = bytes[kBhRecBucket] = bytes[kBhRecOrder] = 4 * n;
  bytes[kBhRecHist] = 4 * 2 * kCostBuckets;
  int64_t at = 0;
  for (int k = 0; k < kBhBufCount; ++k) {
    L.off[k] = at;
    at += (bytes[k] + 255) / 256 * 256;
  }
  L.off[kBhBufCount] = at;
  L.sort_blocks = sort_blocks;
  L.max_nodes = bound;
  return L;
}

// An octree node, 32 bytes: all that a walk reads of it. The eight children of a
// node are two cache lines.
struct alignas(32) nb_node {
  float4 com;  // (cx, cy, cz, m)
  float r2;    // squared opening radius (s / theta + |COM - cell centre|)^2
  int first;   // first child, -1 for a leaf
  int start;   // first sorted body
  int span;    // count << 4 | level
};

// Largest system nb_bh_forces_noalloc accepts (its static scratch is sized for it).
constexpr int64_t kNoAllocMaxBodies = NB_NOALLOC_MAX_BODIES;

// Device arrays of the Barnes-Hut pipeline (sized once at nb_create).
struct nb_bh_state {
  void* block = nullptr;        // owning allocation the arrays below are carved from (or null)
  int64_t max_nodes = 0;
  // bbox: per-block partial min/max and the final (min xyz, max xyz, side2[11])
  float* bbox_part = nullptr;   // [2 * 3 * bbox_blocks]
  float* geom = nullptr;        // [6 + 11]: bmin[3], bmax[3], side^2 per level
  int bbox_blocks = 0;
  // Morton keys and body indices, double-buffered for the radix sort
  uint32_t* keys[2] = {nullptr, nullptr};
  uint32_t* vals[2] = {nullptr, nullptr};
  uint32_t* codes = nullptr;    // unsorted codes (debug tap)
  int* digit_hist = nullptr;    // radix: [sort_blocks][256] digit counts of the current pass
  int* group_hist = nullptr;    // radix: [4][groups][256] digit counts of each pass, kSortGroup tiles
  int sort_blocks = 0;
  float4* pms = nullptr;        // bodies in sorted order (x, y, z, m)
  double4* prefix = nullptr;    // exclusive FP64 prefix of (m, m x, m y, m z), n+1 entries
  double4* scan_part = nullptr; // scan block partials
  // octree, breadth-first
  nb_node* nodes = nullptr;
  int* node_next = nullptr;     // rope: next node in pre-order after the subtree, -1 at the end
  int* level_off = nullptr;     // [kMaxLevel + 2] node index where each level begins
  unsigned char* marks = nullptr;  // per sorted body: levels at which a node starts there
  int* node_end = nullptr;      // end of each node's body range
  int* level_cnt = nullptr;     // [kLevels][tiles] node starts per tile, then their exclusive scan
  int* counters = nullptr;      // [0] wave ranges, [1] traversal ticket, [2 + l] nodes of level l
  int4* waves = nullptr;        // records of one or two sibling wave ranges (start, count, start, count)
  // traversal order: records by the device time their bodies took in the last pass
  float* rec_cost = nullptr;    // per body (original index): last pass's time of its record / its bodies
  int* rec_bucket = nullptr;    // per record: cost bucket of this pass
  int* rec_order = nullptr;     // tickets -> records, costliest buckets first
  int* rec_hist = nullptr;      // [kCostBuckets] records per bucket, then [kCostBuckets] cursors
  int persist_blocks = 0;       // traversal workgroups (persistent)
  unsigned long long* inter = nullptr;  // interaction counter (diagnostic traversal)
};

// Pinned host buffer of one context or batch: what crosses the bus in small calls,
// and large results in halves (nb_pack.hip). Used by one host thread at a time,
// on the owner's stream only.
constexpr int64_t kStageBytes = 2 << 20;
constexpr int64_t kLargeStageBytes = 16 << 20;  // from twice as many bytes in one call on
struct nb_stage {
  char* host = nullptr;
  int64_t bytes = 0;
  hipEvent_t done[2] = {};  // each half has been filled
  bool busy = false;        // an enqueued kernel still reads it
};

// Equal masses m > 0 leave the direct sum's inner loop. The coordinates of its FP32
// view are then multiplied by `scale`, a power of two (exact), at or below m^{-1/3}
// and at most 1, and the sum by m * scale^2: its terms r^-3 are then no smaller than the
// m r^-3 they stand for, so nothing underflows that did not before, and with the
// scaled eps2 at 1e-20 or more nothing overflows. Not used where eps2 is smaller
// (the guarded kernels).
struct nb_equal_mass {
  bool on = false;
  float scale = 1.f, eps2 = 0.f;  // of the view
  double factor = 1.0;            // G times the sum's factor
};
nb_equal_mass nb_find_equal_mass(const float* mass, int64_t n, float eps2, double G);

// Division of the direct sum: units of (i-block, 16 sources) per workgroup, and the
// most workgroups that any i-block is divided among.
struct nb_shares {
  int units, parts;
};

struct nb_ctx {
  nb_config cfg{};
  int64_t cap_n = 0;  // bodies the device buffers were sized for (nb_ctx_rebind limit)
  int n = 0;
  int n_pad = 0;
  int device = 0;
  hipStream_t stream = nullptr;
  float theta2 = 0.25f;
  double G = 1.0;

  // particle state, FP64 structure-of-arrays: [x(0..n), y(0..n), z(0..n)]
  double* pos = nullptr;
  double* vel = nullptr;
  double* acc = nullptr;
  double* force = nullptr;   // last force pass, [3][n]
  float* mass = nullptr;     // [n_pad], zero in the padding
  float4* pm = nullptr;      // FP32 force view (x, y, z, m), [n_pad], far-away padding
  int* flags = nullptr;      // device status word (bit 0: non-finite state)

  // direct-sum launch shape
  int bpl = 2;     // i-bodies per lane
  int jsplit = 2;  // waves per workgroup of an i-block
  bool small = false;  // direct sum of a small system: one launch per step (k_direct_small)
  float4* pm_next = nullptr;  // its second view: a step reads pm, writes pm_next and swaps them
  int share = 0;   // units of work per workgroup of the direct sum (nb_shares)
  int parts = 1;   // most workgroups that share an i-block
  double* part = nullptr;  // their partial sums [parts][3][n], behind force
  bool guard = false;
  nb_equal_mass equal;  // k_direct's form for equal masses
  int walk_stack = 0;  // BH traversal stack region cap (0: the full kStackCap); a test hook

  nb_bh_state bh;
  // Morton reordering (nb_reorder): order[slot] = the caller's index of the
  // body held in that slot; empty while slots are in the caller's order.
  std::vector<int32_t> order;
  int* slot_of = nullptr;    // its inverse on the device, allocated by the first nb_reorder
  double* tmp = nullptr;     // [3][n] permutation staging, allocated on first use
  nb_stage stage;
  bool uploaded = false;
  bool tree_valid = false;

  // captured step graph: graph_steps consecutive steps
  hipGraph_t graph = nullptr;
  hipGraphExec_t graph_exec = nullptr;
  int graph_steps = 1;
  const float4* graph_pm = nullptr;  // the view that the graph's first step reads

  // timing
  bool timing = false;
  hipEvent_t ev[8] = {};
  nb_timing tim{};
};

// Release a captured step graph. Launches of it may still be queued on `s`,
// and the executable graph owns the kernel-argument memory they read, so the
// stream is drained first.
inline void nb_drop_graph(hipStream_t s, hipGraphExec_t& exec, hipGraph_t& graph) {
  if (exec || graph) (void)hipStreamSynchronize(s);
  if (exec) (void)hipGraphExecDestroy(exec);
  if (graph) (void)hipGraphDestroy(graph);
  exec = nullptr;
  graph = nullptr;
}

// ---- host copies (nb_pack.hip) ----------------------------------------------
// Packed layouts: double[3] per body, float4 (x, y, z, 0), and the render view
// (x, y, z, |v|), which reads positions and velocities into one array.
enum nb_pack_layout { kPackD3, kPackF4, kPackView };
struct nb_planes {
  int64_t n = 0;       // bodies
  int64_t stride = 0;  // from one component's plane to the next
  const int* slot_of = nullptr;  // device: slot of each body, or null (body i in slot i)
  int parts = 1;       // > 1: values are G times the sum of part 0, in place, and the others:
  int64_t part_first = 0, part_stride = 0;  // from it to part 1, from one to the next
  double G = 1.0;
};
int nb_stage_ready(nb_stage& st, hipStream_t s, int64_t bytes);  // at least that large, and free
// Copies `arrays` device arrays to the host arrays dst, packed, and waits for
// them; *flags_out receives the device word *flags (0 if null).
int nb_fetch(nb_stage& st, hipStream_t s, const nb_planes& p, int layout, int arrays,
             const double* const* src, void* const* dst, const int* flags, int* flags_out);
struct nb_put_args {
  const void *pos, *vel, *acc;  // host, packed (kPackD3 or kPackF4); acc may be null (zero)
  const float* mass;            // host
  int64_t n, n_pad;             // pm is zero from n to n_pad
  int64_t stride;
  double* dst[3];               // device: first planes of positions, velocities, accelerations
  float* mass_dst;
  float4* pm;
  float scale;                  // of the coordinates in pm
  int* flags;                   // four words to clear, or null
};
// Copies a system to the device. The host arrays may be reused on return; the
// copy is complete in stream order. dev_tmp: 24 n bytes of device scratch.
int nb_put(nb_stage& st, hipStream_t s, void* dev_tmp, int layout, const nb_put_args& p);
void nb_stage_free(nb_stage& st);

// ---- launchers (return hipError_t of the launch) ---------------------------
hipError_t nb_launch_direct(nb_ctx* c);  // pm -> force, or part when parts > 1
hipError_t nb_launch_small_step(nb_ctx* c);  // force + integration of a `small` context
hipError_t nb_launch_integrate(nb_ctx* c);  // force or part + state -> state, pm
hipError_t nb_launch_refresh_pm(nb_ctx* c, float scale);  // pos * scale, mass -> pm
hipError_t nb_launch_fill_i32(int* p, int v, int64_t count, hipStream_t s);
// state -> part: 4 * kEnergyKinBlocks kinetic, then nb_energy_pot_blocks(n) potential
// partials, then the device status word (as an int)
constexpr int kEnergyKinBlocks = 128;
int nb_energy_pot_blocks(int n);
hipError_t nb_launch_energy(nb_ctx* c, double* part);
// FP64 direct-sum accelerations of the bodies in slots[0..k) -> acc3[3k]
hipError_t nb_launch_ref_f64(nb_ctx* c, const int* slots, int k, double* acc3);

// Barnes-Hut pipeline
int nb_sort_alloc(nb_ctx* c);  // bbox, Morton and radix-sort buffers only
int nb_bh_alloc(nb_ctx* c);    // everything, one allocation
// Point every Barnes-Hut array of c (n bodies) into `base`, laid out by
// nb_bh_layout_for(n); `upto` = kBhBufCount for all of them, kBhPms for the
// sort buffers only. Sets max_nodes, sort_blocks, bbox_blocks, persist_blocks.
void nb_bh_carve(nb_ctx* c, char* base, int upto);
hipError_t nb_morton_sort(nb_ctx* c);  // bbox, Morton codes, stable sort: perm in bh.vals[0]
// slots of pos/vel/acc/force/mass take the bodies of bh.vals[0] (staging in c->tmp)
hipError_t nb_launch_permute_state(nb_ctx* c);
void nb_bh_free(nb_ctx* c);
hipError_t nb_bh_build(nb_ctx* c);     // bbox, Morton, sort, permute, prefix, octree
hipError_t nb_bh_traverse(nb_ctx* c, bool count_interactions);  // -> force
// Per-body traversal with the default (modified) opening test, counting only:
// the interactions the group traversal's test needs body by body -> bh.inter
hipError_t nb_bh_count_per_body(nb_ctx* c);

// nb_batch_create; spare: with room for partial sums beyond the pool (see batch_parts)
int nb_batch_create_with(nb_batch** out, const nb_batch_config* cfg, bool spare);

// nb_create; tuned: zero shape fields take the autotuner's values, if there are any
int nb_create_with(nb_ctx** out, const nb_config* cfg, bool tuned);

// Launch-shape defaults: fill the zero fields from the autotuner's table, then
// from the built-in defaults.
bool nb_tuned_shape(int64_t n, int* bpl, int* jsplit, int* leaf);
void nb_default_shape(int64_t n, int* bpl, int* jsplit, int* leaf);
nb_shares nb_direct_shares(int n_pad, int bpl, int jsplit, int cus);
bool nb_valid_shape(int bpl, int jsplit);  // a direct-sum kernel exists for it

// step = forces + integration (no sync)
hipError_t nb_enqueue_step(nb_ctx* c);
// Reuse a Barnes-Hut context for another system of the same solver:
// cfg->n <= c->cap_n; the buffers are re-laid out for cfg->n, the captured step
// graph is dropped and the state must be uploaded again. Allocates nothing.
int nb_ctx_rebind(nb_ctx* c, const nb_config* cfg);
