// nb_batch.hip — batched ensembles: many independent clusters of uneven size
// in one persistent force launch (see the nb_batch_* block of nbody.h).
//
// Layout in HBM: one body pool of `cap` bodies. A cluster occupies a contiguous
// segment [off, off + n_pad) (n_pad = n rounded up to 256, far-away padding),
// so its FP32 view pm[off..], FP64 state pos/vel/acc[k * cap + off..] and forces
// are plain slices. Per-slot parameters (offset, n, n_pad, eps2, dt, G) live in
// device arrays indexed by slot.
//
// Work decomposition:
//   force      work item = (slot, i-block of 64*B bodies), with everything the
//              kernel needs to know of its cluster; items are sorted by cluster
//              size, largest first; as many workgroups as can be resident at
//              once take one each, then more from an atomic ticket until none is
//              left (persistent kernel). The K waves of a
//              workgroup split the cluster's sources; partial sums merge in LDS
//              in wave order, so a cluster's forces do not depend on scheduling
//              or on the other clusters.
//   integrate  one 256-thread block per 256-body block of the pool, via a
//              (slot, first body) table.
// Tables and counts are device-resident, so the captured step graph stays valid
// when clusters are added or removed.
#include <algorithm>
#include <cmath>
#include <map>
#include <new>
#include <vector>

#include "nb_force_core.h"
#include "nb_internal.h"

// One work item of the force pass.
struct alignas(32) nb_batch_item {
  int head;             // slot << 6 | parts - 1 << 4 | its part << 2 | all parts << 1 | equal masses
  int ibase, off, end;  // bodies [off, end); targets from ibase on
  int shift;            // from a body's index to where its sums go
  float eps2;           // of the scaled view (nb_equal_mass)
  double G;
};

struct nb_batch {
  nb_batch_config cfg{};
  hipStream_t stream = nullptr;
  int64_t cap = 0;
  int bpl = 1, jsplit = 8;
  int cus = 256;  // compute units: the persistent grid fills every CU to its occupancy
  // device pool
  float4* pm = nullptr;
  double *pos = nullptr, *vel = nullptr, *acc = nullptr;
  double* force = nullptr;  // [3][force_cap]; past the bodies and in free segments: partial sums
  int64_t force_cap = 0;
  float* mass = nullptr;
  // device slot table
  int* c_off = nullptr;
  int* c_n = nullptr;
  double* c_dt = nullptr;
  float* c_scale = nullptr;  // of the cluster's FP32 view
  int* c_quota = nullptr;  // steps the cluster takes per nb_batch_step call (INT32_MAX: all)
  // device work tables
  nb_batch_item* items = nullptr;
  int4* blocks = nullptr;  // per 256-body block: slot, first body, n_pad << 2 | stored parts - 1,
                           // from a body's index to its sum of part 1
  // [0] items, [1] blocks, [4] step of the call, [5] the same for the integrator, then
  // the tickets
  int* counts = nullptr;
  double* red = nullptr;   // energy partials
  // host mirror
  std::vector<int> h_off, h_n, h_npad, h_quota;
  std::vector<float> h_eps2;
  std::vector<double> h_G;
  std::vector<nb_equal_mass> h_equal;
  std::vector<int> h_stored, h_shift;  // a cluster's parts stored apart, as in blocks
  nb_stage stage;
  std::vector<char> used;
  std::map<int64_t, int64_t> free_list;  // offset -> size
  int64_t used_bodies = 0;
  int64_t interactions = 0;
  bool dirty = true;  // work tables need a rebuild
  // graph, timing
  hipGraph_t graph = nullptr;
  hipGraphExec_t graph_exec = nullptr;
  bool timing = false;
  hipEvent_t ev[3] = {};
  nb_timing tim{};
};

namespace {

constexpr int kUnlimited = NB_BATCH_UNLIMITED;

// Parts that a cluster's sources are cut into, each an item of its own with partial
// sums that the integrator adds in order: a few large clusters then fill the chip
// (four of 8000 bodies were 500 items of eight waves for 1024 places), and the last
// items are short. Items keep about 4096 sources, and a cluster that fills the chip
// by itself gets no more. By the cluster's size alone, so that its sums do not depend
// on the others. Steps in us without / with parts: 16 clusters of 1000 to 16,000
// bodies 111 / 101, four of 8000 109 / 101, 24 of 256 to 16,384 203 / 197, 256 of 256
// to 8192 671 / 655, 512 of 256 to 32,768 12,152 / 12,330; 24 served jobs 9.16 / 7.34 ms.
// The sums of the parts past the first lie where the force array has no bodies: in the
// pool's free segments and, in a batch of its own, in up to kSpareBodies entries (100 MB)
// behind the pool; the parts thus cost a server's pool no memory. A cluster that finds
// no room has an item sum its parts one after the other, with the same bits. That is as
// fast where an item has eight waves or more, but not below, as its items are longer: 512
// clusters of 256 to 32,768 bodies with room for a twelfth of their parts / for nearly
// all, us: 1 x 8 11,426 / 11,411, 2 x 8 11,400 / 11,403, 1 x 4 11,886 / 11,492, 1 x 2
// 12,584 / 12,125.
constexpr int kMaxParts = 4;
constexpr int64_t kSpareBodies = 1 << 22;
int batch_parts(int npad) {
  return std::max(1, std::min({kMaxParts, (npad + 4095) / 4096, 1024 / (npad / 64)}));
}

// Ticket k of the force pass. Its workgroups are dealt to kTickets classes, which take every
// kTickets-th of the remaining items (they are in the order of their length): atomics on
// one address follow each other at about 10 ns, and 3,000 items from one were 30 us of a
// pass (500 clusters of 64 to 1024 bodies: step 74 us, now 60; 16 of 1000 to 16,000: 93,
// now 84; 64 classes the same). The tickets lie 128 bytes apart.
constexpr int kTickets = 16, kCounts = 64 + 32 * kTickets;
__device__ __forceinline__ int* ticket(int* counts, int k) { return counts + 64 + 32 * k; }

// use_quota: skip the clusters whose quota is used up in this call (steps);
// force-only passes (nb_batch_forces, nb_batch_tune) evaluate every cluster.
// A workgroup's first item is its own index, so a small ensemble takes no tickets
// (one per workgroup from one address: 100 clusters of 128 bodies took 45 us per
// step with them, 17 without), and a next ticket is taken while the
// current item is summed: an atomic's way across the chip, the item's record and
// its targets are a chain of waits.
// Nothing but this kernel and the integrator runs in a step: this one passes the
// step on in counts[5], the integrator counts it in counts[4] and resets the ticket,
// each where the other does not read.
// At most 80 scalar registers: with 96 the hardware holds seven waves per SIMD, not
// eight, and a CU one workgroup of sixteen waves instead of two (256 clusters of 256
// to 8192 bodies: 711 and 876 us at eight and sixteen waves, 675 and 666 with 80).
template <int B, int K>
__global__ __launch_bounds__(64 * K) __attribute__((amdgpu_num_sgpr(80))) void k_batch_force(
    const float4* __restrict__ pm, const int* __restrict__ c_quota, int use_quota,
    const nb_batch_item* __restrict__ items, int* __restrict__ counts, int64_t force_cap,
    double* __restrict__ force) {
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int nitems = counts[0];
  const int call_step = use_quota ? counts[4] : -1;
  __shared__ int s_item[2];  // in turn, so that one barrier per item is enough
  __shared__ double part[K > 1 ? K : 1][3][B][64];
  if (use_quota && blockIdx.x == 0 && threadIdx.x == 0) counts[5] = call_step;
  const int tickets = min((int)gridDim.x, kTickets), mine = blockIdx.x % tickets;
  int next = blockIdx.x;
  for (int turn = 0;; turn ^= 1) {
    if (threadIdx.x == 0) s_item[turn] = next;
    __syncthreads();
    const int item = __builtin_amdgcn_readfirstlane(s_item[turn]);
    if (item >= nitems) break;
    if (threadIdx.x == 0)
      next = nitems > (int)gridDim.x
                 ? (int)gridDim.x + mine + tickets * atomicAdd(ticket(counts, mine), 1)
                 : nitems;
    const nb_batch_item& it = items[item];  // wave-uniform
    if (__builtin_amdgcn_readfirstlane(c_quota[it.head >> 6]) <= call_step) continue;  // block-uniform
    const int ibase = it.ibase + lane;
    const int parts = (it.head >> 4 & 3) + 1, first = it.head >> 2 & 3;
    const int last = it.head & 2 ? parts - 1 : first;
    // of 16 sources; times a slice's number it fits 32 bits: at most 2^26 units are cut
    // into at most 16 slices, 2048 (clusters in parts) into 64
    const uint32_t units = (uint32_t)(it.end - it.off + 255) / 256 * 16;
    for (int q = first; q <= last; ++q) {
      nbcore::Targets<B> t;
      nbcore::load_targets<B>(pm, ibase, t);
      const uint32_t slices = K * parts, slice = K * q + wave;
      const int j0 = it.off + 16 * (int)(units * slice / slices);
      const int j1 = it.off + 16 * (int)(units * (slice + 1) / slices);
      if (it.head & 1)
        nbcore::accumulate<B, false, true>(pm, j0, j1, it.eps2, t);
      else if (it.eps2 >= 1e-20f)
        nbcore::accumulate<B, false, false>(pm, j0, j1, it.eps2, t);
      else
        nbcore::accumulate<B, true, false>(pm, j0, j1, it.eps2, t);
      if (q > first) __syncthreads();  // the last part's sums are read before these replace them
      nbcore::merge_waves<B, K>(part, wave, lane, t, [&](int a, int b, double sum) {
#pragma clang fp contract(off)  // parts are added rounded, as the integrator adds stored ones
        const int i = ibase + 64 * b;
        if (i >= it.end) return;
        double* at = force + a * force_cap + i + it.shift;
        const double f = it.G * sum;
        *at = q > first ? *at + f : f;
      });
    }
  }
}

__global__ void k_batch_reset(int* __restrict__ counts) {
  if (threadIdx.x < kTickets) *ticket(counts, threadIdx.x) = 0;
}

template <bool kEuler>
__global__ __launch_bounds__(256) void k_batch_integrate(
    const int4* __restrict__ blocks, int* __restrict__ counts, const int* __restrict__ c_off,
    const int* __restrict__ c_n, const double* __restrict__ c_dt, const float* __restrict__ c_scale,
    const int* __restrict__ c_quota, int64_t cap, double* __restrict__ pos, double* __restrict__ vel, double* __restrict__ acc,
    const double* __restrict__ force, int64_t force_cap, const float* __restrict__ mass, float4* __restrict__ pm) {
  // grid-stride over the pool blocks in use: the launch is sized for the
  // device, not for the pool's capacity, so an almost empty pool costs little
  const int nblocks = counts[1];
  const int step = counts[5];
  if (blockIdx.x == 0) {  // the next step's force pass
    if (threadIdx.x < kTickets) *ticket(counts, threadIdx.x) = 0;
    if (threadIdx.x == 0 && step < 0x7fffffff) counts[4] = step + 1;
  }
  for (int blk = blockIdx.x; blk < nblocks; blk += gridDim.x) {
    const int4 bl = blocks[blk];
    const int stored = (bl.z & 3) + 1, npad = bl.z >> 2;
    if (c_quota[bl.x] <= step) continue;  // quota used up in this call
    const int i = bl.y + threadIdx.x;
    if (i - c_off[bl.x] >= c_n[bl.x]) continue;  // padding stays far away
    const double dt = c_dt[bl.x];
    const double h = dt * 0.5;
    const float scale = c_scale[bl.x];
    double x[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      const int64_t k = a * cap + i;
      double v = vel[k];
      double p = pos[k];
      const double* mine = force + a * force_cap + i;
      double f = *mine;
      for (int q = 1; q < stored; ++q) f += mine[bl.w + (q - 1) * npad];
      if (kEuler) {
        v = v + f * dt;
        p = p + v * dt;
      } else {
        v = v + acc[k] * h;
        p = p + v * dt;
        v = v + f * h;
      }
      acc[k] = f;
      vel[k] = v;
      pos[k] = p;
      x[a] = p;
    }
    pm[i] = make_float4((float)x[0] * scale, (float)x[1] * scale, (float)x[2] * scale, mass[i]);
  }
}

__global__ void k_batch_admit(int slot, int off, int n, double dt, float scale,
                              int* __restrict__ c_off, int* __restrict__ c_n,
                              double* __restrict__ c_dt, float* __restrict__ c_scale,
                              int* __restrict__ c_quota) {
  if (threadIdx.x != 0) return;
  c_off[slot] = off;
  c_n[slot] = n;
  c_dt[slot] = dt;
  c_scale[slot] = scale;
  c_quota[slot] = kUnlimited;
}

// FP64 energy of one cluster: block partials of (ekin, sum_i m_i phi_i).
__global__ __launch_bounds__(256) void k_batch_energy(int off, int n, int64_t cap, double eps2,
                                                      const double* __restrict__ pos,
                                                      const double* __restrict__ vel,
                                                      const float* __restrict__ mass,
                                                      double* __restrict__ part) {
  __shared__ double red[2][256];
  const int k = blockIdx.x * 256 + threadIdx.x;
  const int kk = k < n ? k : n - 1;
  const int i = off + kk;
  const double xi = pos[i], yi = pos[cap + i], zi = pos[2 * cap + i];
  double phi = 0.0;
  for (int q = 0; q < n; ++q) {
    const int j = off + q;
    const double dx = pos[j] - xi, dy = pos[cap + j] - yi, dz = pos[2 * cap + j] - zi;
    const double r2 = dx * dx + dy * dy + dz * dz + eps2;
    phi += (q != kk) ? (double)mass[j] * rsqrt(r2) : 0.0;
  }
  const double m = mass[i];
  const double vx = vel[i], vy = vel[cap + i], vz = vel[2 * cap + i];
  red[0][threadIdx.x] = k < n ? 0.5 * m * (vx * vx + vy * vy + vz * vz) : 0.0;
  red[1][threadIdx.x] = k < n ? m * phi : 0.0;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if (threadIdx.x < s) {
      red[0][threadIdx.x] += red[0][threadIdx.x + s];
      red[1][threadIdx.x] += red[1][threadIdx.x + s];
    }
    __syncthreads();
  }
  if (threadIdx.x < 2) part[2 * blockIdx.x + threadIdx.x] = red[threadIdx.x][0];
}

template <int B, int K>
hipError_t launch_force(nb_batch* b, int use_quota) {
  // Persistent: as many blocks as can be resident at once, which depends on the
  // shape's registers and LDS (one body per lane fits 8 waves per SIMD, two
  // bodies 4).
  // (Queried per launch, for the current device: a host-side query, and steps
  // replay a captured graph, so it runs once per capture.)
  int per_cu = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_batch_force<B, K>, 64 * K, 0) !=
          hipSuccess ||
      per_cu < 1)
    per_cu = std::max(1, 16 / K);
  const int grid = b->cus * per_cu;
  hipLaunchKernelGGL((k_batch_force<B, K>), dim3(grid), dim3(64 * K), 0, b->stream, b->pm,
                     b->c_quota, use_quota, b->items, b->counts, b->force_cap, b->force);
  return hipGetLastError();
}

template <int B>
hipError_t launch_force_b(nb_batch* b, int use_quota) {
  switch (b->jsplit) {
    case 1: return launch_force<B, 1>(b, use_quota);
    case 2: return launch_force<B, 2>(b, use_quota);
    case 4: return launch_force<B, 4>(b, use_quota);
    case 8:
      if constexpr (B <= 2) return launch_force<B, 8>(b, use_quota);
      return hipErrorInvalidValue;
    case 16:
      if constexpr (B == 1) return launch_force<B, 16>(b, use_quota);
      return hipErrorInvalidValue;
    default: return hipErrorInvalidValue;
  }
}

// Every pass finds the ticket at zero: a step's integrator leaves it so, and a
// force pass without one is followed by a reset.
hipError_t enqueue_force(nb_batch* b, int use_quota = 0) {
  hipError_t e = hipErrorInvalidValue;
  switch (b->bpl) {
    case 1: e = launch_force_b<1>(b, use_quota); break;
    case 2: e = launch_force_b<2>(b, use_quota); break;
    case 4: e = launch_force_b<4>(b, use_quota); break;
    default: break;
  }
  if (e != hipSuccess || use_quota) return e;
  hipLaunchKernelGGL(k_batch_reset, dim3(1), dim3(64), 0, b->stream, b->counts);
  return hipGetLastError();
}

hipError_t enqueue_step(nb_batch* b) {
  hipError_t e = enqueue_force(b, 1);
  if (e != hipSuccess) return e;
  if (b->timing) (void)hipEventRecord(b->ev[1], b->stream);
  const unsigned nblk = (unsigned)std::min<int64_t>(b->cap / 256, (int64_t)b->cus * 64);
  if (b->cfg.integrator == NB_INTEG_EULER)
    hipLaunchKernelGGL((k_batch_integrate<true>), dim3(nblk), dim3(256), 0, b->stream, b->blocks,
                       b->counts, b->c_off, b->c_n, b->c_dt, b->c_scale, b->c_quota, b->cap, b->pos, b->vel,
                       b->acc, b->force, b->force_cap, b->mass, b->pm);
  else
    hipLaunchKernelGGL((k_batch_integrate<false>), dim3(nblk), dim3(256), 0, b->stream, b->blocks,
                       b->counts, b->c_off, b->c_n, b->c_dt, b->c_scale, b->c_quota, b->cap, b->pos, b->vel,
                       b->acc, b->force, b->force_cap, b->mass, b->pm);
  return hipGetLastError();
}

// Rebuild the work tables after clusters were added or removed.
int rebuild_tables(nb_batch* b) {
  if (!b->dirty) return NB_OK;
  std::vector<int> slots;
  for (int s = 0; s < (int)b->used.size(); ++s)
    if (b->used[s]) slots.push_back(s);
  std::stable_sort(slots.begin(), slots.end(),
                   [&](int a, int c) { return b->h_npad[a] > b->h_npad[c]; });
  // partial sums, largest clusters first, in free segments of the force array
  std::vector<std::pair<int64_t, int64_t>> room(b->free_list.begin(), b->free_list.end());
  room.push_back({b->cap, b->force_cap - b->cap});
  for (int s : slots) {
    const int npad = b->h_npad[s], parts = batch_parts(npad);
    const int64_t need = (int64_t)(parts - 1) * npad;
    b->h_stored[s] = 1;
    b->h_shift[s] = 0;
    if (parts == 1) continue;
    const auto seg = std::find_if(room.begin(), room.end(), [&](const auto& r) { return r.second >= need; });
    if (seg == room.end()) continue;
    b->h_stored[s] = parts;
    b->h_shift[s] = (int)(seg->first - b->h_off[s]);
    seg->first += need;
    seg->second -= need;
  }
  std::stable_sort(slots.begin(), slots.end(),
                   [&](int a, int c) {  // sources per item
                     return b->h_npad[a] / b->h_stored[a] > b->h_npad[c] / b->h_stored[c];
                   });
  std::vector<nb_batch_item> items;
  std::vector<int4> blocks;
  int64_t inter = 0;
  const int iblock = 64 * b->bpl;
  for (int s : slots) {
    const int npad = b->h_npad[s], off = b->h_off[s], stored = b->h_stored[s], parts = batch_parts(npad);
    for (int q = 0; q < npad / iblock; ++q)
      for (int p = 0; p < stored; ++p)
        items.push_back({s << 6 | (parts - 1) << 4 | p << 2 | (stored < parts) << 1 | (b->h_equal[s].on ? 1 : 0),
                         off + q * iblock, off, off + b->h_n[s], p > 0 ? b->h_shift[s] + (p - 1) * npad : 0,
                         b->h_equal[s].eps2, b->h_equal[s].factor});
    inter += (int64_t)b->h_n[s] * (b->h_n[s] - 1);
  }
  std::vector<int> by_off(slots);
  std::sort(by_off.begin(), by_off.end(), [&](int a, int c) { return b->h_off[a] < b->h_off[c]; });
  for (int s : by_off)
    for (int q = 0; q < b->h_npad[s]; q += 256)
      blocks.push_back(make_int4(s, b->h_off[s] + q, b->h_stored[s] > 1 ? b->h_npad[s] << 2 | (b->h_stored[s] - 1) : 0,
                                 b->h_shift[s]));
  const int counts[2] = {(int)items.size(), (int)blocks.size()};
  if (!items.empty())
    NB_HIP(hipMemcpyAsync(b->items, items.data(), items.size() * sizeof(nb_batch_item),
                          hipMemcpyHostToDevice, b->stream));
  if (!blocks.empty())
    NB_HIP(hipMemcpyAsync(b->blocks, blocks.data(), blocks.size() * sizeof(int4),
                          hipMemcpyHostToDevice, b->stream));
  NB_HIP(hipMemcpyAsync(b->counts, counts, sizeof(counts), hipMemcpyHostToDevice, b->stream));
  NB_HIP(hipStreamSynchronize(b->stream));  // the host vectors die here
  b->interactions = inter;
  b->dirty = false;
  return NB_OK;
}

void free_batch(nb_batch* b) {
  if (!b) return;
  nb_drop_graph(b->stream, b->graph_exec, b->graph);
  nb_stage_free(b->stage);
  for (auto& e : b->ev)
    if (e) (void)hipEventDestroy(e);
  void* ps[] = {b->pm,     b->pos,    b->vel,   b->acc,   b->force, b->mass,  b->c_off,
                b->c_n,    b->c_dt,   b->items, b->blocks, b->counts, b->red,  b->c_quota,
                b->c_scale};
  for (void* p : ps)
    if (p) (void)hipFree(p);
  if (b->stream) (void)hipStreamDestroy(b->stream);
  delete b;
}

int check_slot(nb_batch* b, int32_t id) {
  if (!b) return nb_fail(NB_E_ARG, "nb_batch: null batch");
  if (id < 0 || id >= (int)b->used.size() || !b->used[id])
    return nb_fail(NB_E_ARG, "nb_batch: no such cluster");
  return NB_OK;
}

}  // namespace

int nb_batch_create_with(nb_batch** out, const nb_batch_config* cfg, bool spare) {
  NB_TRY
  NB_API_SHARED;
  if (!out || !cfg) return nb_fail(NB_E_ARG, "nb_batch_create: null argument");
  *out = nullptr;
  if (cfg->max_bodies < 256 || cfg->max_bodies >= (int64_t(1) << 30))
    return nb_fail(NB_E_ARG, "nb_batch_create: max_bodies must be in [256, 2^30)");
  if (cfg->max_clusters < 1 || cfg->max_clusters > (1 << 20))
    return nb_fail(NB_E_ARG, "nb_batch_create: max_clusters must be in [1, 2^20]");
  if (cfg->integrator != NB_INTEG_KDK_LAGGED && cfg->integrator != NB_INTEG_EULER)
    return nb_fail(NB_E_ARG, "nb_batch_create: unknown integrator");
  if (cfg->bodies_per_lane != 0 && cfg->bodies_per_lane != 1 && cfg->bodies_per_lane != 2 &&
      cfg->bodies_per_lane != 4)
    return nb_fail(NB_E_ARG, "nb_batch_create: bodies_per_lane must be 0, 1, 2 or 4");
  if (cfg->j_split != 0 && cfg->j_split != 1 && cfg->j_split != 2 && cfg->j_split != 4 &&
      cfg->j_split != 8 && cfg->j_split != 16)
    return nb_fail(NB_E_ARG, "nb_batch_create: j_split must be 0, 1, 2, 4, 8 or 16");
  if (cfg->bodies_per_lane > 0 && cfg->j_split > 0 &&
      !nb_valid_shape(cfg->bodies_per_lane, cfg->j_split))
    return nb_fail(NB_E_ARG, "nb_batch_create: j_split 8 needs bodies_per_lane <= 2, 16 needs 1");
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev < 1)
    return nb_fail(NB_E_NOGPU, "nb_batch_create: no HIP device visible");
  nb_batch* b = new (std::nothrow) nb_batch();
  if (!b) return nb_fail(NB_E_OOM, "nb_batch_create: host allocation failed");
  b->cfg = *cfg;
  b->cap = (cfg->max_bodies + 255) / 256 * 256;
  // Built-in shape, measured on MI355X over whole steps: one body per lane and eight
  // waves per work item. In us, four / eight / sixteen waves: 512 clusters of 256 to
  // 32,768 bodies 12,495 / 12,193 / 12,733; 256 of 256 to 8192 733 / 675 / 666; 24 of
  // 256 to 16,384 274 / 205 / 207; 500 of 64 to 1024 91 / 76 / 74. nb_batch_tune times
  // every shape on the batch's own clusters.
  b->bpl = cfg->bodies_per_lane > 0 ? cfg->bodies_per_lane : 1;
  b->jsplit = cfg->j_split > 0 ? cfg->j_split : 8;
  int dev = 0, cus = 256;
  (void)hipGetDevice(&dev);
  (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
  b->cus = cus;
  auto fail = [&](int code, const char* m) {
    free_batch(b);
    return nb_fail(code, m);
  };
  if (hipStreamCreateWithFlags(&b->stream, hipStreamNonBlocking) != hipSuccess)
    return fail(NB_E_HIP, "nb_batch_create: hipStreamCreate failed");
  const size_t cap = b->cap, mc = cfg->max_clusters;
  auto A = [](void** p, size_t bytes) { return hipMalloc(p, bytes < 256 ? 256 : bytes); };
  b->force_cap = b->cap + (spare && b->cap > 4096 ? std::min(3 * b->cap, kSpareBodies) : 0);
  if (A((void**)&b->force, 3 * b->force_cap * sizeof(double))) {  // the spare entries may go
    (void)hipGetLastError();
    b->force_cap = b->cap;
    if (A((void**)&b->force, 3 * cap * sizeof(double)))
      return fail(NB_E_OOM, "nb_batch_create: device allocation failed");
  }
  const size_t fcap = b->force_cap;
  if (A((void**)&b->pm, cap * sizeof(float4)) || A((void**)&b->pos, 3 * cap * sizeof(double)) ||
      A((void**)&b->vel, 3 * cap * sizeof(double)) || A((void**)&b->acc, 3 * cap * sizeof(double)) ||
      A((void**)&b->mass, cap * sizeof(float)) || A((void**)&b->c_off, mc * sizeof(int)) || A((void**)&b->c_n, mc * sizeof(int)) ||
      A((void**)&b->c_dt, mc * sizeof(double)) || A((void**)&b->c_scale, mc * sizeof(float)) ||
      A((void**)&b->c_quota, mc * sizeof(int)) ||
      A((void**)&b->items, fcap / 64 * sizeof(nb_batch_item)) ||
      A((void**)&b->blocks, (cap / 256) * sizeof(int4)) || A((void**)&b->counts, kCounts * sizeof(int)) ||
      A((void**)&b->red, (2 * (cap / 256) + 16) * sizeof(double)))
    return fail(NB_E_OOM, "nb_batch_create: device allocation failed");
  if (hipMemset(b->pm, 0, cap * sizeof(float4)) != hipSuccess ||
      hipMemset(b->mass, 0, cap * sizeof(float)) != hipSuccess ||
      hipMemset(b->force, 0, 3 * fcap * sizeof(double)) != hipSuccess ||
      hipMemset(b->counts, 0, kCounts * sizeof(int)) != hipSuccess)
    return fail(NB_E_HIP, "nb_batch_create: hipMemset failed");
  for (auto& e : b->ev)
    if (hipEventCreate(&e) != hipSuccess) return fail(NB_E_HIP, "nb_batch_create: event failed");
  b->h_off.assign(mc, 0);
  b->h_n.assign(mc, 0);
  b->h_npad.assign(mc, 0);
  b->h_eps2.assign(mc, 0.f);
  b->h_G.assign(mc, 1.0);
  b->h_equal.assign(mc, nb_equal_mass{});
  b->h_stored.assign(mc, 1);
  b->h_shift.assign(mc, 0);
  b->used.assign(mc, 0);
  b->h_quota.assign(mc, kUnlimited);
  b->free_list[0] = b->cap;
  *out = b;
  return NB_OK;
  NB_CATCH("nb_batch_create")
}

extern "C" {

int nb_batch_create(nb_batch** out, const nb_batch_config* cfg) {
  return nb_batch_create_with(out, cfg, true);
}

void nb_batch_destroy(nb_batch* b) {
  NB_API_SHARED;
  if (!b) return;
  (void)hipStreamSynchronize(b->stream);
  free_batch(b);
}

int nb_batch_add(nb_batch* b, const double* pos3, const double* vel3, const double* acc3,
                 const float* mass, int64_t n, float eps2, float dt, float G, int32_t* id) {
  NB_TRY
  NB_API_SHARED;
  if (!b || !pos3 || !vel3 || !mass || !id) return nb_fail(NB_E_ARG, "nb_batch_add: null argument");
  if (n < 1) return nb_fail(NB_E_ARG, "nb_batch_add: n < 1");
  if (!(eps2 >= 0.f) || !std::isfinite(eps2) || !std::isfinite(dt))
    return nb_fail(NB_E_ARG, "nb_batch_add: bad eps2 or dt");
  const int64_t npad = (n + 255) / 256 * 256;
  int slot = -1;
  for (int s = 0; s < (int)b->used.size(); ++s)
    if (!b->used[s]) { slot = s; break; }
  if (slot < 0) return nb_fail(NB_E_BUDGET, "nb_batch_add: cluster table full");
  auto it = b->free_list.begin();
  for (; it != b->free_list.end(); ++it)
    if (it->second >= npad) break;
  if (it == b->free_list.end()) return nb_fail(NB_E_BUDGET, "nb_batch_add: body pool full");
  const int64_t off = it->first, len = it->second;
  b->free_list.erase(it);
  if (len > npad) b->free_list[off + npad] = len - npad;
  const int io = (int)off, in = (int)n, inp = (int)npad;
  nb_put_args p{};
  p.pos = pos3;
  p.vel = vel3;
  p.acc = acc3;
  p.mass = mass;
  p.n = n;
  p.n_pad = npad;
  p.stride = b->cap;
  p.dst[0] = b->pos + off;
  p.dst[1] = b->vel + off;
  p.dst[2] = b->acc + off;
  p.mass_dst = b->mass + off;
  p.pm = b->pm + off;
  const nb_equal_mass equal = nb_find_equal_mass(mass, n, eps2, G == 0.f ? 1.0 : (double)G);
  p.scale = equal.scale;
  int rc = nb_put(b->stage, b->stream, b->force, kPackD3, p);  // every force pass writes force anew
  if (rc == NB_OK) {
    hipLaunchKernelGGL(k_batch_admit, dim3(1), dim3(64), 0, b->stream, slot, io, in, (double)dt,
                       p.scale, b->c_off, b->c_n, b->c_dt, b->c_scale, b->c_quota);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) rc = nb_fail(NB_E_HIP, std::string("nb_batch_add: ") + hipGetErrorString(e));
  }
  if (rc != NB_OK) {
    // give the segment back (coalescing happens on the next remove)
    if (len > npad) b->free_list.erase(off + npad);
    b->free_list[off] = len;
    return rc;
  }
  b->used[slot] = 1;
  b->h_off[slot] = io;
  b->h_n[slot] = in;
  b->h_npad[slot] = inp;
  b->h_eps2[slot] = eps2;
  b->h_G[slot] = G == 0.f ? 1.0 : (double)G;
  b->h_equal[slot] = equal;
  b->h_quota[slot] = kUnlimited;
  b->used_bodies += npad;
  b->dirty = true;
  *id = slot;
  return NB_OK;
  NB_CATCH("nb_batch_add")
}

int nb_batch_remove(nb_batch* b, int32_t id) {
  NB_TRY
  NB_API_SHARED;
  int rc = check_slot(b, id);
  if (rc) return rc;
  int64_t off = b->h_off[id], len = b->h_npad[id];
  // zero the FP32 view so a stale body can never be read as a source (in stream
  // order: after the steps that still use it, before a later cluster's upload)
  NB_HIP(nb_launch_fill_i32(reinterpret_cast<int*>(b->pm + off), 0, 4 * len, b->stream));
  b->used[id] = 0;
  b->used_bodies -= len;
  // return the segment to the free list, coalescing neighbours
  auto nx = b->free_list.lower_bound(off);
  if (nx != b->free_list.end() && nx->first == off + len) {
    len += nx->second;
    b->free_list.erase(nx);
  }
  auto pv = b->free_list.lower_bound(off);
  if (pv != b->free_list.begin()) {
    --pv;
    if (pv->first + pv->second == off) {
      off = pv->first;
      len += pv->second;
      b->free_list.erase(pv);
    }
  }
  b->free_list[off] = len;
  b->dirty = true;
  return NB_OK;
  NB_CATCH("nb_batch_remove")
}

int nb_batch_set_quotas(nb_batch* b, const int32_t* ids, const int32_t* steps, int32_t count) {
  NB_TRY
  NB_API_SHARED;
  if (!b || count < 0 || (count > 0 && (!ids || !steps)))
    return nb_fail(NB_E_ARG, "nb_batch_set_quotas: bad argument");
  for (int32_t k = 0; k < count; ++k) {
    int rc = check_slot(b, ids[k]);
    if (rc) return rc;
    if (steps[k] < 0) return nb_fail(NB_E_ARG, "nb_batch_set_quotas: negative quota");
  }
  // the previous upload of the table may still read the host mirror
  NB_HIP(hipStreamSynchronize(b->stream));
  for (int32_t k = 0; k < count; ++k) b->h_quota[ids[k]] = steps[k];
  NB_HIP(hipMemcpyAsync(b->c_quota, b->h_quota.data(), b->h_quota.size() * sizeof(int),
                        hipMemcpyHostToDevice, b->stream));
  return NB_OK;
  NB_CATCH("nb_batch_set_quotas")
}

int nb_batch_step(nb_batch* b, int32_t nsteps) {
  NB_TRY
  NB_RANGE("nb_batch_step");
  if (!b) return nb_fail(NB_E_ARG, "nb_batch_step: null batch");
  if (nsteps < 0) return nb_fail(NB_E_ARG, "nb_batch_step: nsteps < 0");
  {
    NB_API_SHARED;  // the rebuild copies and synchronises; released before any capture
    int rc = rebuild_tables(b);
    if (rc) return rc;
  }
  if (nsteps == 0) return NB_OK;
  // the steps of this call count from 0 for the clusters' quotas
  NB_HIP(nb_launch_fill_i32(b->counts + 4, 0, 1, b->stream));
  if (b->timing) {
    NB_API_SHARED;
    for (int s = 0; s < nsteps; ++s) {
      (void)hipEventRecord(b->ev[0], b->stream);
      NB_HIP(enqueue_step(b));
      (void)hipEventRecord(b->ev[2], b->stream);
      NB_HIP(hipEventSynchronize(b->ev[2]));
      float f = 0, t = 0;
      NB_HIP(hipEventElapsedTime(&f, b->ev[0], b->ev[1]));
      NB_HIP(hipEventElapsedTime(&t, b->ev[0], b->ev[2]));
      b->tim.force_ms += f;
      b->tim.force_calls++;
      b->tim.step_ms += t;
      b->tim.step_calls++;
    }
    return NB_OK;
  }
  if (b->cfg.flags & NB_F_NO_GRAPH) {
    for (int s = 0; s < nsteps; ++s) NB_HIP(enqueue_step(b));
    return NB_OK;
  }
  if (!b->graph_exec) {
    NB_API_CAPTURE;
    NB_HIP(hipStreamBeginCapture(b->stream, hipStreamCaptureModeThreadLocal));
    hipError_t e = enqueue_step(b);
    hipGraph_t g = nullptr;
    hipError_t e2 = hipStreamEndCapture(b->stream, &g);
    if (e != hipSuccess || e2 != hipSuccess) {
      if (g) (void)hipGraphDestroy(g);
      return nb_fail(NB_E_HIP, "nb_batch_step: graph capture failed");
    }
    const hipError_t ei = hipGraphInstantiate(&b->graph_exec, g, nullptr, nullptr, 0);
    if (ei != hipSuccess) {
      (void)hipGraphDestroy(g);
      b->graph_exec = nullptr;
      return nb_fail(NB_E_HIP, std::string("nb_batch_step: graph instantiation failed: ") +
                                   hipGetErrorString(ei));
    }
    b->graph = g;
  }
  for (int s = 0; s < nsteps; ++s) NB_HIP(hipGraphLaunch(b->graph_exec, b->stream));
  return NB_OK;
  NB_CATCH("nb_batch_step")
}

int nb_batch_sync(nb_batch* b) {
  NB_TRY
  NB_API_SHARED;
  if (!b) return nb_fail(NB_E_ARG, "nb_batch_sync: null batch");
  NB_HIP(hipStreamSynchronize(b->stream));
  return NB_OK;
  NB_CATCH("nb_batch_sync")
}

static int fetch(nb_batch* b, const nb_planes& p, int32_t id, const double* const* src, double* const* dst,
                 int arrays) {
  const double* from[3];
  void* to[3];
  int count = 0;
  for (int k = 0; k < arrays; ++k)
    if (dst[k]) {
      from[count] = src[k] + b->h_off[id];
      to[count++] = dst[k];
    }
  if (count == 0) {
    NB_HIP(hipStreamSynchronize(b->stream));
    return NB_OK;
  }
  return nb_fetch(b->stage, b->stream, p, kPackD3, count, from, to, nullptr, nullptr);
}

int nb_batch_forces(nb_batch* b, int32_t id, double* force3) {
  NB_TRY
  NB_RANGE("nb_batch_forces");
  NB_API_SHARED;
  int rc = check_slot(b, id);
  if (rc) return rc;
  if (!force3) return nb_fail(NB_E_ARG, "nb_batch_forces: null output");
  rc = rebuild_tables(b);
  if (rc) return rc;
  NB_HIP(enqueue_force(b));
  nb_planes p;
  p.n = b->h_n[id];
  p.stride = b->force_cap;
  p.parts = b->h_stored[id];
  p.part_first = b->h_shift[id];
  p.part_stride = b->h_npad[id];
  const double* src = b->force;
  return fetch(b, p, id, &src, &force3, 1);
  NB_CATCH("nb_batch_forces")
}

int nb_batch_download(nb_batch* b, int32_t id, double* pos3, double* vel3, double* acc3) {
  NB_TRY
  NB_API_SHARED;
  int rc = check_slot(b, id);
  if (rc) return rc;
  nb_planes p;
  p.n = b->h_n[id];
  p.stride = b->cap;
  const double* src[3] = {b->pos, b->vel, b->acc};
  double* dst[3] = {pos3, vel3, acc3};
  return fetch(b, p, id, src, dst, 3);
  NB_CATCH("nb_batch_download")
}

int nb_batch_energy(nb_batch* b, int32_t id, double* ekin, double* epot) {
  NB_TRY
  NB_API_SHARED;
  int rc = check_slot(b, id);
  if (rc) return rc;
  const int n = b->h_n[id], off = b->h_off[id];
  const int blocks = (n + 255) / 256;
  const float eps2 = b->h_eps2[id];
  const double G = b->h_G[id];
  hipLaunchKernelGGL(k_batch_energy, dim3(blocks), dim3(256), 0, b->stream, off, n, b->cap,
                     (double)eps2, b->pos, b->vel, b->mass, b->red);
  NB_HIP(hipGetLastError());
  std::vector<double> part(2 * blocks);
  NB_HIP(hipMemcpyAsync(part.data(), b->red, part.size() * sizeof(double), hipMemcpyDeviceToHost,
                        b->stream));
  NB_HIP(hipStreamSynchronize(b->stream));
  double ek = 0, ep = 0;
  for (int q = 0; q < blocks; ++q) {
    ek += part[2 * q];
    ep += part[2 * q + 1];
  }
  if (ekin) *ekin = ek;
  if (epot) *epot = -0.5 * G * ep;
  return NB_OK;
  NB_CATCH("nb_batch_energy")
}

int nb_batch_info(nb_batch* b, int32_t* clusters, int64_t* bodies, int64_t* interactions) {
  NB_TRY
  if (!b) return nb_fail(NB_E_ARG, "nb_batch_info: null batch");
  int rc = rebuild_tables(b);
  if (rc) return rc;
  if (clusters) *clusters = (int32_t)std::count(b->used.begin(), b->used.end(), 1);
  if (bodies) *bodies = b->used_bodies;
  if (interactions) *interactions = b->interactions;
  return NB_OK;
  NB_CATCH("nb_batch_info")
}

int nb_batch_set_timing(nb_batch* b, int32_t enable) {
  NB_TRY
  NB_API_SHARED;
  if (!b) return nb_fail(NB_E_ARG, "nb_batch_set_timing: null batch");
  NB_HIP(hipStreamSynchronize(b->stream));
  b->timing = enable != 0;
  b->tim = nb_timing{};
  return NB_OK;
  NB_CATCH("nb_batch_set_timing")
}

int nb_batch_get_timing(nb_batch* b, nb_timing* out) {
  NB_TRY
  if (!b || !out) return nb_fail(NB_E_ARG, "nb_batch_get_timing: null argument");
  *out = b->tim;
  out->interactions = b->interactions;
  return NB_OK;
  NB_CATCH("nb_batch_get_timing")
}

int nb_batch_tune(nb_batch* b, int32_t reps, nb_tuning* out) {
  NB_TRY
  NB_RANGE("nb_batch_tune");
  NB_API_SHARED;
  if (!b) return nb_fail(NB_E_ARG, "nb_batch_tune: null batch");
  if (reps < 1) reps = 3;
  NB_HIP(hipStreamSynchronize(b->stream));
  const int bpl0 = b->bpl, js0 = b->jsplit;
  int best_b = bpl0, best_k = js0;
  double best_ms = -1.0;
  // The force pass leaves the state untouched (the next step recomputes the
  // forces it integrates), so every shape can be timed on the live clusters.
  for (int bb : {1, 2, 4})
    for (int k : {1, 2, 4, 8, 16}) {
      if (!nb_valid_shape(bb, k)) continue;
      b->bpl = bb;
      b->jsplit = k;
      b->dirty = true;
      int rc = rebuild_tables(b);
      if (rc) return rc;
      NB_HIP(enqueue_force(b));  // warm-up
      NB_HIP(hipEventRecord(b->ev[0], b->stream));
      for (int r = 0; r < reps; ++r) NB_HIP(enqueue_force(b));
      NB_HIP(hipEventRecord(b->ev[2], b->stream));
      NB_HIP(hipEventSynchronize(b->ev[2]));
      float ms = 0.f;
      NB_HIP(hipEventElapsedTime(&ms, b->ev[0], b->ev[2]));
      const double per = ms / reps;
      if (best_ms < 0 || per < best_ms) {
        best_ms = per;
        best_b = bb;
        best_k = k;
      }
    }
  b->bpl = best_b;
  b->jsplit = best_k;
  b->dirty = true;
  nb_drop_graph(b->stream, b->graph_exec, b->graph);
  int rc = rebuild_tables(b);
  if (rc) return rc;
  if (out) {
    *out = nb_tuning{};
    int64_t bodies = 0;
    for (size_t q = 0; q < b->used.size(); ++q)
      if (b->used[q]) bodies += b->h_n[q];
    out->n = bodies;
    out->bodies_per_lane = best_b;
    out->j_split = best_k;
    out->direct_ms = best_ms;
  }
  return NB_OK;
  NB_CATCH("nb_batch_tune")
}

}  // extern "C"
