// nb_direct.hip — O(N^2) direct-sum force pass and the FP64 integrator.
//
// Replaces the reference's tiled GLSL force shader (forceCalculationOptimized.glsl:28-76,
// dispatched by ParticleSolverGPU.cpp:31-35) and the update shader
// (updateParticles.glsl:34-58, ParticleSolverGPU.cpp:37-40).
//
// Direct-sum design (gfx950, wave64, vector ALU):
//   * Each lane owns B target bodies (i), held in VGPRs. A workgroup of K waves
//     shares one i-block of 64*B bodies and splits the source range (j) into K
//     contiguous slices, one per wave.
//   * Source bodies are read at wave-uniform addresses, so they arrive through
//     the scalar data cache into SGPRs (s_load_dwordx16 = 4 bodies) and feed the
//     VALU directly as scalar operands: no LDS staging, no barriers in the j-loop.
//   * One interaction = 3 v_sub + 3 v_fma (r^2) + v_rsq + 3 v_mul + 3 v_fma.
//     The self pair needs no branch: dx = 0 contributes exactly 0 when eps2 > 0.
//   * Compensated accumulation: plain FP32 partial sums over a chunk of
//     256 sources, folded into a (sum, error) pair with Knuth's TwoSum once
//     per chunk, so compensation costs < 1% of the ALU work. The K wave partials
//     are merged in LDS in fixed wave order and widened to FP64; G is applied in
//     FP64. Results are deterministic (no atomics, fixed order).
#include <algorithm>
#include <type_traits>

#include "nb_force_core.h"
#include "nb_internal.h"

namespace {

// The work is the pairs of i-blocks and units of 16 sources, block by block; a
// workgroup takes `share` of them, whatever blocks they belong to, and its waves cut
// each block's stretch into K slices. share = a whole block's units: the workgroup
// writes the block's forces. Otherwise it writes FP64 partial sums, without G, to
// out[p][3][n], p counting the workgroups of that block, and whoever reads them adds
// the parts in order; the block's last workgroup sets the unused ones to zero.
template <int B, int K, bool kGuard, bool kUniform, bool kShares>
__global__ __launch_bounds__(64 * K) void k_direct(const float4* __restrict__ pm, int n,
                                                   int n_pad, float eps2, double G, int share,
                                                   int parts, double* __restrict__ out) {
  __shared__ double part[K > 1 ? K : 1][3][B][64];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t units = n_pad / 16, blocks = n_pad / (64 * B);
  // the pairs of this workgroup's waves in block, len units from the given one on
  const auto sum = [&](uint32_t block, uint32_t from, uint32_t len, auto put) {
    const int ibase = block * (64 * B) + lane;
    nbcore::Targets<B> t;
    nbcore::load_targets<B>(pm, ibase, t);
    const uint32_t begin = 16 * (from + len * wave / K), end = 16 * (from + len * (wave + 1) / K);
    nbcore::accumulate<B, kGuard, kUniform>(pm, (int)begin, (int)end, eps2, t,
                                            kShares ? nbcore::even_chunk(end - begin) : nbcore::kChunk);
    nbcore::merge_waves<B, K>(part, wave, lane, t, [&](int a, int b, double f) {
      const int i = ibase + 64 * b;
      if (i < n) put((int64_t)a * n + i, f);
    });
  };
  if (!kShares) {
    sum(blockIdx.x, 0, units, [&](int64_t at, double f) { out[at] = G * f; });
    return;
  }
  const uint32_t x = blockIdx.x * (uint32_t)share;  // blocks * units fits 32 bits
  uint32_t block = x / units, from = x - block * units, left = share;
  for (;;) {
    const uint32_t len = min(left, units - from);
    const uint32_t p = blockIdx.x - block * units / (uint32_t)share;
    const bool last = from + len == units;
    sum(block, from, len, [&](int64_t at, double f) {
      out[3 * (int64_t)n * p + at] = f;
      if (last)
        for (int r = p + 1; r < parts; ++r) out[3 * (int64_t)n * r + at] = 0.0;
    });
    left -= len;
    if (left == 0 || ++block == blocks) return;
    from = 0;
    __syncthreads();  // the sums are read before the next block's replace them
  }
}

template <int B, int K>
hipError_t launch_bk(const nb_ctx* c) {
  const int64_t work = (int64_t)(c->n_pad / (64 * B)) * (c->n_pad / 16);
  const dim3 grid((unsigned)((work + c->share - 1) / c->share));
  double* out = c->parts > 1 ? c->part : c->force;
  const auto launch = [&](auto kernel, float eps2) {
    hipLaunchKernelGGL(kernel, grid, dim3(64 * K), 0, c->stream, c->pm, c->n, c->n_pad, eps2,
                       c->equal.factor, c->share, c->parts, out);
  };
  const bool shares = c->parts > 1;
  if (c->equal.on)
    shares ? launch(k_direct<B, K, false, true, true>, c->equal.eps2)
           : launch(k_direct<B, K, false, true, false>, c->equal.eps2);
  else if (c->guard)
    shares ? launch(k_direct<B, K, true, false, true>, c->cfg.eps2)
           : launch(k_direct<B, K, true, false, false>, c->cfg.eps2);
  else
    shares ? launch(k_direct<B, K, false, false, true>, c->cfg.eps2)
           : launch(k_direct<B, K, false, false, false>, c->cfg.eps2);
  return hipGetLastError();
}

// force = G * the sum of the parts, in order.
__device__ __forceinline__ double fold_parts(const double* __restrict__ part, int parts,
                                             int64_t stride, int64_t k, double G) {
  double f = part[k];
  for (int p = 1; p < parts; ++p) f += part[p * stride + k];
  return G * f;
}
// Shapes: B in {1, 2, 4}; K in {1, 2, 4}, plus K = 8 for B <= 2 and K = 16 for
// B = 1 (small systems need the extra waves; the LDS merge holds K*6*B*64 floats).
template <int B>
hipError_t launch_b(const nb_ctx* c) {
  switch (c->jsplit) {
    case 1: return launch_bk<B, 1>(c);
    case 2: return launch_bk<B, 2>(c);
    case 4: return launch_bk<B, 4>(c);
    case 8:
      if constexpr (B <= 2) return launch_bk<B, 8>(c);
      return hipErrorInvalidValue;
    case 16:
      if constexpr (B == 1) return launch_bk<B, 16>(c);
      return hipErrorInvalidValue;
    default: return hipErrorInvalidValue;
  }
}

// ---- FP64 integration -----------------------------------------------------
// Lagged kick-drift-kick (ParticleSystem.h:34-51):
//   v += a*dt/2; x += v*dt; a = F (evaluated at the pre-drift x); v += a*dt/2
// and semi-implicit Euler (updateParticles.glsl:44-55): v += F*dt; x += v*dt.
// Also refreshes the FP32 force view pm = (x, y, z, m) and flags non-finite state.
// kParts: `force` holds the direct sum's partial sums [parts][3][n].
template <bool kEuler, bool kParts>
__global__ __launch_bounds__(256) void k_integrate(int n, double dt, double* __restrict__ pos,
                                                   double* __restrict__ vel,
                                                   double* __restrict__ acc,
                                                   const double* __restrict__ force, int parts,
                                                   double G, const float* __restrict__ mass,
                                                   float scale, float4* __restrict__ pm,
                                                   int* __restrict__ flags) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const double h = dt * 0.5;
  double x[3];
  bool finite = true;
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    const int k = a * n + i;
    double v = vel[k];
    double p = pos[k];
    const double f = kParts ? fold_parts(force, parts, 3 * (int64_t)n, k, G) : force[k];
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
    finite = finite && isfinite(p) && isfinite(v);
  }
  pm[i] = make_float4((float)x[0] * scale, (float)x[1] * scale, (float)x[2] * scale, mass[i]);
  if (!finite) atomicOr(flags, 1);
}

// ---- small systems: forces and integration in one launch ------------------------
// At most kSmallBodies bodies: every workgroup holds all sources in LDS and owns
// kTargets bodies, kLanes per wave row and kPer per lane; its 1024 threads are
// (source slice, target lane), so even 4096 bodies fill 256 compute units, and a
// workgroup that has all the forces of its bodies can integrate them. The next
// positions go to pm_next (other workgroups still read pm); contexts alternate two
// views. Slices are interleaved: the lanes of a wave read 64 / kLanes neighbouring
// sources. Bound by latencies (staging, merge) and the LDS reads; fewer lanes with
// more bodies each halve the reads but lengthen the merge (2048 bodies: 8 x 1 5.9 us,
// 4 x 2 7.3, 2 x 4 10.6; 4096: 16 x 1 10.6, 8 x 2 11.7). Steps in us, k_direct and
// k_integrate against this: 256 bodies 6.9 / 4.2, 1000 9.7 / 4.7, 2048 11.0 / 5.8,
// 4096 14.5 / 10.4, 6000 22.3 / 19.7, 8192 29.7 / 24.9, where the LDS ends it.
// A slice is at most 128 terms in FP32; slices are added in FP64.
// kMode 0: forces only, to `force`; 1: KDK step; 2: Euler step (as k_integrate).
constexpr int kSmallThreads = 1024;

// The sum over the lanes l, l + kLanes, l + 2 kLanes, ... of a wave, in every one of
// them: lane swaps and rotations in registers, without the LDS round trips of a
// shuffle (steps: 256 bodies 4.8 -> 4.2 us, 1000 5.1 -> 4.7, 2048 6.0 -> 5.8).
template <int kLanes>
__device__ __forceinline__ double sum_slices(double v) {
  static_assert(kLanes == 4 || kLanes == 8 || kLanes == 16, "rows of 16 lanes");
  const auto halves = [](double x, auto exchange) {  // both halves of x moved alike, added
    const uint64_t b = (uint64_t)__double_as_longlong(x);
    const auto lo = exchange((uint32_t)b), hi = exchange((uint32_t)(b >> 32));
    return __longlong_as_double((long long)((uint64_t)hi[0] << 32 | lo[0])) +
           __longlong_as_double((long long)((uint64_t)hi[1] << 32 | lo[1]));
  };
  // swapping a register's odd rows (or upper half) with the even ones of its copy
  // leaves the two lanes' values side by side
  v = halves(v, [](uint32_t w) { return __builtin_amdgcn_permlane32_swap(w, w, false, false); });
  v = halves(v, [](uint32_t w) { return __builtin_amdgcn_permlane16_swap(w, w, false, false); });
  const auto rotate = [](double x, auto ctrl) {
    const uint64_t b = (uint64_t)__double_as_longlong(x);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)b, decltype(ctrl)::value, 0xf, 0xf, false);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(b >> 32), decltype(ctrl)::value, 0xf, 0xf, false);
    return x + __longlong_as_double((long long)((uint64_t)hi << 32 | lo));
  };
  if constexpr (kLanes <= 8) v = rotate(v, std::integral_constant<int, 0x128>{});  // row_ror:8
  if constexpr (kLanes <= 4) v = rotate(v, std::integral_constant<int, 0x124>{});  // row_ror:4
  return v;
}

template <int kLanes, int kPer, int kMaxPad, bool kGuard, int kMode>
__global__ __launch_bounds__(kSmallThreads) void k_direct_small(
    const float4* __restrict__ pm, int n, int n_pad, float eps2, double G, double dt,
    double* __restrict__ pos, double* __restrict__ vel, double* __restrict__ acc,
    double* __restrict__ force, float4* __restrict__ pm_next, int* __restrict__ flags) {
  constexpr int kTargets = kLanes * kPer, kSlices = kSmallThreads / kLanes;
  constexpr int kWaves = kSmallThreads / 64;
  __shared__ float4 src[kMaxPad];
  __shared__ double sums[kWaves][3][kTargets];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int base = blockIdx.x * kTargets;
  // thread t < 3 * kTargets finishes component t / kTargets of body base + t % kTargets
  const int comp = tid / kTargets, own = tid % kTargets, body = base + own;
  const bool finish = tid < 3 * kTargets && body < n;
  const int at = comp * n + body;
  double p = 0, v = 0, a = 0;
  for (int k = tid; k < n_pad; k += kSmallThreads) src[k] = pm[k];
  if (kMode != 0 && finish) {
    p = pos[at];
    v = vel[at];
    if (kMode == 1) a = acc[at];
  }
  __syncthreads();
  float x[kPer], y[kPer], z[kPer], fx[kPer], fy[kPer], fz[kPer];
#pragma unroll
  for (int r = 0; r < kPer; ++r) {
    const float4 q = src[base + tid % kLanes + kLanes * r];  // base + kTargets <= n_pad
    x[r] = q.x;
    y[r] = q.y;
    z[r] = q.z;
    fx[r] = fy[r] = fz[r] = 0.f;
  }
  const auto pairs = [&](auto count, int k) {  // with sources k, k + kSlices, ...
    constexpr int kCount = decltype(count)::value;
    float dx[kCount * kPer], dy[kCount * kPer], dz[kCount * kPer], r2[kCount * kPer],
        inv[kCount * kPer], w[kCount];
#pragma unroll
    for (int u = 0; u < kCount; ++u) {
      const float4 q = src[k + u * kSlices];
      w[u] = q.w;
#pragma unroll
      for (int r = 0; r < kPer; ++r) {
        const int e = u * kPer + r;
        dx[e] = q.x - x[r], dy[e] = q.y - y[r], dz[e] = q.z - z[r];
        r2[e] = fmaf(dz[e], dz[e], fmaf(dy[e], dy[e], fmaf(dx[e], dx[e], eps2)));
      }
    }
    nbcore::rsq_group(r2, inv);
#pragma unroll
    for (int u = 0; u < kCount; ++u)
#pragma unroll
      for (int r = 0; r < kPer; ++r) {
        const int e = u * kPer + r;
        float s = (w[u] * inv[e]) * (inv[e] * inv[e]);
        if (kGuard) s = r2[e] > 0.f ? s : 0.f;
        fx[r] = fmaf(dx[e], s, fx[r]);
        fy[r] = fmaf(dy[e], s, fy[r]);
        fz[r] = fmaf(dz[e], s, fz[r]);
      }
  };
  int k = tid / kLanes;
  for (; k + 3 * kSlices < n_pad; k += 4 * kSlices) pairs(std::integral_constant<int, 4>{}, k);
  for (; k < n_pad; k += kSlices) pairs(std::integral_constant<int, 1>{}, k);
#pragma unroll
  for (int r = 0; r < kPer; ++r) {
    double f[3] = {fx[r], fy[r], fz[r]};
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      f[c] = sum_slices<kLanes>(f[c]);
      if (lane < kLanes) sums[wave][c][lane + kLanes * r] = f[c];
    }
  }
  __syncthreads();
  if (!finish) return;
  double f = sums[0][comp][own];
#pragma unroll
  for (int w = 1; w < kWaves; ++w) f += sums[w][comp][own];
  f *= G;
  if (kMode == 0) {
    force[at] = f;
    return;
  }
  if (kMode == 2) {
    v = v + f * dt;
    p = p + v * dt;
  } else {
    const double h = dt * 0.5;
    v = v + a * h;
    p = p + v * dt;
    v = v + f * h;
  }
  acc[at] = f;
  vel[at] = v;
  pos[at] = p;
  reinterpret_cast<float*>(pm_next + body)[comp] = (float)p;
  if (comp == 0) pm_next[body].w = src[body].w;
  if (!(isfinite(p) && isfinite(v))) atomicOr(flags, 1);
}

template <int kMode>
hipError_t launch_small(const nb_ctx* c, float4* pm_next) {
  const auto launch = [&](auto kernel, int targets) {
    hipLaunchKernelGGL(kernel, dim3((c->n + targets - 1) / targets), dim3(kSmallThreads), 0,
                       c->stream, c->pm, c->n, c->n_pad, c->cfg.eps2, c->G, (double)c->cfg.dt, c->pos,
                       c->vel, c->acc, c->force, pm_next, c->flags);
  };
  const auto pick = [&](auto guard) {
    constexpr bool kGuard = decltype(guard)::value;
    if (c->n_pad <= 1024) launch(k_direct_small<4, 1, 1024, kGuard, kMode>, 4);
    else if (c->n_pad <= 2048) launch(k_direct_small<8, 1, 2048, kGuard, kMode>, 8);
    else if (c->n_pad <= 4096) launch(k_direct_small<16, 1, 4096, kGuard, kMode>, 16);
    else launch(k_direct_small<16, 2, 8192, kGuard, kMode>, 32);
  };
  c->guard ? pick(std::true_type{}) : pick(std::false_type{});
  return hipGetLastError();
}

__global__ __launch_bounds__(256) void k_refresh_pm(int n, int n_pad, const double* __restrict__ pos,
                                                    const float* __restrict__ mass, float scale,
                                                    float4* __restrict__ pm) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n_pad) return;
  if (i < n)
    pm[i] = make_float4((float)pos[i] * scale, (float)pos[n + i] * scale,
                        (float)pos[2 * n + i] * scale, mass[i]);
  else
    pm[i] = nbcore::far_pad();
}

__global__ __launch_bounds__(256) void k_fill_i32(int* __restrict__ p, int v, int64_t count) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < count) p[i] = v;
}

// ---- FP64 diagnostics -------------------------------------------------------
// Partial sums per block, added on the host in block order, so the result is
// deterministic: blocks 0 .. kin_blocks - 1 hold (ekin, px, py, pz) each, the
// others sum_{i < j} m_i m_j / sqrt(r_ij^2 + eps2) over their pairs.
// A unit of pairs is 64 targets (one wave) against `chunk` sources read at
// wave-uniform addresses; rows of units above the diagonal are taken two by two,
// the p-th and the p-th last, whose lengths add up to a constant, and dealt to the
// waves. Bound by the FP64 arithmetic of 1/sqrt; the half of the pairs that
// symmetry spares is not computed (one thread per body against all others, 16
// workgroups at 4096 bodies: 655 us, now 16; 65,536 bodies 9.9 -> 1.9 ms). The
// partials go straight to pinned host memory.
constexpr int kEnergyThreads = 256;
constexpr int kEnergyWaves = kEnergyThreads / 64;
constexpr int kPotBlocks = 2048;

struct EnergyUnits {
  int chunk, chunks, rows;  // sources per chunk; rows of 64 targets, chunk / 64 * chunks of them
  int64_t units;
};
inline EnergyUnits energy_units(int n) {
  EnergyUnits u;
  u.chunk = n <= 16384 ? 64 : 256;  // short chains where there are few units
  u.chunks = (int)(((int64_t)n + u.chunk - 1) / u.chunk);
  if (u.chunk == 64) u.chunks += u.chunks & 1;  // an even number of rows
  u.rows = u.chunk / 64 * u.chunks;
  u.units = (int64_t)(u.rows / 2) * (u.chunks + 1);
  return u;
}

__global__ __launch_bounds__(kEnergyThreads) void k_energy(int n, const double* __restrict__ pos,
                                                           const double* __restrict__ vel,
                                                           const float* __restrict__ mass,
                                                           double eps2, const int* __restrict__ flags,
                                                           EnergyUnits units,
                                                           double* __restrict__ part) {
  constexpr int kin_blocks = kEnergyKinBlocks;
  __shared__ double red[4][kEnergyThreads];
  const int tid = threadIdx.x;
  const bool kin = (int)blockIdx.x < kin_blocks;
  double v[4] = {0, 0, 0, 0};
  if (kin) {
    for (int64_t i = (int64_t)blockIdx.x * kEnergyThreads + tid; i < n; i += (int64_t)kin_blocks * kEnergyThreads) {
      const double m = mass[i];
      const double vx = vel[i], vy = vel[n + i], vz = vel[2 * (int64_t)n + i];
      v[0] += 0.5 * m * (vx * vx + vy * vy + vz * vz);
      v[1] += m * vx;
      v[2] += m * vy;
      v[3] += m * vz;
    }
  } else {
    const int lane = tid & 63;
    const int64_t wave = (int64_t)(blockIdx.x - kin_blocks) * kEnergyWaves + (tid >> 6);
    const int64_t waves = (int64_t)(gridDim.x - kin_blocks) * kEnergyWaves;
    const int per = units.chunk / 64, span = units.chunks + 1;
    for (int64_t u = wave; u < units.units; u += waves) {
      const int p = (int)(u / span), k = (int)(u - (int64_t)p * span), len = units.chunks - p / per;
      const int row = __builtin_amdgcn_readfirstlane(k < len ? p : units.rows - 1 - p);
      const int col = __builtin_amdgcn_readfirstlane(k < len ? p / per + k : row / per + k - len);
      if ((int64_t)row * 64 >= n) continue;
      const int64_t i = (int64_t)row * 64 + lane, ii = i < n ? i : n - 1;
      const double xi = pos[ii], yi = pos[n + ii], zi = pos[2 * (int64_t)n + ii];
      double phi[4] = {0, 0, 0, 0};
      const auto add = [&](int64_t j, int q) {  // wave-uniform j
        const double dx = pos[j] - xi, dy = pos[n + j] - yi, dz = pos[2 * (int64_t)n + j] - zi;
        const double r2 = dx * dx + dy * dy + dz * dz + eps2;
        phi[q] += j > i ? (double)mass[j] * rsqrt(r2) : 0.0;
      };
      const int64_t j0 = (int64_t)col * units.chunk;
      const int64_t j1 = j0 + units.chunk < n ? j0 + units.chunk : n;
      int64_t j = j0;
      for (; j + 4 <= j1; j += 4)
#pragma unroll
        for (int q = 0; q < 4; ++q) add(j + q, q);
      for (; j < j1; ++j) add(j, 0);
      if (i < n) v[0] += (double)mass[i] * ((phi[0] + phi[1]) + (phi[2] + phi[3]));
    }
  }
#pragma unroll
  for (int q = 0; q < 4; ++q) red[q][tid] = v[q];
  __syncthreads();
  for (int s = kEnergyThreads / 2; s > 0; s >>= 1) {
    if (tid < s)
      for (int q = 0; q < 4; ++q) red[q][tid] += red[q][tid + s];
    __syncthreads();
  }
  if (kin && tid < 4) part[4 * blockIdx.x + tid] = red[tid][0];
  if (!kin && tid == 0) part[3 * kin_blocks + blockIdx.x] = red[0][0];
  if (blockIdx.x == 0 && tid == 0) *reinterpret_cast<int*>(part + 3 * kin_blocks + gridDim.x) = *flags;
}

// FP64 direct-sum acceleration of selected bodies: the error reference for the
// FP32 solvers, computed on the device from the same FP32 (x, y, z, m) view the
// force passes read, widened to FP64. One workgroup per target; thread t adds
// the sources t, t + 256, ... in order, and the 256 partials are added in a
// fixed tree, so the result does not depend on scheduling.
__global__ __launch_bounds__(256) void k_ref_f64(const float4* __restrict__ pm, int n,
                                                 const int* __restrict__ slots, double eps2,
                                                 double G, double unscale,
                                                 double* __restrict__ acc3) {
  __shared__ double red[3][256];
  const int i = slots[blockIdx.x];
  const float4 me = pm[i];
  const double xi = me.x * unscale, yi = me.y * unscale, zi = me.z * unscale;  // exact
  double ax = 0.0, ay = 0.0, az = 0.0;
  for (int j = threadIdx.x; j < n; j += 256) {
    const float4 q = pm[j];
    const double dx = q.x * unscale - xi, dy = q.y * unscale - yi, dz = q.z * unscale - zi;
    const double r2 = dx * dx + dy * dy + dz * dz + eps2;
    const double s = j == i ? 0.0 : (double)q.w / (r2 * sqrt(r2));
    ax += s * dx;
    ay += s * dy;
    az += s * dz;
  }
  red[0][threadIdx.x] = ax;
  red[1][threadIdx.x] = ay;
  red[2][threadIdx.x] = az;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if (threadIdx.x < w)
      for (int a = 0; a < 3; ++a) red[a][threadIdx.x] += red[a][threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x < 3) acc3[3 * blockIdx.x + threadIdx.x] = G * red[threadIdx.x][0];
}

}  // namespace

hipError_t nb_launch_ref_f64(nb_ctx* c, const int* slots, int k, double* acc3) {
  if (k <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_ref_f64, dim3(k), dim3(256), 0, c->stream, c->pm, c->n, slots,
                     (double)c->cfg.eps2, c->G, 1.0 / c->equal.scale, acc3);
  return hipGetLastError();
}

hipError_t nb_launch_direct(nb_ctx* c) {
  if (c->small) return launch_small<0>(c, nullptr);
  switch (c->bpl) {
    case 1: return launch_b<1>(c);
    case 2: return launch_b<2>(c);
    case 4: return launch_b<4>(c);
    default: return hipErrorInvalidValue;
  }
}

// One step of a small system; the context's views change places.
hipError_t nb_launch_small_step(nb_ctx* c) {
  const hipError_t e = c->cfg.integrator == NB_INTEG_EULER ? launch_small<2>(c, c->pm_next)
                                                           : launch_small<1>(c, c->pm_next);
  std::swap(c->pm, c->pm_next);
  return e;
}

hipError_t nb_launch_integrate(nb_ctx* c) {
  const bool parts = c->parts > 1;
  const auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3((c->n + 255) / 256), dim3(256), 0, c->stream, c->n,
                       (double)c->cfg.dt, c->pos, c->vel, c->acc, parts ? c->part : c->force,
                       c->parts, c->equal.factor, c->mass, c->equal.scale, c->pm, c->flags);
  };
  if (c->cfg.integrator == NB_INTEG_EULER)
    parts ? launch(k_integrate<true, true>) : launch(k_integrate<true, false>);
  else
    parts ? launch(k_integrate<false, true>) : launch(k_integrate<false, false>);
  return hipGetLastError();
}

hipError_t nb_launch_refresh_pm(nb_ctx* c, float scale) {
  hipLaunchKernelGGL(k_refresh_pm, dim3(c->n_pad / 256), dim3(256), 0, c->stream, c->n, c->n_pad,
                     c->pos, c->mass, scale, c->pm);
  return hipGetLastError();
}

hipError_t nb_launch_fill_i32(int* p, int v, int64_t count, hipStream_t s) {
  if (count <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_fill_i32, dim3((unsigned)((count + 255) / 256)), dim3(256), 0, s, p, v,
                     count);
  return hipGetLastError();
}

int nb_energy_pot_blocks(int n) {
  return (int)std::min<int64_t>(kPotBlocks, (energy_units(n).units + kEnergyWaves - 1) / kEnergyWaves);
}

hipError_t nb_launch_energy(nb_ctx* c, double* part) {
  hipLaunchKernelGGL(k_energy, dim3(kEnergyKinBlocks + nb_energy_pot_blocks(c->n)),
                     dim3(kEnergyThreads), 0, c->stream, c->n, c->pos, c->vel, c->mass,
                     (double)c->cfg.eps2, c->flags, energy_units(c->n), part);
  return hipGetLastError();
}
