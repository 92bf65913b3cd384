// nb_force_core.h — the direct-sum inner loop shared by the single-system
// kernel (nb_direct.hip) and the batched-ensemble kernel (nb_batch.hip).
//
// A lane owns B target bodies held in VGPRs; the sources [j0, j1) are read at
// wave-uniform addresses, so they come through the scalar cache into SGPRs and
// feed the VALU as scalar operands. One interaction is
//   3 v_sub + 3 v_fma (r^2) + v_rsq + 3 v_mul (2 for equal masses) + 3 v_fma,
// the reciprocal square roots four by four (rsq_group).
// Sums are plain FP32 within a chunk of kChunk sources and folded into a
// (sum, error) pair with Knuth's TwoSum once per chunk.
#pragma once
#include <hip/hip_runtime.h>

namespace nbcore {

constexpr int kChunk = 256;

// Chunks of equal length, in 16 sources, for a slice of len: 304 sources as 160 + 144
// lose fewer bits than as 256 + 48. Short slices are those of small systems, whose sums
// have few folds to average over: theirs are at most 128 long (uniform ball of 12,345
// bodies: error of the forces 4.8e-8, 4.05e-8 so).
__device__ __forceinline__ int even_chunk(uint32_t len) {
  const uint32_t longest = len < 2 * kChunk ? kChunk / 2 : kChunk;
  const uint32_t folds = (len + longest - 1) / longest;
  return folds > 1 ? (int)((len / 16 + folds - 1) / folds * 16) : kChunk;
}

// Coordinates of the padding of an FP32 view, and its mass: r^2 is infinite and
// 1/r zero against any body, so it adds nothing with or without its mass. (Zero mass
// alone is not enough: at a distance whose r^-2 overflows, its term is not a number.)
__host__ __device__ __forceinline__ float4 far_pad() { return make_float4(1e30f, 1e30f, 1e30f, 0.f); }

__device__ __forceinline__ void two_sum_fold(float& s, float& c, float x) {
  const float t = s + x;
  const float bp = t - s;
  const float e = (s - (t - bp)) + (x - bp);
  s = t;
  c += e;
}

// inv = 1 / sqrt(r2), N of them one after the other, at raised wave priority.
// A SIMD takes full-rate vector instructions of two waves at a time, one per 2.0 to 2.4
// cycles (4.1 from one wave alone), and a reciprocal square root in 8.1. Mixed, with
// all waves alike, they do not add up: an interaction of eleven and one took 40 to 52
// cycles at eight waves per SIMD, by the order of its instructions, as waves waiting for
// the slow unit hold up the pairing of the others. With the four of a group raised it
// takes 33 in any order, which is the sum of the parts; groups of two, six or eight,
// or a raise some instructions earlier or later, are within 3%. Direct sum of 2^18
// bodies 15.8 -> 14.6 ms, 65,536 1.044 -> 0.962; ensembles of 256 clusters 659 -> 609 us,
// of 512 12.3 -> 11.3 ms; Barnes-Hut traversal of 300,007 bodies 488 -> 450 us, 2^22
// 4.31 -> 4.13 ms. The barriers keep the scheduler from moving the group apart.
template <int N>
__device__ __forceinline__ void rsq_group(const float (&r2)[N], float (&inv)[N]) {
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_setprio(3);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int k = 0; k < N; ++k) inv[k] = __builtin_amdgcn_rsqf(r2[k]);
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_setprio(0);
}

template <int B>
struct Targets {
  float x[B], y[B], z[B];
  float sx[B], sy[B], sz[B];  // compensated sums
  float cx[B], cy[B], cz[B];  // their error terms
};

// Accumulate the sources [j0, j1) (wave-uniform, j1 - j0 a multiple of 16) in plain sums
// of `chunk` sources (a multiple of 16).
// kUniform: all masses are equal, so the sum leaves them out (the caller's factor
// holds them): one multiply of twelve operations less. N = 2^18 17.35 -> 15.75 ms,
// 65,536 1.138 -> 1.042 ms. The padding then has to be far away, not massless.
template <int B, bool kGuard, bool kUniform>
__device__ __forceinline__ void accumulate(const float4* __restrict__ pm, int j0, int j1,
                                           float eps2_s, Targets<B>& t, int chunk = kChunk) {
  // eps2 is uniform and would stay an SGPR operand; a VGPR copy (the empty asm
  // hides its uniformity) turns the r^2 seed v_fma into an all-VGPR form.
  float eps2 = eps2_s;
  asm volatile("" : "+v"(eps2));
  for (int jc = j0; jc < j1; jc += chunk) {
    const int je = min(jc + chunk, j1);
    float px[B], py[B], pz[B];
#pragma unroll
    for (int b = 0; b < B; ++b) px[b] = py[b] = pz[b] = 0.f;
    // One register set of four sources: once their differences are taken, the scalar
    // loads of the next four are issued, so the load latency overlaps the rest of the
    // arithmetic. Two sets gained 10% over loads right before their use at N = 2^18;
    // with the sums in the order below one does as well. The memory clobbers keep the
    // compiler from sinking the loads next to their first use.
    // je - jc is a multiple of 4 (ranges are multiples of 16 sources).
    float4 q[4];
    auto load = [&](int j) {
      asm volatile("" ::: "memory");
#pragma unroll
      for (int u = 0; u < 4; ++u) q[u] = pm[j + u];  // wave-uniform: scalar loads
      asm volatile("" ::: "memory");
    };
    load(jc);
    for (int j = jc; j < je; j += 4) {
      float dx[4 * B], dy[4 * B], dz[4 * B], r2[4 * B], inv[4 * B], w[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        w[u] = q[u].w;
#pragma unroll
        for (int b = 0; b < B; ++b) {
          const int k = u * B + b;
          dx[k] = q[u].x - t.x[b];
          dy[k] = q[u].y - t.y[b];
          dz[k] = q[u].z - t.z[b];
          r2[k] = fmaf(dz[k], dz[k], fmaf(dy[k], dy[k], fmaf(dx[k], dx[k], eps2)));
        }
      }
      __builtin_amdgcn_sched_barrier(0);
      load(j + 4 < je ? j + 4 : j);  // the last step reloads its own (in range)
      rsq_group(r2, inv);
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int b = 0; b < B; ++b) {
          const int k = u * B + b;
          float s = (kUniform ? inv[k] : w[u] * inv[k]) * (inv[k] * inv[k]);
          if (kGuard) s = r2[k] > 0.f ? s : 0.f;
          px[b] = fmaf(dx[k], s, px[b]);
          py[b] = fmaf(dy[k], s, py[b]);
          pz[b] = fmaf(dz[k], s, pz[b]);
        }
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int b = 0; b < B; ++b) {
      two_sum_fold(t.sx[b], t.cx[b], px[b]);
      two_sum_fold(t.sy[b], t.cy[b], py[b]);
      two_sum_fold(t.sz[b], t.cz[b], pz[b]);
    }
  }
}

template <int B>
__device__ __forceinline__ void load_targets(const float4* __restrict__ pm, int ibase,
                                             Targets<B>& t) {
#pragma unroll
  for (int b = 0; b < B; ++b) {
    const float4 p = pm[ibase + 64 * b];
    t.x[b] = p.x;
    t.y[b] = p.y;
    t.z[b] = p.z;
    t.sx[b] = t.sy[b] = t.sz[b] = 0.f;
    t.cx[b] = t.cy[b] = t.cz[b] = 0.f;
  }
}

// Merge the K wave partials of one i-block, widened to FP64, in wave order 0..K-1
// through LDS. All K waves must call it; put(component, b, sum) is called for
// every component and target of the block, by the lane that holds the sum of its
// lane's target: one wave per component where there are three.
template <int B, int K, typename Put>
__device__ __forceinline__ void merge_waves(double (*part)[3][B][64], int wave, int lane,
                                            const Targets<B>& t, Put put) {
  if constexpr (K == 1) {
#pragma unroll
    for (int b = 0; b < B; ++b) {
      put(0, b, (double)t.sx[b] + (double)t.cx[b]);
      put(1, b, (double)t.sy[b] + (double)t.cy[b]);
      put(2, b, (double)t.sz[b] + (double)t.cz[b]);
    }
    return;
  }
#pragma unroll
  for (int b = 0; b < B; ++b) {
    part[wave][0][b][lane] = (double)t.sx[b] + (double)t.cx[b];
    part[wave][1][b][lane] = (double)t.sy[b] + (double)t.cy[b];
    part[wave][2][b][lane] = (double)t.sz[b] + (double)t.cz[b];
  }
  __syncthreads();
  for (int a = wave; a < 3; a += K)
#pragma unroll
    for (int b = 0; b < B; ++b) {
      double f = part[0][a][b][lane];
#pragma unroll
      for (int w = 1; w < K; ++w) f += part[w][a][b][lane];
      put(a, b, f);
    }
}

}  // namespace nbcore
