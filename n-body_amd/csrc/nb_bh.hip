// nb_bh.hip — Barnes-Hut force pass on gfx950.
//
// Replaces the reference's GPU octree (ParallelOctreeGPU.cpp:77-300 with the
// shaders boundingBoxPass1/2, resetOctree, expandOctree, countParticlesPerTask,
// prefixSum, addBlockSums, distributeParticles, insertParticles,
// propagateFatherOctree, pruneFather, pruneSubtrees) and the traversal shader
// forceCalcuBarnesHut.glsl:54-118, driven by ParticleSolverBHutGPU.cpp:25-50.
// It uses the reference's dormant Morton encoding (morton.glsl:37-98) as the
// spatial key instead of top-down bucketing.
//
// Pipeline per force pass (all on one stream, no host synchronisation, so the
// whole step can be captured into a hipGraph):
//   1. bbox        per-block min/max; every block of the next kernel folds them.
//   2. encode      30-bit Morton code per body (bit-exact restatement of
//                  morton.glsl: IEEE divide, clamp, 10-bit quantisation).
//   3. sort        LSD radix sort of (code, body index), 4 passes of 8 bits.
//                  Each pass: block digit histograms (the first one in 2.) and
//                  a stable scatter, whose blocks add up the counts before
//                  theirs themselves and whose per-wave ranks come from
//                  64-bit ballots (8 ballots give each lane the mask of lanes
//                  holding the same digit). From 2^22 bodies on a launch between
//                  the two adds up the counts. Small systems: 3 passes of 10 bits,
//                  whose blocks count all keys. Stable => sorted by (code, index).
//   4. mark        gather (x, y, z, m) into sorted order; per body the levels at
//                  which a node starts there; per tile the node counts of every
//                  level and the FP64 sums of (m, m x, m y, m z).
//   5. scan        of the tiles' counts and sums.
//   6. emit        per body the nodes that start or end there, and the FP64
//                  prefix: any node's mass and centre of mass is a difference of
//                  two prefix entries (cells are contiguous code ranges). The
//                  octree is breadth-first: a node with more than leaf_size bodies
//                  (and level < 10) splits into its non-empty Morton-digit
//                  children, which get consecutive indices. Ropes (`next`) point to
//                  the next sibling, or the parent's rope for the last child —
//                  the firstChild/next contract of Octree.cpp:264-294.
//   7. com         per node from the prefix; single-body nodes copy the body.
//                  Also the wave ranges of the traversal.
//   8. traverse    one lane per sorted body, stackless rope walk with the
//                  reference's opening test s^2 < theta^2 d^2 (Octree.cpp:320);
//                  a leaf that is not accepted is evaluated body by body.
#include <algorithm>
#include <cfloat>
#include <type_traits>
#include <vector>

#include "nb_force_core.h"
#include "nb_internal.h"

namespace {

// Block and tile sizes shared with the buffer layout are in nb_internal.h.
constexpr int kScanThreads = 256;
constexpr int kScanWaves = kScanThreads / 64;
// Traversal groups: each wave of the traversal takes one "wave range" of at
// most kWaveBodies consecutive sorted bodies. Ranges are cut along the tree: the
// children of a node holding more than kWaveBodies bodies are packed in order
// into ranges of at most kWaveBodies bodies (a child that itself holds more is
// handled at its own level; a level-10 leaf that holds more is split into
// chunks), so every range lies inside one parent cell and its bounding box
// stays tight. (With leaf_size <= kWaveBodies only level-10 leaves can hold
// more than kWaveBodies bodies.) A wave holds 64 / P copies of its range (P = the
// range's body count rounded up to a power of two), so at 32 bodies every range
// is evaluated by at least two slices: against 64-body ranges this measured 8%
// fewer interactions and a 4% faster traversal on the 4M two-disc system (16
// bodies: 14% slower, the walks dominate).
constexpr int kWaveBodies = NB_BH_WAVE_BODIES;
static_assert(kWaveBodies >= 4 && kWaveBodies <= 32 && (kWaveBodies & (kWaveBodies - 1)) == 0,
              "two wave ranges fit one wave");

// ---- 0. wave64 prefix sums on DPP ----------------------------------------------------
// Inclusive prefix over the 64 lanes of a wave, entirely in cross-lane DPP adds:
// shifts by 1, 2, 4 and 8 lanes inside each row of 16 (row_shr; a lane whose
// source lies outside its row adds 0), then lane 15 of rows 0 and 2 is added to
// rows 1 and 3 (row_bcast:15) and lane 31 to rows 2 and 3 (row_bcast:31). Six
// adds and no LDS round trips; the association is fixed, so FP64 prefixes are
// deterministic.
template <int kCtrl, int kRowMask>
__device__ __forceinline__ int dpp_shift(int v) {
  return __builtin_amdgcn_update_dpp(0, v, kCtrl, kRowMask, 0xf, false);
}
template <int kCtrl, int kRowMask>
__device__ __forceinline__ double dpp_shift(double v) {  // the two halves moved alike
  const uint64_t b = (uint64_t)__double_as_longlong(v);
  const uint32_t lo =
      (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)b, kCtrl, kRowMask, 0xf, false);
  const uint32_t hi =
      (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(b >> 32), kCtrl, kRowMask, 0xf, false);
  return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}
template <typename T>
__device__ __forceinline__ T wave_incl_scan(T v) {
  v += dpp_shift<0x111, 0xf>(v);  // row_shr:1
  v += dpp_shift<0x112, 0xf>(v);  // row_shr:2
  v += dpp_shift<0x114, 0xf>(v);  // row_shr:4
  v += dpp_shift<0x118, 0xf>(v);  // row_shr:8
  v += dpp_shift<0x142, 0xa>(v);  // row_bcast:15 into rows 1 and 3
  v += dpp_shift<0x143, 0xc>(v);  // row_bcast:31 into rows 2 and 3
  return v;
}

// Exclusive prefix of v over the threads of a kScanThreads-thread block (wave
// prefixes, then the wave totals added in wave order); total = the block's sum.
// wsum: kScanThreads / 64 ints of LDS, free again when this returns.
__device__ __forceinline__ int block_excl_scan(int v, int* wsum, int& total) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int incl = wave_incl_scan(v);
  if (lane == 63) wsum[wave] = incl;
  __syncthreads();
  int before = 0;
  total = 0;
#pragma unroll
  for (int w = 0; w < kScanThreads / 64; ++w) {
    before += w < wave ? wsum[w] : 0;
    total += wsum[w];
  }
  __syncthreads();
  return before + incl - v;
}

// ---- 1. bounding box --------------------------------------------------------
// Minimum and maximum per axis over a workgroup's threads; every thread gets them.
// red: 6 floats of LDS per wave.
template <int kWaves>
__device__ __forceinline__ void block_bounds(float (&mn)[3], float (&mx)[3], float (*red)[6]) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int off = 32; off > 0; off >>= 1)
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      mn[a] = fminf(mn[a], __shfl_xor(mn[a], off));
      mx[a] = fmaxf(mx[a], __shfl_xor(mx[a], off));
    }
  if (lane == 0)
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      red[wave][a] = mn[a];
      red[wave][3 + a] = mx[a];
    }
  __syncthreads();
#pragma unroll
  for (int w = 0; w < kWaves; ++w)
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      mn[a] = fminf(mn[a], red[w][a]);
      mx[a] = fmaxf(mx[a], red[w][3 + a]);
    }
}

// One thread's share of the bounds: bodies from, from + step, ...
__device__ __forceinline__ void fold_bounds(const float4* __restrict__ pm, int from, int step, int n,
                                            float (&mn)[3], float (&mx)[3]) {
#pragma unroll 4
  for (int i = from; i < n; i += step) {
    const float4 p = pm[i];
    mn[0] = fminf(mn[0], p.x); mx[0] = fmaxf(mx[0], p.x);
    mn[1] = fminf(mn[1], p.y); mx[1] = fmaxf(mx[1], p.y);
    mn[2] = fminf(mn[2], p.z); mx[2] = fmaxf(mx[2], p.z);
  }
}

// Partial bounds per block, folded by every block of k_morton. Also clears the
// radix passes' group counts.
__global__ __launch_bounds__(1024) void k_bbox_partial(const float4* __restrict__ pm, int n,
                                                       float* __restrict__ part,
                                                       int* __restrict__ group_hist, int counts) {
  __shared__ float red[16][6];
  const int step = gridDim.x * 1024;
  float mn[3] = {FLT_MAX, FLT_MAX, FLT_MAX};
  float mx[3] = {-FLT_MAX, -FLT_MAX, -FLT_MAX};
  for (int i = blockIdx.x * 1024 + threadIdx.x; i < counts; i += step) group_hist[i] = 0;
  fold_bounds(pm, blockIdx.x * 1024 + threadIdx.x, step, n, mn, mx);
  block_bounds<16>(mn, mx, red);
  if (threadIdx.x == 0)
    for (int a = 0; a < 3; ++a) {
      part[6 * blockIdx.x + a] = mn[a];
      part[6 * blockIdx.x + 3 + a] = mx[a];
    }
}

// ---- 2. Morton encode (morton.glsl:37-98) ------------------------------------
__device__ __forceinline__ uint32_t expand_bits(uint32_t v) {
  v = (v * 0x00010001u) & 0xFF0000FFu;
  v = (v * 0x00000101u) & 0x0F00F00Fu;
  v = (v * 0x00000011u) & 0xC30C30C3u;
  v = (v * 0x00000005u) & 0x49249249u;
  return v;
}

// Inverse of expand_bits on 10-bit values: gathers bits 0, 3, 6, ... of v.
__device__ __forceinline__ uint32_t compact_bits(uint32_t v) {
  v &= 0x49249249u;
  v = (v ^ (v >> 2)) & 0xC30C30C3u;
  v = (v ^ (v >> 4)) & 0x0F00F00Fu;
  v = (v ^ (v >> 8)) & 0xFF0000FFu;
  v = (v ^ (v >> 16)) & 0x000003FFu;
  return v;
}

// morton.glsl:68-75 and :49-51 with the extent given: n = clamp((p - lo) / ext, 0, 1),
// q = uint(clamp(n * 1024, 0, 1023)).
__device__ __forceinline__ uint32_t quantize(float p, float lo, float ext) {
  float nrm = __fdiv_rn(__fsub_rn(p, lo), ext);
  nrm = fminf(fmaxf(nrm, 0.f), 1.f);
  const float g = fminf(fmaxf(__fmul_rn(nrm, 1024.f), 0.f), 1023.f);
  return (uint32_t)g;
}

// Digit counts of one tile (kSortTile keys, 1024 threads) from the LDS histogram
// h: to the tile's row and, added up, to its group's.
__device__ __forceinline__ void publish_counts(const int* h, int* __restrict__ hist,
                                               int* __restrict__ group_hist) {
  if (threadIdx.x < 256) {
    const int c = h[threadIdx.x];
    hist[blockIdx.x * 256 + threadIdx.x] = c;
    if (c) atomicAdd(&group_hist[blockIdx.x / kSortGroup * 256 + threadIdx.x], c);
  }
}

// Codes, and the digit counts of the first radix pass. Every block folds
// the partial bounds itself (6 KB of L2 reads), which spares a launch of one block;
// kSelf: it takes the bounds of all bodies itself, which spares that launch, too.
// cubic = 1: one extent E = max_a max(max_a - min_a, 1e-6) on every axis (a cubic
// root cell, so every cell is a cube of side E / 2^level); cubic = 0: each axis
// over its own extent max(max_a - min_a, 1e-6), exactly morton.glsl's inputs.
template <bool kSelf>
__global__ __launch_bounds__(1024) void k_morton(const float4* __restrict__ pm, int n, int cubic,
                                                 const float* __restrict__ part, int nparts,
                                                 float* __restrict__ geom,
                                                 uint32_t* __restrict__ codes,
                                                 int* __restrict__ hist,
                                                 int* __restrict__ group_hist) {
  __shared__ float red[16][6];
  __shared__ int h[256];
  if (threadIdx.x < 256) h[threadIdx.x] = 0;
  float mn[3] = {FLT_MAX, FLT_MAX, FLT_MAX};
  float mx[3] = {-FLT_MAX, -FLT_MAX, -FLT_MAX};
  if (kSelf) {
    fold_bounds(pm, threadIdx.x, 1024, n, mn, mx);
  } else if ((int)threadIdx.x < nparts) {  // nparts <= kBboxBlocks
    for (int a = 0; a < 3; ++a) {
      mn[a] = part[6 * threadIdx.x + a];
      mx[a] = part[6 * threadIdx.x + 3 + a];
    }
  }
  block_bounds<16>(mn, mx, red);  // ends behind a barrier: h is clear
  float ext[3], E = 0.f;
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    ext[a] = fmaxf(__fsub_rn(mx[a], mn[a]), 1e-6f);
    E = fmaxf(E, ext[a]);
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    for (int a = 0; a < 3; ++a) {
      geom[a] = mn[a];
      geom[3 + a] = mx[a];
    }
    for (int l = 0; l <= kMaxLevel; ++l) {
      const float s = ldexpf(E, -l);
      geom[6 + l] = __fmul_rn(s, s);
    }
    geom[6 + kMaxLevel + 1] = E;  // cubic root extent
  }
#pragma unroll
  for (int r = 0; r < kSortTile / 1024; ++r) {
    const int i = blockIdx.x * kSortTile + r * 1024 + threadIdx.x;
    if (i < n) {
      const float4 p = pm[i];
      const uint32_t qx = quantize(p.x, mn[0], cubic ? E : ext[0]);
      const uint32_t qy = quantize(p.y, mn[1], cubic ? E : ext[1]);
      const uint32_t qz = quantize(p.z, mn[2], cubic ? E : ext[2]);
      const uint32_t code = expand_bits(qx) * 4u + expand_bits(qy) * 2u + expand_bits(qz);
      codes[i] = code;
      if (!kSelf) atomicAdd(&h[code & 255u], 1);
    }
  }
  if (kSelf) return;  // as its digits are counted where they are sorted
  __syncthreads();
  publish_counts(h, hist, group_hist);
}

// FP64 prefix of (m, m x, m y, m z): prefix[k] = sum over sorted bodies < k.
__device__ __forceinline__ double4 body_moments(float4 p) {
  const double m = p.w;
  return make_double4(m, m * (double)p.x, m * (double)p.y, m * (double)p.z);
}
__device__ __forceinline__ double4 add4(double4 a, double4 b) {
  return make_double4(a.x + b.x, a.y + b.y, a.z + b.z, a.w + b.w);
}

__device__ __forceinline__ double4 shfl_up4(double4 v, int off) {
  return make_double4(__shfl_up(v.x, off), __shfl_up(v.y, off), __shfl_up(v.z, off),
                      __shfl_up(v.w, off));
}
__device__ __forceinline__ double4 shfl4(double4 v, int lane) {
  return make_double4(__shfl(v.x, lane), __shfl(v.y, lane), __shfl(v.z, lane), __shfl(v.w, lane));
}
__device__ __forceinline__ double4 wave_incl_scan4(double4 v) {
  return make_double4(wave_incl_scan(v.x), wave_incl_scan(v.y), wave_incl_scan(v.z),
                      wave_incl_scan(v.w));
}

// ---- 3. radix sort ------------------------------------------------------------
__global__ __launch_bounds__(1024) void k_radix_hist(const uint32_t* __restrict__ keys, int n,
                                                     int shift, int* __restrict__ hist,
                                                     int* __restrict__ group_hist) {
  __shared__ int h[256];
  if (threadIdx.x < 256) h[threadIdx.x] = 0;
  __syncthreads();
#pragma unroll
  for (int r = 0; r < kSortTile / 1024; ++r) {
    const int e = blockIdx.x * kSortTile + r * 1024 + threadIdx.x;
    if (e < n) atomicAdd(&h[(keys[e] >> shift) & 255u], 1);
  }
  __syncthreads();
  publish_counts(h, hist, group_hist);
}

// A pass's group counts made first output indices of each group's digits: the number of
// smaller digits anywhere plus that of the same digit in earlier groups. One workgroup,
// four threads per digit. Without it every block of the scatter adds up all groups'
// counts itself, n / 2^17 KB for 2048 keys: from kScanGroups groups (2^22 bodies) on that
// takes longer than this launch. Build in ns per body without / with it: 2^20 0.155 /
// 0.156, 2^21 0.137 / 0.140, 2^22 0.133 / 0.129, 2^23 0.126 / 0.117, 2^24 0.140 / 0.122,
// 2^25 0.159 / 0.125, 2^26 0.196 / 0.123.
constexpr int kScanGroups = 32;
__global__ __launch_bounds__(1024) void k_radix_groups(int* __restrict__ group_hist, int groups) {
  constexpr int kBatch = 8;  // loads in flight
  __shared__ int part[4][256];
  __shared__ int wsum[4];
  const int d = threadIdx.x & 255, q = threadIdx.x >> 8;
  const int per = (groups + 3) / 4, g0 = min(q * per, groups), g1 = min(g0 + per, groups);
  int* const mine = group_hist + d;
  int sum = 0;
#pragma unroll 8
  for (int g = g0; g < g1; ++g) sum += mine[g * 256];
  part[q][d] = sum;
  __syncthreads();
  int total = 0, at = 0;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    total += part[k][d];
    at += k < q ? part[k][d] : 0;
  }
  const int incl = wave_incl_scan(total), wave = d >> 6;  // each quarter scans the same totals
  if (q == 0 && (d & 63) == 63) wsum[wave] = incl;
  __syncthreads();
  at += incl - total;
  for (int w = 0; w < wave; ++w) at += wsum[w];
  for (int g = g0; g < g1; g += kBatch) {
    int c[kBatch];
#pragma unroll
    for (int k = 0; k < kBatch; ++k) c[k] = g + k < g1 ? mine[(g + k) * 256] : 0;
#pragma unroll
    for (int k = 0; k < kBatch; ++k) {
      if (g + k < g1) mine[(g + k) * 256] = at;
      at += c[k];
    }
  }
}

// Mask of the active lanes whose digit of kBits bits equals this lane's digit.
template <int kBits>
__device__ __forceinline__ uint64_t match_digit(uint32_t d, uint64_t active) {
  uint64_t m = active;
#pragma unroll
  for (int b = 0; b < kBits; ++b) {
    const bool bit = (d >> b) & 1u;
    const uint64_t bb = __builtin_amdgcn_ballot_w64(bit);
    m &= bit ? bb : ~bb;
  }
  return m;
}

// Stable scatter of one digit's pass. A tile's first output index of a digit
// is the number of smaller digits anywhere plus the number of its own digit in
// earlier tiles: each block adds these up itself from the groups' counts and the
// counts of the tiles before it in its group (four threads per digit; at most 31
// groups and 63 tiles), so a pass is two launches without a scan between them; of
// larger systems k_radix_groups has added up the groups' (groups = 0). The tile is first reordered in LDS by digit (stable ranks from
// per-wave ballots, waves and rounds in element order), then written out in LDS
// order: consecutive threads write the runs of equal digits to consecutive global
// addresses instead of 64 scattered lines per wave store. Two keys per thread: a
// pass over a small system is a chain of latencies (65,536 keys, counts and scatter:
// 27 us in four launches with eight keys per thread, 11 us now; 2^22 keys 56 and 53).
// Eight bits per pass: four passes. kSelf: the blocks count the digits of all keys
// themselves, before and after their tile, which spares the counting launches, and
// as no table of counts goes through memory the digits have ten bits: three passes,
// three launches of 8.3 us at 20,011 keys in place of seven (30 us in all).
// kFirst: the values are the indices themselves.
constexpr int kCopies = 2;  // of a count, for even and odd lanes: fewer atomics on one word
template <bool kFirst, bool kSelf>
__global__ __launch_bounds__(1024) void k_radix_scatter(
    const uint32_t* __restrict__ keys_in, const uint32_t* __restrict__ vals_in, int n, int shift,
    const int* __restrict__ hist, const int* __restrict__ group_hist, int groups,
    uint32_t* __restrict__ keys_out, uint32_t* __restrict__ vals_out) {
  constexpr int kRounds = kSortTile / 1024;
  constexpr int kBits = kSelf ? 10 : 8, kDigits = 1 << kBits, kShare = kSelf ? kCopies : 1024 / kDigits;
  __shared__ int whist[16][kDigits];  // per wave: digit counts, then those of the waves before
  __shared__ int s_part[2][kShare][kDigits + (kSelf ? 64 / kCopies : 0)];
  __shared__ int s_local[kDigits];      // a digit's first tile slot
  __shared__ int s_to_global[kDigits];  // a digit's first output index minus its first tile slot
  __shared__ uint32_t sk[kSortTile], sv[kSortTile];
  __shared__ int wsum[2][kDigits / 64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const uint64_t lt = (uint64_t(1) << lane) - 1;
  const int tile0 = blockIdx.x * kSortTile;
  // Wave w owns the tile elements [w * kSortTile / 16, (w + 1) * kSortTile / 16)
  const int base = tile0 + wave * (kSortTile / 16) + lane;
  uint32_t key[kRounds], val[kRounds];
#pragma unroll
  for (int r = 0; r < kRounds; ++r) {
    const int e = base + 64 * r;
    key[r] = e < n ? keys_in[e] : 0u;
    val[r] = kFirst ? (uint32_t)e : e < n ? vals_in[e] : 0u;
  }
  if (kSelf) {
    // s_part[0]: digits of the tiles after this one, s_part[1]: of those before
    int* const parts = &s_part[0][0][0];
    for (int i = threadIdx.x; i < (int)(sizeof(s_part) / 4); i += 1024) parts[i] = 0;
    __syncthreads();
    const auto count = [&](int from, int to, int* h) {  // from: a multiple of four
      for (int e = from + 4 * threadIdx.x; e < to; e += 4096) {
        uint32_t k[4];
        if (e + 3 < to) {
          const uint4 v = *reinterpret_cast<const uint4*>(keys_in + e);
          k[0] = v.x, k[1] = v.y, k[2] = v.z, k[3] = v.w;
        } else {
          for (int u = 0; u < 4; ++u) k[u] = e + u < to ? keys_in[e + u] : 0u;
        }
#pragma unroll
        for (int u = 0; u < 4; ++u)
          if (e + u < to) atomicAdd(&h[(k[u] >> shift) & (kDigits - 1)], 1);
      }
    };
    count(0, tile0, s_part[1][lane & (kCopies - 1)]);
    count(tile0 + kSortTile, n, s_part[0][lane & (kCopies - 1)]);
  } else {
    const int d = threadIdx.x & (kDigits - 1), q = threadIdx.x >> kBits;
    const int mine = blockIdx.x / kSortGroup;
    int total = 0, before = 0;
    for (int g = q; g < groups; g += kShare) {
      const int c = group_hist[g * kDigits + d];
      total += c;
      before += g < mine ? c : 0;
    }
    if (groups == 0 && q == 0) before = group_hist[mine * kDigits + d];
    for (int t = mine * kSortGroup + q; t < (int)blockIdx.x; t += kShare) before += hist[t * kDigits + d];
    s_part[0][q][d] = total;
    s_part[1][q][d] = before;
  }
#pragma unroll
  for (int k = 0; k < kDigits / 64; ++k) whist[wave][64 * k + lane] = 0;  // the wave's own row
  __builtin_amdgcn_wave_barrier();
  int rank[kRounds];
#pragma unroll
  for (int r = 0; r < kRounds; ++r) {
    const bool in = base + 64 * r < n;
    const uint32_t d = (key[r] >> shift) & (kDigits - 1);
    const uint64_t m = match_digit<kBits>(d, __builtin_amdgcn_ballot_w64(in));
    rank[r] = whist[wave][d] + __popcll(m & lt);
    __builtin_amdgcn_wave_barrier();
    if (in && (m & lt) == 0) whist[wave][d] += __popcll(m);
    __builtin_amdgcn_wave_barrier();
  }
  __syncthreads();
  int cnt = 0, total = 0, before = 0, incl_c = 0, incl_t = 0;
  if (threadIdx.x < kDigits) {
    const int d = threadIdx.x;
#pragma unroll
    for (int w = 0; w < 16; ++w) {
      const int c = whist[w][d];
      whist[w][d] = cnt;
      cnt += c;
    }
#pragma unroll
    for (int q = 0; q < kShare; ++q) {
      total += s_part[0][q][d];
      before += s_part[1][q][d];
    }
    if (kSelf) total += before + cnt;
    incl_c = wave_incl_scan(cnt);
    incl_t = wave_incl_scan(total);
    if (lane == 63) {
      wsum[0][wave] = incl_c;
      wsum[1][wave] = incl_t;
    }
  }
  __syncthreads();
  if (threadIdx.x < kDigits) {
    const int d = threadIdx.x;
    int local = incl_c - cnt, global = incl_t - total + before;
    for (int w = 0; w < wave; ++w) {
      local += wsum[0][w];
      global += wsum[1][w];
    }
    s_local[d] = local;
    s_to_global[d] = global - local;
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < kRounds; ++r) {
    const uint32_t d = (key[r] >> shift) & (kDigits - 1);
    const int slot = s_local[d] + whist[wave][d] + rank[r];
    if (base + 64 * r < n && slot >= 0 && slot < kSortTile) {  // always, for consistent counts
      sk[slot] = key[r];
      sv[slot] = val[r];
    }
  }
  __syncthreads();
  const int count = min(kSortTile, n - tile0);
#pragma unroll
  for (int r = 0; r < kRounds; ++r) {
    const int i = r * 1024 + threadIdx.x;
    if (i < count) {
      const uint32_t k = sk[i];
      const int dst = i + s_to_global[(k >> shift) & (kDigits - 1)];
      if (dst >= 0 && dst < n) {
        keys_out[dst] = k;
        vals_out[dst] = sv[i];
      }
    }
  }
}

// ---- 4. bodies in sorted order ------------------------------------------------
// Morton reordering of the resident state: dst[k] = src[perm[k]] per component.
__global__ __launch_bounds__(256) void k_permute_d3(const double* __restrict__ src,
                                                    const uint32_t* __restrict__ perm, int n,
                                                    double* __restrict__ dst) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < n) {
    const uint32_t p = perm[i];
    if (p < (uint32_t)n) {
      dst[i] = src[p];
      dst[n + i] = src[n + p];
      dst[2 * n + i] = src[2 * n + p];
    }
  }
}

__global__ __launch_bounds__(256) void k_permute_f32(const float* __restrict__ src,
                                                     const uint32_t* __restrict__ perm, int n,
                                                     float* __restrict__ dst) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < n) {
    const uint32_t p = perm[i];
    if (p < (uint32_t)n) dst[i] = src[p];
  }
}

// ---- 6. octree ------------------------------------------------------------------------
__device__ __forceinline__ int span_count(int w) { return w >> 4; }
__device__ __forceinline__ int span_level(int w) { return w & 15; }

// Octal digits that two 30-bit codes share from the top (0..10).
__device__ __forceinline__ int common_level(uint32_t a, uint32_t b) {
  const uint32_t x = a ^ b;
  return x ? (29 - (31 - __clz((int)x))) / 3 : kMaxLevel;
}

constexpr int kTreeWaves = kTreeTile / 64;  // one body per thread
constexpr int kMaxLeaf = 64;  // bodies per leaf that nb_create accepts

// The octree without a loop over its levels. In the sorted codes every cell is a
// run of bodies, so a body i can start one cell per level, from the level d(i) at
// which it parts from the body before it (d = digits in common + 1) downwards;
// such a cell is a node if it is the root or its parent holds more than `leaf`
// bodies. The cell of level l around i does so exactly when some leaf + 1
// consecutive bodies, i among them, share l digits. With
//   c(k) = digits in common of the codes k and k + leaf,
//   depth(i) = max of c(k) over k = i - leaf .. i,
// the nodes that start at i are therefore those of the levels d(i) .. D(i),
// D(i) = min(depth(i) + 1, 10), and a node of level l there has children exactly
// when l < D(i). A node's index is the number of nodes of the levels above plus
// the number of nodes of its level that start before i: a count per tile and
// level (here), a scan of the counts (k_tree_scan), and a rank inside the tile
// (k_tree_emit). Three launches of one coalesced pass each take the place of a
// count, a scan and an emission for each of the ten levels with their binary
// searches (gather to centres of mass at 65,536 bodies: 31 launches, 175 us -> 4
// launches, 30 us; at 2^22: 508 -> 260 us).
//
// This kernel also brings the bodies into sorted order and sums the moments of
// its tile for the FP64 prefix: it reads the permutation and the codes anyway.
// Tiles of 1024 bodies, one per thread: at 65,536 bodies these kernels are chains
// of latencies, and eight bodies per thread took 17 + 28 us where one takes 7 + 7 us.
__global__ __launch_bounds__(kTreeTile) void k_tree_mark(
    const uint32_t* __restrict__ codes, const uint32_t* __restrict__ perm,
    const float4* __restrict__ pm, int n, int leaf, float4* __restrict__ pms,
    double4* __restrict__ part, unsigned char* __restrict__ marks, int* __restrict__ level_cnt) {
  __shared__ uint32_t s_code[kTreeTile + 2 * kMaxLeaf];  // the tile and kMaxLeaf on either side
  __shared__ signed char s_win[2][kTreeTile + kMaxLeaf];
  __shared__ int s_cnt[kLevels][kTreeWaves];
  __shared__ double4 s_mom[kTreeWaves];
  const int base = blockIdx.x * kTreeTile;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int i = base + threadIdx.x;
  float4 q = make_float4(0.f, 0.f, 0.f, 0.f);
  if (i < n) {
    const uint32_t p = perm[i];
    if (p < (uint32_t)n) q = pm[p];
  }
  for (int x = threadIdx.x; x < kTreeTile + 2 * kMaxLeaf; x += kTreeTile) {
    const int k = base - kMaxLeaf + x;
    s_code[x] = k >= 0 && k < n ? codes[k] : 0u;
  }
  __syncthreads();
  // c(k) at s_win[0][k - (base - kMaxLeaf)]; leaf <= kMaxLeaf, so k + leaf is staged
  for (int x = threadIdx.x; x < kTreeTile + kMaxLeaf; x += kTreeTile) {
    const int k = base - kMaxLeaf + x;
    s_win[0][x] = k >= 0 && k + leaf < n ? (signed char)common_level(s_code[x], s_code[x + leaf]) : -1;
  }
  // windows of 2, 4, ... entries ending at x, up to the largest power of two
  // that leaf + 1 holds: two of those cover a window of leaf + 1
  int buf = 0, span = 1;
  for (; 2 * span <= leaf + 1; span *= 2, buf ^= 1) {
    __syncthreads();
    for (int x = threadIdx.x; x < kTreeTile + kMaxLeaf; x += kTreeTile) {
      const signed char v = s_win[buf][x];
      s_win[buf ^ 1][x] = x >= span ? max(v, s_win[buf][x - span]) : v;
    }
  }
  __syncthreads();
  int d = kLevels, D = 0;  // no node
  if (i < n) {
    const int x = kMaxLeaf + threadIdx.x;
    const int depth = max(s_win[buf][x], s_win[buf][x - (leaf + 1 - span)]);
    D = min(depth + 1, kMaxLevel);
    d = i == 0 ? 0 : common_level(s_code[x - 1], s_code[x]) + 1;
    marks[i] = (unsigned char)(d << 4 | D);
    pms[i] = q;
  }
  int cnt = 0;  // lane l: this wave's nodes of level l
#pragma unroll
  for (int l = 0; l < kLevels; ++l) {
    const int c = __popcll(__ballot(d <= l && l <= D));
    cnt = lane == l ? c : cnt;
  }
  const double4 mom = wave_incl_scan4(body_moments(q));
  if (lane < kLevels) s_cnt[lane][wave] = cnt;
  if (lane == 63) s_mom[wave] = mom;
  __syncthreads();
  if (threadIdx.x < kLevels) {
    int c = 0;
    for (int w = 0; w < kTreeWaves; ++w) c += s_cnt[threadIdx.x][w];
    level_cnt[threadIdx.x * gridDim.x + blockIdx.x] = c;
  } else if (threadIdx.x == 64) {
    double4 m = s_mom[0];
    for (int w = 1; w < kTreeWaves; ++w) m = add4(m, s_mom[w]);
    part[blockIdx.x] = m;
  }
}

// Wave ranges of one node's children (see kWaveBodies): calls out(start, count)
// for each range in order; returns how many there are.
template <typename Out>
__device__ __forceinline__ int pack_ranges(const int* starts, const int* ends, int nc, int l,
                                           int leaf, Out out) {
  int r = 0, run_s = 0, run_n = 0;
  for (int q = 0; q < nc; ++q) {
    const int cn = ends[q] - starts[q];
    if (cn > kWaveBodies) {
      if (run_n) { out(r++, run_s, run_n); }
      run_n = 0;
      if (l + 1 == kMaxLevel || cn <= leaf)  // a leaf: chunks (internal: its own level)
        for (int o = 0; o < cn; o += kWaveBodies) out(r++, starts[q] + o, min(kWaveBodies, cn - o));
    } else {
      if (run_n + cn > kWaveBodies) {
        out(r++, run_s, run_n);
        run_n = 0;
      }
      if (run_n == 0) run_s = starts[q];
      run_n += cn;
    }
  }
  if (run_n) out(r++, run_s, run_n);
  return r;
}

// P lanes per copy of a range of `count` bodies: a power of two >= count, >= 4.
__device__ __forceinline__ int copy_lanes(int count) {
  return count <= 4 ? 4 : 1 << (32 - __clz(count - 1));
}

// Number of records emit_records makes of one node's wave ranges.
__device__ __forceinline__ int count_records(const int* starts, const int* ends, int nc, int l,
                                             int leaf, bool pairs) {
  if (!pairs) return pack_ranges(starts, ends, nc, l, leaf, [](int, int, int) {});
  int per_width[4] = {0, 0, 0, 0};  // ranges of width 4, 8, 16, 32
  pack_ranges(starts, ends, nc, l, leaf, [&](int, int, int c) {
    const int k = 29 - __clz(copy_lanes(c));
#pragma unroll
    for (int j = 0; j < 4; ++j) per_width[j] += j == k ? 1 : 0;
  });
  return ((per_width[0] + 1) >> 1) + ((per_width[1] + 1) >> 1) + ((per_width[2] + 1) >> 1) +
         ((per_width[3] + 1) >> 1);
}

// One node's wave ranges (pack_ranges) as records of two sibling ranges of the
// same copy width (a pair shares one lane layout, so neither range idles
// lanes), (start, count, start, count), or of one range, (start, count, 0, 0):
// each range waits for the next of its width, in order. Writes count_records()
// records from record `first` on. There are at most as many records as ranges,
// and at most n ranges. Without `pairs` every range is a record of its own.
__device__ __forceinline__ void emit_records(int4* __restrict__ waves, int first, int n,
                                             const int* starts, const int* ends, int nc, int l,
                                             int leaf, bool pairs) {
  int2 wait[4];  // one waiting range per width 4, 8, 16, 32
#pragma unroll
  for (int k = 0; k < 4; ++k) wait[k] = make_int2(0, 0);
  int r = 0;
  auto put = [&](int4 v) {
    if (first + r < n) waves[first + r] = v;
    ++r;
  };
  if (!pairs) {
    pack_ranges(starts, ends, nc, l, leaf, [&](int, int a, int c) { put(make_int4(a, c, 0, 0)); });
    return;
  }
  pack_ranges(starts, ends, nc, l, leaf, [&](int, int a, int c) {
    const int k = 29 - __clz(copy_lanes(c));  // 4 -> 0, ..., 32 -> 3
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (j == k) {
        if (wait[j].y > 0) {
          put(make_int4(wait[j].x, wait[j].y, a, c));
          wait[j] = make_int2(0, 0);
        } else {
          wait[j] = make_int2(a, c);
        }
      }
  });
#pragma unroll
  for (int j = 0; j < 4; ++j)
    if (wait[j].y > 0) put(make_int4(wait[j].x, wait[j].y, 0, 0));
}

// Where the traversal's work items go.
struct Records {
  int4* waves;
  int* ctl;   // [0] records, [1] traversal ticket
  int* hist;  // [kCostBuckets] records per cost bucket, then [kCostBuckets] cursors
};

// Before a build's first record: no records, a fresh ticket, empty buckets, and the
// ranges of a system that no node packs. One workgroup.
__device__ __forceinline__ void start_records(const Records& R, int n, int leaf, int pairs) {
  for (int k = threadIdx.x; k < 2 * kCostBuckets; k += blockDim.x) R.hist[k] = 0;
  __syncthreads();
  if (threadIdx.x != 0) return;
  int r = 0;
  if (n <= kWaveBodies) {
    R.waves[r++] = make_int4(0, n, 0, 0);
  } else if (n <= leaf) {
    // the root is itself a leaf, so no node packs ranges below it: chunk it,
    // two full chunks per record, a shorter last chunk on its own
    for (int o = 0; o < n; o += kWaveBodies) {
      const int k = min(kWaveBodies, n - o), o2 = o + kWaveBodies;
      if (pairs && k == kWaveBodies && n - o2 >= kWaveBodies) {
        R.waves[r++] = make_int4(o, k, o2, kWaveBodies);
        o = o2;
      } else {
        R.waves[r++] = make_int4(o, k, 0, 0);
      }
    }
  }
  R.ctl[0] = r;
  R.ctl[1] = 0;  // traversal ticket
}

// ---- 6b. scan and emission -------------------------------------------------------------
// Block 0: exclusive scan of the tiles' moments in a fixed order: each thread
// folds a contiguous run of tiles, the 256 run totals are scanned (wave DPP
// prefixes, then the 4 wave totals in wave order), then each thread rewrites its
// run; part[tiles] receives the total. Block 1 + l: the same for the tiles' node
// counts of level l, whose total goes to counters[2 + l]. The last block starts the
// records. A system of at most 64 tiles needs no launch for this (k_tree_emit).
__global__ __launch_bounds__(kScanThreads) void k_tree_scan(double4* __restrict__ part,
                                                            int* __restrict__ level_cnt,
                                                            int tiles, int n, int leaf, int pairs,
                                                            int* __restrict__ counters,
                                                            Records records) {
  if (blockIdx.x == 1 + kLevels) {
    start_records(records, n, leaf, pairs);
    return;
  }
  const int per = (tiles + kScanThreads - 1) / kScanThreads;
  const int b0 = min((int)threadIdx.x * per, tiles);
  const int b1 = min(b0 + per, tiles);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (blockIdx.x == 0) {
    double4 tot = make_double4(0, 0, 0, 0);
    for (int b = b0; b < b1; ++b) tot = add4(tot, part[b]);
    const double4 incl = wave_incl_scan4(tot);
    __shared__ double4 wtot[kScanWaves];
    if (lane == 63) wtot[wave] = incl;
    __syncthreads();
    double4 run = make_double4(0, 0, 0, 0), grand = make_double4(0, 0, 0, 0);
    for (int w = 0; w < kScanWaves; ++w) {
      if (w < wave) run = add4(run, wtot[w]);
      grand = add4(grand, wtot[w]);
    }
    const double4 below = shfl_up4(incl, 1);  // inclusive value of the lane below
    if (lane > 0) run = add4(run, below);
    for (int b = b0; b < b1; ++b) {
      const double4 v = part[b];
      part[b] = run;
      run = add4(run, v);
    }
    if (threadIdx.x == 0) part[tiles] = grand;
    return;
  }
  int* cnt = level_cnt + (blockIdx.x - 1) * tiles;
  __shared__ int wsum[kScanWaves];
  int sum = 0, total = 0;
  for (int b = b0; b < b1; ++b) sum += cnt[b];
  int run = block_excl_scan(sum, wsum, total);
  for (int b = b0; b < b1; ++b) {
    const int v = cnt[b];
    cnt[b] = run;
    run += v;
  }
  if (threadIdx.x == 0) counters[1 + blockIdx.x] = total;
}

// Per tile: the exclusive FP64 prefix of the moments (wave DPP prefixes, then a
// DPP prefix of the 16 wave totals: a fixed association, no atomics) and the
// nodes that start or end in it. The body i that starts a node writes its first
// child (which starts at i too), its start and its level; the last body i of a
// node writes its end and its rope: the node of the lowest level that starts at
// i + 1, which is a sibling of it or of the closest ancestor that has one. Few
// levels are active in 64 neighbouring bodies, so the others are branched over
// (at 2^22 bodies 141 us without that, 94 us with it).
// kSelf: at most 64 tiles, whose counts and moments every block scans itself, one
// lane per tile (a launch less: 4.6 us of 65,536 bodies' step); the first block
// starts the records.
template <bool kSelf>
__global__ __launch_bounds__(kTreeTile) void k_tree_emit(
    const float4* __restrict__ pms, int n, int leaf, int pairs, const double4* __restrict__ part,
    const unsigned char* __restrict__ marks, const int* __restrict__ level_cnt,
    const int* __restrict__ counters, Records records, int64_t max_nodes, double4* __restrict__ prefix,
    nb_node* __restrict__ nodes, int* __restrict__ next, int* __restrict__ node_end,
    int* __restrict__ level_off, int* __restrict__ flags) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const uint64_t lt = (uint64_t(1) << lane) - 1;
  const int e = blockIdx.x * kTreeTile + threadIdx.x;
  __shared__ double4 s_mom[kTreeWaves];
  __shared__ int s_off[kLevels][kTreeWaves];  // node starts per wave, then their first index
  __shared__ int s_tot[kLevels];              // nodes of each level
  const int tile = blockIdx.x, tiles = gridDim.x;
  if (kSelf && tile == 0) start_records(records, n, leaf, pairs);
  const double4 x0 = e < n ? body_moments(pms[e]) : make_double4(0, 0, 0, 0);
  const int mark = e < n ? marks[e] : kLevels << 4;
  const int dn = e + 1 < n ? marks[e + 1] >> 4 : 0;  // after the last body every node ends
  const int d = mark >> 4, D = e < n ? mark & 15 : -1;
  const double4 x = wave_incl_scan4(x0);
  int cnt = 0;
#pragma unroll
  for (int l = 0; l < kLevels; ++l) {
    const int c = __popcll(__ballot(d <= l && l <= D));
    cnt = lane == l ? c : cnt;
  }
  if (lane == 63) s_mom[wave] = x;
  if (lane < kLevels) s_off[lane][wave] = cnt;
  // level `wave`: its nodes in earlier tiles, and in all
  int earlier = 0;
  if (wave < kLevels) {
    int total;
    if (kSelf) {
      const int v = lane < tiles ? level_cnt[wave * tiles + lane] : 0;
      const int incl = wave_incl_scan(v);
      earlier = __shfl(incl - v, tile);
      total = __shfl(incl, 63);
    } else {
      earlier = level_cnt[wave * tiles + tile];
      total = counters[2 + wave];
    }
    if (lane == 0) s_tot[wave] = total;
  }
  __syncthreads();
  if (wave < kLevels) {  // level l's node index at the start of every wave
    const int l = wave;
    int lo = 0;
    for (int k = 0; k < l; ++k) lo += s_tot[k];
    const int v = lane < kTreeWaves ? s_off[l][lane] : 0;
    const int at = wave_incl_scan(v) - v;
    if (lane < kTreeWaves) s_off[l][lane] = lo + earlier + at;
    if (tile == 0 && lane == 0) {
      level_off[l] = lo;
      if (l == kMaxLevel) level_off[l + 1] = lo + s_tot[l];
    }
  } else if (wave == kLevels) {
    const double4 v = lane < kTreeWaves ? s_mom[lane] : make_double4(0, 0, 0, 0);
    const double4 below = shfl_up4(wave_incl_scan4(v), 1);
    double4 run, all;  // exclusive start of this tile, and the total
    if (kSelf) {
      const double4 t = lane < tiles ? part[lane] : make_double4(0, 0, 0, 0);
      const double4 incl = wave_incl_scan4(t);
      const double4 before = shfl4(incl, max(tile - 1, 0));
      run = tile > 0 ? before : make_double4(0, 0, 0, 0);
      all = shfl4(incl, 63);
    } else {
      run = part[tile];
      all = part[tiles];
    }
    if (lane < kTreeWaves) s_mom[lane] = lane > 0 ? add4(run, below) : run;
    if (tile == tiles - 1 && lane == 0) prefix[n] = all;
  }
  __syncthreads();
  const double4 below = shfl_up4(x, 1);  // inclusive value of the lane below
  const double4 start = s_mom[wave];
  if (e < n) prefix[e] = lane > 0 ? add4(start, below) : start;
  // idx[l]: index of a node of level l that starts at e
  int idx[kLevels + 1], rope = -1;
#pragma unroll
  for (int l = 0; l < kLevels; ++l) {
    const bool starts = d <= l && l <= D;
    idx[l] = s_off[l][wave] + __popcll(__ballot(starts) & lt);
    if (l == dn && e + 1 < n) rope = idx[l] + (starts ? 1 : 0);
  }
  idx[kLevels] = -1;
  bool over = false;
#pragma unroll
  for (int l = 0; l < kLevels; ++l) {
    const bool starts = d <= l && l <= D, ends = dn <= l && l <= D;
    if (__ballot(starts || ends) == 0) continue;
    const int64_t at = idx[l];
    if (starts && at < max_nodes) {
      nodes[at].first = l < D ? idx[l + 1] : -1;
      nodes[at].start = e;
      nodes[at].span = l;
    }
    const int64_t in = at - (starts ? 0 : 1);  // the node of level l around e
    if (ends && in >= 0 && in < max_nodes) {
      next[in] = rope;
      node_end[in] = e + 1;
    }
    over = over || (starts && at >= max_nodes);
  }
  if (over) atomicOr(flags, 2);
}

// ---- 7. centre of mass and opening radius -------------------------------------------
// Squared opening radius of the default traversal: r = s_l / theta + delta, where
// s_l is the cell side of the reference's test (Octree.cpp:311-320) and delta the
// distance from the COM to the cell's geometric centre. This is the offset term of
// Barnes' modified criterion (J. Comput. Phys. 87, 1990; the default of his
// treecode 1.4): a cell whose mass sits near one face can hold bodies much closer
// to a target than s_l / theta suggests. The cell is the 3l-bit prefix of its first
// body's code, so its centre is bmin + (index + 1/2) * extent / 2^l per axis.
// Every operation is one IEEE operation rounded to nearest, in a fixed order and
// with contraction into FMAs off (HIP's __fadd_rn and __fmul_rn are plain
// operators that -ffp-contract=fast may fuse, and its __fsqrt_rn is the native
// approximation; division and sqrtf are correctly rounded by default), so the
// CPU build computes the same bits from the same COM. Massless cells get -1:
// always accepted, never listed.
__device__ __forceinline__ float open_radius2(float4 cm, uint32_t code, int l,
                                              const float* __restrict__ geom, int cubic,
                                              float theta) {
#pragma clang fp contract(off)
  if (!(cm.w > 0.f)) return -1.f;
  const float E = geom[6 + kMaxLevel + 1];
  const uint32_t q = code >> (30 - 3 * l);
  const float cmv[3] = {cm.x, cm.y, cm.z};
  float d2 = 0.f;
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    const float ext = cubic ? E : fmaxf(geom[3 + a] - geom[a], 1e-6f);
    const float h = ldexpf(ext, -l);
    const uint32_t idx = compact_bits(q >> (2 - a));
    const float ctr = geom[a] + ((float)idx + 0.5f) * h;
    const float d = cmv[a] - ctr;
    d2 = a == 0 ? d * d : d2 + d * d;
  }
  const float rc = ldexpf(E, -l) / theta + sqrtf(d2);
  return rc * rc;
}

// One thread per node: its centre of mass from the prefix, its opening radius,
// its span (count << 4 | level), and the wave ranges of the children
// of nodes holding more than kWaveBodies bodies, in records of one or two: one
// atomic per wave reserves the records of all its lanes.
__global__ __launch_bounds__(256) void k_tree_com(nb_node* __restrict__ nodes,
                                                  const int* __restrict__ node_end, int n,
                                                  int64_t max_nodes,
                                                  const int* __restrict__ level_off,
                                                  const double4* __restrict__ prefix,
                                                  const float4* __restrict__ pms,
                                                  const uint32_t* __restrict__ codes,
                                                  const float* __restrict__ geom, int cubic,
                                                  float theta, int leaf, int pairs,
                                                  int4* __restrict__ waves,
                                                  int* __restrict__ wctl) {
  const int total = (int)min((int64_t)level_off[kMaxLevel + 1], max_nodes);
  const int lane = threadIdx.x & 63;
  // Rounds are uniform across the block, so every lane of a wave reaches the
  // wave-wide record reservation.
  for (int k0 = blockIdx.x * 256; k0 < total; k0 += gridDim.x * 256) {
    const int k = k0 + threadIdx.x;
    int starts[8], ends[8], nc = 0, nrec = 0, l = 0;
    if (k < total) {
      const int first = nodes[k].first, start = nodes[k].start;
      l = nodes[k].span & 15;
      const int end = node_end[k], cnt = end - start;
      nb_node nd{make_float4(0.f, 0.f, 0.f, 0.f), -1.f, first, start, cnt << 4 | l};
      if (start < 0 || cnt < 1 || end > n) {
        nodes[k].com = nd.com;
        nodes[k].r2 = nd.r2;
        nodes[k].span = nd.span;
      } else {
        if (cnt == 1) {
          nd.com = pms[start];
        } else {
          const double4 a = prefix[start], b = prefix[end];
          const double m = b.x - a.x;
          const double inv = m > 0.0 ? 1.0 / m : 0.0;
          nd.com = make_float4((float)((b.y - a.y) * inv), (float)((b.z - a.z) * inv),
                               (float)((b.w - a.w) * inv), (float)m);
        }
        nd.r2 = open_radius2(nd.com, codes[start], l, geom, cubic, theta);
        // the other threads read `first` and `start` only, which stay as they are
        nodes[k].com = nd.com;
        nodes[k].r2 = nd.r2;
        nodes[k].span = nd.span;
        if (cnt > kWaveBodies && first >= 0 && l < kMaxLevel) {
          // the children are consecutive nodes of the next level and tile the range
          const int last = min(level_off[l + 2], total);
          int s[8];  // eight independent loads; past the last child: >= end
#pragma unroll
          for (int q = 0; q < 8; ++q)
            s[q] = first + q < last ? nodes[first + q].start : end;
#pragma unroll
          for (int q = 0; q < 8; ++q)
            if (s[q] < end) {
              starts[q] = s[q];
              ends[q] = q < 7 ? min(s[q < 7 ? q + 1 : 7], end) : end;
              nc = q + 1;
            }
          nrec = count_records(starts, ends, nc, l, leaf, pairs);
        }
      }
    }
    const int incl = wave_incl_scan(nrec);
    const int all = __shfl(incl, 63);
    int wbase = 0;
    if (lane == 63 && all > 0) wbase = atomicAdd(&wctl[0], all);
    wbase = __shfl(wbase, 63);
    if (nrec > 0) emit_records(waves, wbase + incl - nrec, n, starts, ends, nc, l, leaf, pairs);
  }
}

// ---- 8. traversal ---------------------------------------------------------------------------
// kModified: open with the default traversal's radius (r2 < d^2) instead of
// the reference's test; used only to count what that test needs per body.
template <bool kCount, bool kModified = false>
__global__ __launch_bounds__(256) void k_traverse(const float4* __restrict__ pms,
                                                  const uint32_t* __restrict__ perm, int n,
                                                  const nb_node* __restrict__ nodes,
                                                  const int* __restrict__ next,
                                                  const int* __restrict__ level_off,
                                                  int64_t max_nodes,
                                                  const float* __restrict__ geom, float theta2,
                                                  float eps2, double G,
                                                  double* __restrict__ force,
                                                  unsigned long long* __restrict__ inter,
                                                  int* __restrict__ flags) {
  __shared__ float side2[kMaxLevel + 1];
  if (threadIdx.x <= kMaxLevel) side2[threadIdx.x] = geom[6 + threadIdx.x];
  __syncthreads();
  const int t = blockIdx.x * 256 + threadIdx.x;
  // A rope walk visits each node at most once; the bound and the index check
  // turn a corrupt tree into an error flag instead of a hang or a fault.
  const int total = (int)min((int64_t)level_off[kMaxLevel + 1], max_nodes);
  unsigned long long cnt = 0;
  if (t < n) {
    const float4 me = pms[t];
    float ax = 0.f, ay = 0.f, az = 0.f;
    int i = 0;
    for (int it = 0; i >= 0; ++it) {
      if (i >= total || it > total) {
        atomicOr(flags, 4);
        break;
      }
      const nb_node nd = nodes[i];
      const float4 c = nd.com;
      const float dx = c.x - me.x, dy = c.y - me.y, dz = c.z - me.z;
      const float d2 = fmaf(dz, dz, fmaf(dy, dy, dx * dx));
      if (kModified ? nd.r2 < d2 : side2[span_level(nd.span)] < theta2 * d2) {
        if (c.w > 0.f && d2 > 0.f) {
          const float inv = __builtin_amdgcn_rsqf(d2 + eps2);
          const float s = (c.w * inv) * (inv * inv);
          ax = fmaf(dx, s, ax);
          ay = fmaf(dy, s, ay);
          az = fmaf(dz, s, az);
          if (kCount) ++cnt;
        }
        i = next[i];
      } else if (nd.first < 0) {
        const int e = min(nd.start + span_count(nd.span), n);
        for (int b = max(nd.start, 0); b < e; ++b) {
          const float4 q = pms[b];
          const float bx = q.x - me.x, by = q.y - me.y, bz = q.z - me.z;
          const float b2 = fmaf(bz, bz, fmaf(by, by, bx * bx));
          if (b2 > 0.f) {
            const float inv = __builtin_amdgcn_rsqf(b2 + eps2);
            const float s = (q.w * inv) * (inv * inv);
            ax = fmaf(bx, s, ax);
            ay = fmaf(by, s, ay);
            az = fmaf(bz, s, az);
            if (kCount) ++cnt;
          }
        }
        i = next[i];
      } else {
        i = nd.first;
      }
    }
    const uint32_t o = perm[t];
    if (!kModified && o < (uint32_t)n) {
      force[o] = G * (double)ax;
      force[n + o] = G * (double)ay;
      force[2 * n + o] = G * (double)az;
    }
  }
  if (kCount) {
    __shared__ unsigned long long red[256];
    red[threadIdx.x] = cnt;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
      if (threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
      __syncthreads();
    }
    if (threadIdx.x == 0) atomicAdd(inter, red[0]);
  }
}

// Wave traversal (the default). A wave takes one range of at most
// NB_BH_WAVE_BODIES Morton-consecutive bodies of one cell (emitted by the build)
// and its lanes share every decision: a cell is accepted for the whole range
// when its opening radius (side / theta + |COM - cell centre|) is less than
// dmin, the distance from its COM to the range's bounding box; otherwise it is
// opened, and a leaf that is not accepted is evaluated body by body by every
// lane. Per body this accepts a subset of what the per-body test accepts (at
// least as accurate), and nothing diverges. For latency, each wave keeps a
// stack of opened nodes in LDS as (first child, level of the children << 27 |
// end of the body range). One iteration pops up to 8 of them and lets 8 lanes
// per node examine its (at most 8) children at once, so one memory round trip
// covers 64 nodes. The walk only appends indices to an interaction list in LDS
// (accepted cells, flagged, and the bodies of unaccepted leaves) and pushes
// opened children; no source data is read while walking. Whenever the list
// fills up, and at the end, the wave gathers the sources 64 at a time into LDS
// and streams them through the direct-sum inner loop (LDS broadcast reads, 13
// VALU per interaction). From NB_BH_PAIR_MIN_BODIES bodies on (or with
// NB_F_BH_PAIRS) the build pairs sibling ranges of equal copy width: such a
// pair walks once for both ranges and leaves to each range only the cells the
// two decide differently (walk() below), which on the 4M two-disc system takes
// 30% fewer walk iterations and stages 34% fewer sources for exactly the same
// interactions.
constexpr int kListWaves = 4;
// LDS (26.7 KB per block) and 80 VGPRs allow six blocks per CU. A 384-entry
// list (instead of 512) is what makes the sixth fit; it measured about 1% faster
// on the two-disc 4M system.
constexpr int kListBlocksPerCU = 6;
// The deepest stack seen on the two-disc 4M system (400 sampled ranges, leaf 8)
// is 73 entries. A pair's deferred entries share the region from its top: a CPU
// replay of the pair walk on 4M-body two-disc, Plummer and uniform-ball systems
// (leaf 1) needs at most 245 stack plus deferred entries. Overflow is detected
// and reported (NB_E_TREE_OVERFLOW).
constexpr int kStackCap = 512;
constexpr int kListCap = 384;                 // source indices per wave
constexpr uint32_t kCellBit = 0x80000000u;    // list entry refers to a cell, not a body

// Stream the list through the direct-sum inner loop: 64 entries at a time,
// each lane gathers one source (cell COM or body) into the LDS staging area,
// then the lanes read the staged sources by broadcast. The bodies of a range are
// held S = 64 / P times (P = its body count rounded up to a power of two, at
// least 4; S = 1 above 32 bodies): the lanes of slice s = lane / P take the
// staged entries s, s + S, s + 2S, ..., so every lane does useful work, and the
// slices' partial sums are added at the end of the range. Entries are staged
// slice-major (entry j at (j % S) * (64 / S) + j / S), so a slice reads its
// entries from consecutive addresses: four reads per step share one base
// address with immediate offsets, and the trip count is wave-uniform.
// Compensated accumulation: each flush sums its (at most kListCap / 2 per lane
// at two slices) terms in plain FP32 and folds the partial sums into the
// running (sum, error) pairs with TwoSum, as the direct sum folds every 256
// sources.
template <bool kCount, bool kGuard>
__device__ __forceinline__ void list_flush(const uint32_t* list, int lc, float4* stage, int lane,
                                           int slice, int log2S, const float4* __restrict__ pms,
                                           const nb_node* __restrict__ nodes, float4 me, float eps2_s,
                                           float& sx, float& sy, float& sz, float& cx, float& cy,
                                           float& cz, unsigned long long& cnt) {
  float ax = 0.f, ay = 0.f, az = 0.f;
  float eps2 = eps2_s;  // a VGPR copy: all-VGPR operand forms issue faster
  asm volatile("" : "+v"(eps2));
  const int S = 1 << log2S;
  const int per = 64 >> log2S;  // entries per slice
  const int put = (lane & (S - 1)) * per + (lane >> log2S);  // slice-major slot of entry `lane`
  const float4* mine = stage + slice * per;
  // lane's source of the chunk starting at e (a far-away pad past the list)
  auto gather = [&](int e) {
    float4 g = nbcore::far_pad();
    if (e + lane < lc) {
      const uint32_t id = list[e + lane];
      g = (id & kCellBit) ? nodes[id & ~kCellBit].com : pms[id];
    }
    return g;
  };
  float4 q = gather(0);
  for (int e = 0; e < lc; e += 64) {
    const int m = min(64, lc - e);
    stage[put] = q;
    __builtin_amdgcn_wave_barrier();
    // the next chunk's gather is in flight while this chunk is evaluated
    if (e + 64 < lc) q = gather(e + 64);
    // T = ceil(m / S) rounded up to 4 entries per slice; S <= 16 divides 64, so
    // 64 / S is a multiple of 4 and T <= 64 / S: every read stays inside this
    // slice's block; entries at or past m are far-away pads.
    const int T = __builtin_amdgcn_readfirstlane((((m + S - 1) >> log2S) + 3) & ~3);
    for (int t = 0; t < T; t += 4) {
      float dx[4], dy[4], dz[4], r2[4], inv[4], w[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const float4 src = mine[t + u];  // few distinct addresses: LDS broadcast
        w[u] = src.w;
        dx[u] = src.x - me.x, dy[u] = src.y - me.y, dz[u] = src.z - me.z;
        r2[u] = fmaf(dz[u], dz[u], fmaf(dy[u], dy[u], fmaf(dx[u], dx[u], eps2)));
      }
      nbcore::rsq_group(r2, inv);
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        float s = (w[u] * inv[u]) * (inv[u] * inv[u]);
        if (kGuard) s = r2[u] > 0.f ? s : 0.f;
        ax = fmaf(dx[u], s, ax);
        ay = fmaf(dy[u], s, ay);
        az = fmaf(dz[u], s, az);
        if (kCount)
          cnt += (w[u] > 0.f && fmaf(dz[u], dz[u], fmaf(dy[u], dy[u], dx[u] * dx[u])) > 0.f) ? 1 : 0;
      }
    }
    __builtin_amdgcn_wave_barrier();
  }
  nbcore::two_sum_fold(sx, cx, ax);
  nbcore::two_sum_fold(sy, cy, ay);
  nbcore::two_sum_fold(sz, cz, az);
}

// The lanes whose b is true; __ballot takes an int and would make one of b first.
__device__ __forceinline__ uint64_t lanes_where(bool b) { return __builtin_amdgcn_ballot_w64(b); }

// Bits of m below this lane.
__device__ __forceinline__ int bits_below(uint64_t m) {
  return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0));
}

// A stack entry: the children of an opened node.
__device__ __forceinline__ int2 stack_entry(int first, int level, int body_end) {
  return make_int2(first, (int)(((uint32_t)level << 27) | (uint32_t)body_end));
}

// Child slot ci (0..7) of entry e: true where the slot holds a child, whose index and
// record are then in child and cl. The nodes from the entry's first on are its children
// as long as they are of the children's level (the last parent of a level is followed by
// the next level) and start before the parent's end. A lane without a candidate reads
// the root's record: no lane is masked off, and the record needs no initial value.
// With the entry read in one piece, nothing looked up per level and nothing held in
// scratch memory a walk's iteration is about a quarter shorter (traversal of 2^22
// bodies 4,672 us, now 4,385).
__device__ __forceinline__ bool child_at(int2 e, int ci, bool have, int total,
                                         const nb_node* __restrict__ nodes, int& child, nb_node& cl) {
  const int cand = e.x + ci;
  const bool ok = have && (uint32_t)cand < (uint32_t)total;
  child = ok ? cand : 0;
  cl = nodes[child];
  const uint32_t w = (uint32_t)e.y;
  return ok && cl.start < (int)(w & ((1u << 27) - 1)) && span_level(cl.span) == (int)(w >> 27);
}

// Append the bodies of the leaves that the lanes hold (in lane order) to a list of
// kCap entries. A prefix sum places each lane's bodies, which it writes itself: at
// most leaf_size rounds for all of them. One round per leaf, the lanes together, was a
// chain of scalar waits that near ranges paid for a dozen leaves per iteration (20,011
// bodies: traversal 120 us, now 73; 65,536 199, now 162). Leaves that do not fit
// together go one by one, 64 bodies at a time.
template <int kCap, typename Flush>
__device__ __forceinline__ void list_leaves(uint32_t* list, int& lc, int lane, bool leaf, int start,
                                            int count, int n, Flush flush) {
  uint64_t bl = lanes_where(leaf);
  if (bl == 0) return;
  const int mine = leaf ? count : 0;
  const int incl = wave_incl_scan(mine);
  const int total = __builtin_amdgcn_readlane(incl, 63);
  if (total <= kCap) {
    if (lc + total > kCap) flush();
    uint32_t* at = list + lc + incl - mine;
    for (int k = 0; lanes_where(k < mine); ++k)
      if (k < mine) at[k] = (uint32_t)min(start + k, n - 1);
    lc += total;
    return;
  }
  while (bl) {
    const int src = __ffsll((unsigned long long)bl) - 1;
    bl &= bl - 1;
    const int ls = __builtin_amdgcn_readlane(start, src);
    const int lcount = __builtin_amdgcn_readlane(count, src);
    for (int off = 0; off < lcount; off += 64) {
      const int m = min(64, lcount - off);
      if (lc + 64 > kCap) flush();
      if (lane < m) list[lc + lane] = (uint32_t)min(ls + off + lane, n - 1);
      lc += m;
    }
  }
}

// Shared LDS of one traversing wave. The stack region holds the walk's stack
// from the bottom and a pair's deferred entries from the top.
struct WaveLds {
  int2* stack;
  uint32_t* list;
  float4* stage;
  int cap;             // entries of the stack region in use (<= kStackCap)
};

// An axis-aligned box held in scalar registers (wave-uniform).
struct Box {
  float lx, ly, lz, hx, hy, hz;
};

// Squared distance from c to the box (0 inside).
__device__ __forceinline__ float box_dist2(const Box& b, const float4& c) {
  const float ex = fmaxf(fmaxf(b.lx - c.x, c.x - b.hx), 0.f);
  const float ey = fmaxf(fmaxf(b.ly - c.y, c.y - b.hy), 0.f);
  const float ez = fmaxf(fmaxf(b.lz - c.z, c.z - b.hz), 0.f);
  return fmaf(ez, ez, fmaf(ey, ey, ex * ex));
}

// Walk the tree for the bodies held by the wave's lanes and accumulate their
// accelerations (lanes of slice s take staged entries s, s + S, ...).
//   kShared: the shared walk of a pair of ranges with boxes A and B. A cell
//     both accept is evaluated for both ranges; a cell exactly one accepts is
//     deferred: its (first sibling, 8-bit sibling mask) entry goes to the top of
//     the stack region and nd counts them. Cells neither accepts are opened (or,
//     as leaves, evaluated body by body) for both.
//   otherwise: the walk of one range with box U, from the root when nd == 0,
//     else from the nd deferred entries (read, not consumed: the pair's other
//     range walks them too).
// For each range this examines and evaluates exactly the cells its own walk
// from the root would: the shared walk only descends where both ranges open,
// and a deferred cell is decided by each range's own test.
template <bool kCount, bool kGuard, bool kShared>
__device__ void walk(const WaveLds& L, int lane, int slice, int log2S, float4 me, int n,
                     const float4* __restrict__ pms, const nb_node* __restrict__ nodes, int total,
                     float eps2, int* __restrict__ flags, const Box& U, const Box& A, const Box& B, int& nd,
                     float& ax, float& ay, float& az, float& cx, float& cy, float& cz,
                     unsigned long long& cnt) {
  int2* stack = L.stack;
  uint32_t* list = L.list;
#define NB_FLUSH()                                                                              \
  do {                                                                                          \
    list_flush<kCount, kGuard>(list, lc, L.stage, lane, slice, log2S, pms, nodes, me, eps2, ax, ay, \
                               az, cx, cy, cz, cnt);                                           \
    lc = 0;                                                                                     \
  } while (0)
  int sp = 0, lc = 0, dpos = 0;
  if (kShared || nd == 0) {
    // a virtual parent whose only child is the root
    if (lane == 0) stack[0] = stack_entry(0, 0, n);
    sp = 1;
    __builtin_amdgcn_wave_barrier();
  }
  int left = total;  // iterations: every node is examined at most once
  for (; left >= 0 && (sp > 0 || (!kShared && dpos < nd)); --left) {
    // room for this iteration's accepted cells (at most 64), flushed while
    // nothing of the iteration is live
    if (lc + 64 > kListCap) NB_FLUSH();
    // opaque per iteration: what follows from the lane is computed where it is used
    // instead of being held, and then spilled, over the whole walk
    asm volatile("" : "+v"(lane));
    const int q = lane >> 3, ci = lane & 7;
    int child, efirst = 0;
    nb_node cl;
    bool valid;
    if (!kShared && sp < 8 && dpos < nd) {
      // deferred entries: up to 32 of them, at most 64 cells, listed in the
      // staging area (free while walking) so that lane j takes the j-th cell
      int2 d = make_int2(0, 0);
      const bool have = lane < 32 && dpos + lane < nd;
      if (have) d = stack[L.cap - 1 - (dpos + lane)];
      const int pc = __popc((uint32_t)d.y);
      const int incl = wave_incl_scan(pc);
      const bool fits = have && incl <= 64;
      const int kd = __popcll(lanes_where(fits));  // >= 1: one entry has at most 8 cells
      int* cells = reinterpret_cast<int*>(L.stage);
      if (fits) {
        int o = incl - pc;
        for (uint32_t mm = (uint32_t)d.y; mm; mm &= mm - 1) cells[o++] = d.x + __ffs(mm) - 1;
      }
      __builtin_amdgcn_wave_barrier();
      valid = lane < __builtin_amdgcn_readlane(incl, kd - 1);
      child = valid ? cells[lane] : 0;
      cl = nodes[child];
      __builtin_amdgcn_wave_barrier();
      dpos += kd;
    } else {
      const int k = min(sp, 8);
      sp -= k;
      const int2 e = stack[sp + min(q, k - 1)];
      efirst = e.x;
      valid = child_at(e, ci, q < k, total, nodes, child, cl);
      __builtin_amdgcn_wave_barrier();
    }
    // the group's modified test (see open_radius2); a pair shares what both accept
    bool accept, defer = false;
    if (kShared) {
      const bool a = cl.r2 < box_dist2(A, cl.com), b = cl.r2 < box_dist2(B, cl.com);
      accept = valid && a && b;
      defer = valid && a != b;
    } else {
      accept = valid && cl.r2 < box_dist2(U, cl.com);
    }
    const bool rest = valid && !accept && !defer;
    const bool leaf = rest && cl.first < 0, open = rest && cl.first >= 0;
    // accepted cells with mass -> list
    const bool acc = accept && cl.com.w > 0.f;
    const uint64_t ba = lanes_where(acc);
    if (acc) list[lc + bits_below(ba)] = (uint32_t)child | kCellBit;
    lc += __popcll(ba);
    // deferred cells -> one entry per stack entry that has any
    int nd_add = 0;
    bool head = false;
    uint32_t dmask = 0;
    uint64_t bg = 0;
    if (kShared) {
      const uint64_t bd = lanes_where(defer);
      if (bd) {
        const uint32_t half = q < 4 ? (uint32_t)bd : (uint32_t)(bd >> 32);
        dmask = (half >> (lane & 24)) & 0xffu;  // bits 8q .. 8q + 7
        head = ci == 0 && dmask != 0;
        bg = lanes_where(head);
        nd_add = __popcll(bg);
      }
    }
    // opened cells -> stack
    const uint64_t bo = lanes_where(open);
    const int opened = __popcll(bo);
    if (sp + opened + nd + nd_add > L.cap) {  // reported; nothing more is walked
      if (lane == 0) atomicOr(flags, 8);
      sp = 0;
      dpos = nd;
    } else {
      if (kShared && head) stack[L.cap - 1 - (nd + bits_below(bg))] = make_int2(efirst, (int)dmask);
      nd += nd_add;
      if (open)
        stack[sp + bits_below(bo)] =
            stack_entry(cl.first, span_level(cl.span) + 1, cl.start + span_count(cl.span));
      sp += opened;
    }
    // leaves that are not accepted -> the indices of their bodies
    list_leaves<kListCap>(list, lc, lane, leaf, cl.start, span_count(cl.span), n,
                          [&] { NB_FLUSH(); });
    __builtin_amdgcn_wave_barrier();
  }
  if (left < 0 && lane == 0) atomicOr(flags, 4);
  NB_FLUSH();
#undef NB_FLUSH
}

// The bounding box of the bodies held by the lanes, reduced over every lane bit
// except `keep` (0: over all lanes; else each half of the lanes split by that
// bit gets its own box), then read from lanes `from0` and `from1`.
__device__ __forceinline__ void lane_boxes(float4 me, int keep, int from0, int from1, Box& b0,
                                           Box& b1) {
  float lx = me.x, ly = me.y, lz = me.z, hx = me.x, hy = me.y, hz = me.z;
  // lanes lane ^ off: ds_swizzle's bit mode inside each half of the wave, one
  // ds_bpermute across the halves
  auto step = [&](auto xor_lanes) {
    lx = fminf(lx, xor_lanes(lx));
    ly = fminf(ly, xor_lanes(ly));
    lz = fminf(lz, xor_lanes(lz));
    hx = fmaxf(hx, xor_lanes(hx));
    hy = fmaxf(hy, xor_lanes(hy));
    hz = fmaxf(hz, xor_lanes(hz));
  };
  auto swz = [](auto off_c) {
    return [](float v) {
      constexpr int kPattern = (decltype(off_c)::value << 10) | 0x1f;  // xor, or 0, and 0x1f
      return __int_as_float(__builtin_amdgcn_ds_swizzle(__float_as_int(v), kPattern));
    };
  };
  if (keep != 32) step([](float v) { return __shfl_xor(v, 32); });
  if (keep != 16) step(swz(std::integral_constant<int, 16>{}));
  if (keep != 8) step(swz(std::integral_constant<int, 8>{}));
  if (keep != 4) step(swz(std::integral_constant<int, 4>{}));
  if (keep != 2) step(swz(std::integral_constant<int, 2>{}));
  if (keep != 1) step(swz(std::integral_constant<int, 1>{}));
  // uniform over each group: keep the boxes in scalar registers
  auto at = [](float v, int l) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
  };
  b0 = Box{at(lx, from0), at(ly, from0), at(lz, from0), at(hx, from0), at(hy, from0), at(hz, from0)};
  b1 = Box{at(lx, from1), at(ly, from1), at(lz, from1), at(hx, from1), at(hy, from1), at(hz, from1)};
}

// Persistent: every wave takes records from a ticket until none is left, so the
// cost of uneven ranges balances dynamically. Its first record it has from its
// own number: that many tickets at once are that many atomics on one address, about
// 10 ns each, so the last of 6,144 waves began 60 us after the first (traversal of
// 2^22 bodies 4,385 us, now 4,229; with workgroups as below 65,536 bodies 147, now
// 132, 20,011 68, now 61). A record is one wave range or a
// pair of sibling ranges (x, y) and (z, w), w > 0. A pair first walks once for
// both (its lanes: [slice][range][slot], P1 lanes per copy of a range), then,
// if cells were deferred, each range walks them with its own lanes ([slice][slot]);
// each body's force is the sum of the two parts in FP64, in that order. The
// counting variant (diagnostics only) needs more registers and is allowed five
// blocks per CU; its surplus blocks start when others retire.
template <bool kCount, bool kGuard>
__global__ __launch_bounds__(64 * kListWaves, kCount ? 5 : kListBlocksPerCU) void k_traverse_list(
    const float4* __restrict__ pms, const uint32_t* __restrict__ perm, int n,
    const nb_node* __restrict__ nodes, const int* __restrict__ level_off, int64_t max_nodes,
    float eps2, double G, double* __restrict__ force,
    unsigned long long* __restrict__ inter, int* __restrict__ flags,
    const int4* __restrict__ waves, int* __restrict__ wctl, const int* __restrict__ order,
    float* __restrict__ cost, int stack_cap) {
  __shared__ int2 s_stack[kListWaves][kStackCap];
  __shared__ uint32_t s_list[kListWaves][kListCap];
  __shared__ float4 s_stage[kListWaves][64];
  const int total = (int)min((int64_t)level_off[kMaxLevel + 1], max_nodes);
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const WaveLds L{s_stack[wave], s_list[wave], s_stage[wave],
                  stack_cap > 0 && stack_cap < kStackCap ? stack_cap : kStackCap};
  const int nrec = min(wctl[0], n);
  unsigned long long cnt = 0;
  const int static_recs = gridDim.x * kListWaves;
  for (int w = wave * gridDim.x + blockIdx.x; w < nrec;) {
    const uint64_t t_start = wall_clock64();
    const int ri = order ? order[w] : w;
    const int4 rec = waves[(unsigned)ri < (unsigned)nrec ? ri : w];  // wave-uniform: scalar registers
    const bool pair = rec.w > 0;
    // shared walk: a single range is held 64 / P1 times, a pair 32 / P1 times
    const int P1 = copy_lanes(pair ? max(rec.y, rec.w) : rec.y);
    const int grp = pair ? 2 * P1 : P1;
    const int slot = lane & (P1 - 1);
    const bool second = pair && (lane & P1);
    const int rs = second ? rec.z : rec.x, rn = second ? rec.w : rec.y;
    const bool valid = slot < rn;
    const int t = min(rs + (valid ? slot : 0), n - 1);  // lanes past a range copy its first body
    const float4 me = pms[t];
    const int log2S = 6 - (31 - __clz(grp)), slice = lane / grp;
    Box A, B;
    lane_boxes(me, pair ? P1 : 0, 0, pair ? P1 : 0, A, B);
    float ax = 0.f, ay = 0.f, az = 0.f, cx = 0.f, cy = 0.f, cz = 0.f;
    unsigned long long c = 0;
    int nd = 0;
    if (pair)
      walk<kCount, kGuard, true>(L, lane, slice, log2S, me, n, pms, nodes, total, eps2, flags,
                                 A, A, B, nd, ax, ay, az, cx, cy, cz, c);
    else
      walk<kCount, kGuard, false>(L, lane, slice, log2S, me, n, pms, nodes, total, eps2, flags,
                                  A, A, B, nd, ax, ay, az, cx, cy, cz, c);
    // each slice's compensated sum in FP64, then the slices added (butterfly
    // over the slice bits, fixed order)
    double fx = (double)ax + (double)cx, fy = (double)ay + (double)cy,
           fz = (double)az + (double)cz;
    for (int off = grp; off < 64; off <<= 1) {
      fx += __shfl_xor(fx, off);
      fy += __shfl_xor(fy, off);
      fz += __shfl_xor(fz, off);
    }
    if (valid) cnt += c;
    if (nd == 0) {
      if (valid && lane < grp) {
        const uint32_t o = perm[t];
        if (o < (uint32_t)n) {
          force[o] = G * fx;
          force[n + o] = G * fy;
          force[2 * n + o] = G * fz;
        }
      }
    }
    // the deferred cells, range by range
    for (int h = 0; h < (nd > 0 ? 2 : 0); ++h) {
      const int hs = h ? rec.z : rec.x, hn = h ? rec.w : rec.y;
      const int P = copy_lanes(hn);
      const int s2 = lane & (P - 1);
      const bool v2 = s2 < hn;
      const int t2 = min(hs + (v2 ? s2 : 0), n - 1);
      const float4 me2 = pms[t2];
      ax = ay = az = cx = cy = cz = 0.f;
      c = 0;
      walk<kCount, kGuard, false>(L, lane, lane / P, 6 - (31 - __clz(P)), me2, n, pms, nodes,
                                  total, eps2, flags, h ? B : A, A, B, nd, ax, ay, az, cx, cy, cz, c);
      double gx = (double)ax + (double)cx, gy = (double)ay + (double)cy,
             gz = (double)az + (double)cz;
      for (int off = P; off < 64; off <<= 1) {
        gx += __shfl_xor(gx, off);
        gy += __shfl_xor(gy, off);
        gz += __shfl_xor(gz, off);
      }
      // the shared part of body s2 of range h sits in lane h * P1 + s2
      const double px = __shfl(fx, h * P1 + s2), py = __shfl(fy, h * P1 + s2),
                   pz = __shfl(fz, h * P1 + s2);
      if (v2) cnt += c;
      if (v2 && lane < P) {
        const uint32_t o = perm[t2];
        if (o < (uint32_t)n) {
          force[o] = G * (px + gx);
          force[n + o] = G * (py + gy);
          force[2 * n + o] = G * (pz + gz);
        }
      }
    }
    // the record's device time, shared out over its bodies for the next pass's order
    const float share = (float)(wall_clock64() - t_start) / (float)(rec.y + rec.w);
    if (cost && valid && lane < grp) {
      const uint32_t o = perm[t];
      if (o < (uint32_t)n) cost[o] = share;
    }
    if (nrec <= static_recs) break;
    if (lane == 0) w = static_recs + atomicAdd(&wctl[1], 1);
    w = __builtin_amdgcn_readfirstlane(w);
  }
  if (kCount) {
    __shared__ unsigned long long red[64 * kListWaves];
    red[threadIdx.x] = cnt;
    __syncthreads();
    for (int s = 64 * kListWaves / 2; s > 0; s >>= 1) {
      if (threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
      __syncthreads();
    }
    if (threadIdx.x == 0) atomicAdd(inter, red[0]);
  }
}

// ---- 8b. one workgroup per range ------------------------------------------------------
// The walk of one range by kWaves waves: what k_traverse_list does with one wave,
// for systems with fewer ranges than the chip has waves, whose pass lasts as long
// as its slowest walk (a range of far-out bodies in a large cell opens most of the
// tree). The waves share the stack: an iteration pops up to 8 * kWaves nodes,
// eight per wave, and every wave lists what it accepts in its own list. Opened
// children go back in wave and lane order, so the stack's content, the lists and
// with them every sum are the same in each run. A wave's list is summed when any
// wave's is full, at the same point for all, so that no wave waits at a barrier
// for another's arithmetic.
// Stack bound: its entries' levels never decrease from bottom to top (children
// are pushed in the order of their parents), and nodes of level l are pushed only
// when all entries of that level or deeper are popped in the same iteration, so at
// most 64 * kWaves entries of each of the levels 1 to 10 are ever held, and a
// level that has a deeper one above it has lost 8 * kWaves of them:
// (9 * 56 + 64) * kWaves entries.
constexpr int block_stack(int waves) { return (9 * 56 + 64) * waves; }
constexpr int kBlockListCap = 256;  // source indices per wave
// Waves per range by the system's size. Measured Barnes-Hut steps in us (Plummer
// sphere / uniform ball, leaf size 8), one (k_traverse_list), four and eight waves:
//     4,000 bodies  148/121  103/ 88   96/ 81
//    20,011         223/145  133/107  122/106
//    30,011         267/158  154/120  146/119
//    40,000         209/174  159/129  165/132
//    65,536         255/180  205/158  220/174
//   131,072         339/260  312/244  340/277
//   200,000         415/319  412/312  470/370
//   300,007         547/423  575/434  672/544
//   524,288         823/580  931/677
// Two gained 2% over four and one in a narrow band below the upper line. Above it
// there are enough ranges for every wave and the barriers only cost.
constexpr int kBlock8Bodies = 1 << 15;    // below: eight waves per range
constexpr int kBlockMaxBodies = 1 << 18;  // below: four; from here on k_traverse_list
constexpr int kBlockWavesPerCU = 24;      // by LDS and 80 VGPRs, as k_traverse_list

template <bool kGuard, int kWaves>
__global__ __launch_bounds__(64 * kWaves, kBlockWavesPerCU / 4) void k_traverse_block(
    const float4* __restrict__ pms, const uint32_t* __restrict__ perm, int n,
    const nb_node* __restrict__ nodes, const int* __restrict__ level_off, int64_t max_nodes,
    float eps2, double G, double* __restrict__ force, int* __restrict__ flags,
    const int4* __restrict__ waves, int* __restrict__ wctl, const int* __restrict__ order,
    float* __restrict__ cost, int stack_cap) {
  __shared__ int2 stack[block_stack(kWaves)];
  __shared__ uint32_t s_list[kWaves][kBlockListCap];
  __shared__ float4 s_stage[kWaves][64];
  __shared__ int2 s_cnt[kWaves];  // (opened children, list length) of each wave
  __shared__ int s_rec;
  static_assert(sizeof(s_stage[0]) >= 3 * kWaveBodies * sizeof(double), "a wave's sums fit its stage");
  const int total = (int)min((int64_t)level_off[kMaxLevel + 1], max_nodes);
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  uint32_t* list = s_list[wave];
  float4* stage = s_stage[wave];
  const int cap = stack_cap > 0 && stack_cap < block_stack(kWaves) ? stack_cap : block_stack(kWaves);
  const int nrec = min(wctl[0], n);
  unsigned long long unused = 0;
  for (int w = blockIdx.x; w < nrec;) {
    const uint64_t t_start = wall_clock64();
    const int ri = order ? order[w] : w;
    const int4 rec = waves[(unsigned)ri < (unsigned)nrec ? ri : w];
    const int P = copy_lanes(rec.y);
    const int log2S = 6 - (31 - __clz(P)), slice = lane / P, slot = lane & (P - 1);
    const bool valid = slot < rec.y;
    const int t = min(rec.x + (valid ? slot : 0), n - 1);  // lanes past the range copy its first body
    const float4 me = pms[t];
    Box A, B;
    lane_boxes(me, 0, 0, 0, A, B);
    float ax = 0.f, ay = 0.f, az = 0.f, cx = 0.f, cy = 0.f, cz = 0.f;
    int lc = 0, sp = 1;
    // the walk, a chain of loads, goes before other waves' arithmetic
    auto flush = [&]() {
      __builtin_amdgcn_s_setprio(0);
      list_flush<false, kGuard>(list, lc, stage, lane, slice, log2S, pms, nodes, me, eps2, ax, ay, az,
                                cx, cy, cz, unused);
      __builtin_amdgcn_s_setprio(1);
      lc = 0;
    };
    __builtin_amdgcn_s_setprio(1);
    // a virtual parent whose only child is the root
    if (threadIdx.x == 0) stack[0] = stack_entry(0, 0, n);
    __syncthreads();
    for (int iter = 0; sp > 0; ++iter) {  // sp is the same in every wave
      if (iter > total) {  // every node is examined at most once
        if (threadIdx.x == 0) atomicOr(flags, 4);
        break;
      }
      const int k = min(sp, 8 * kWaves);
      sp -= k;
      const int q = 8 * wave + (lane >> 3), ci = lane & 7;
      int child;
      nb_node cl;
      const bool valid = child_at(stack[sp + min(q, k - 1)], ci, q < k, total, nodes, child, cl);
      const bool accept = valid && cl.r2 < box_dist2(A, cl.com);
      const bool rest = valid && !accept;
      const bool leaf = rest && cl.first < 0, open = rest && cl.first >= 0;
      const bool acc = accept && cl.com.w > 0.f;
      const uint64_t ba = lanes_where(acc);
      if (acc) list[lc + bits_below(ba)] = (uint32_t)child | kCellBit;
      lc += __popcll(ba);
      list_leaves<kBlockListCap>(list, lc, lane, leaf, cl.start, span_count(cl.span), n, flush);
      const uint64_t bo = lanes_where(open);
      if (lane == 0) s_cnt[wave] = make_int2(__popcll(bo), lc);
      __syncthreads();  // counts are in, and every wave has read its entries
      int before = 0, opened = 0, longest = 0;
#pragma unroll
      for (int v = 0; v < kWaves; ++v) {
        const int2 o = s_cnt[v];
        before += v < wave ? o.x : 0;
        opened += o.x;
        longest = max(longest, o.y);
      }
      opened = __builtin_amdgcn_readfirstlane(opened);
      if (sp + opened > cap) {  // the same in every wave
        if (threadIdx.x == 0) atomicOr(flags, 8);
        break;
      }
      if (open)
        stack[sp + before + bits_below(bo)] =
            stack_entry(cl.first, span_level(cl.span) + 1, cl.start + span_count(cl.span));
      sp += opened;
      // room for the next iteration's accepted cells (at most 64 per wave)
      if (__builtin_amdgcn_readfirstlane(longest) + 64 > kBlockListCap) flush();
      __syncthreads();
    }
    if (lc > 0) flush();
    // each slice's compensated sum in FP64, the slices added (butterfly over the
    // slice bits, fixed order), then the waves in order
    double f[3] = {(double)ax + (double)cx, (double)ay + (double)cy, (double)az + (double)cz};
    double* sums = reinterpret_cast<double*>(stage);
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      for (int off = P; off < 64; off <<= 1) f[a] += __shfl_xor(f[a], off);
      if (lane < P) sums[a * kWaveBodies + lane] = f[a];
    }
    __syncthreads();
    const uint32_t o = perm[t];
    if (wave == 0 && valid && lane < P && o < (uint32_t)n) {
      for (int a = 0; a < 3; ++a) {
        double all = f[a];
        for (int v = 1; v < kWaves; ++v)
          all += reinterpret_cast<const double*>(s_stage[v])[a * kWaveBodies + lane];
        force[(int64_t)a * n + o] = G * all;
      }
      // the range's device time, shared out over its bodies for the next pass's order
      if (cost) cost[o] = (float)(wall_clock64() - t_start) / (float)rec.y;
    }
    if (nrec <= (int)gridDim.x) break;
    if (threadIdx.x == 0) s_rec = gridDim.x + atomicAdd(&wctl[1], 1);
    __syncthreads();  // the waves' sums have been read, too
    w = __builtin_amdgcn_readfirstlane(s_rec);
  }
}

// ---- 8c. traversal order ---------------------------------------------------------------
// A persistent launch ends when its last wave finishes its last record, so the
// records are taken costliest first: each record's estimate is the device time
// its bodies' records took in the previous pass (stored per body, by original
// index, so it survives the rebuild), bucketed by half-octaves. Within a bucket
// the order is that of the atomics. The order changes only which wave takes a
// record and when; every record's arithmetic, and so every force, is the same.

// Half-octave of an estimate; anything not a finite value >= 1 (no history yet,
// or memory not written by a pass) goes last.
__device__ __forceinline__ int cost_bucket(float est) {
  if (!(est >= 1.f) || !(est <= FLT_MAX)) return 0;
  const uint32_t u = __float_as_uint(est);
  return min(kCostBuckets - 1, 2 * ((int)(u >> 23) - 127) + (int)((u >> 22) & 1));
}

// Records are handled in chunks of kOrderChunk by a grid of at most kOrderBlocks
// blocks; each block counts in LDS and makes one global atomic per bucket per
// chunk, so the few busy buckets see few atomics. (Bucketing a record where it is
// made, in k_tree_com, spares a launch of 4.7 us but its gathers made that kernel 7
// us longer at 65,536 bodies and 35 at 2^22.)
constexpr int kOrderChunk = 1024;
constexpr int kOrderBlocks = 256;
// Below this the ordering costs more than the tail it saves (Plummer steps with
// single ranges, ordered against not, when it took three launches: 0.577 against
// 0.583 ms at 65,536 bodies, 0.858 against 0.881 at 262,144, 1.267 against 1.296 at
// 524,288).
constexpr int kOrderMinBodies = 1 << 16;

__global__ __launch_bounds__(256) void k_rec_bucket(const int4* __restrict__ waves,
                                                    const int* __restrict__ wctl, int n,
                                                    const float* __restrict__ cost,
                                                    const uint32_t* __restrict__ perm,
                                                    int* __restrict__ bucket,
                                                    int* __restrict__ hist) {
  __shared__ int h[kCostBuckets];
  if (threadIdx.x < kCostBuckets) h[threadIdx.x] = 0;
  __syncthreads();
  const int nrec = min(wctl[0], n);
  for (int i = blockIdx.x * 256 + threadIdx.x; i < nrec; i += gridDim.x * 256) {
    const int4 r = waves[i];  // starts are sorted body indices < n
    float est = cost[perm[r.x]] * (float)r.y;
    if (r.w > 0) est += cost[perm[r.z]] * (float)r.w;
    const int b = cost_bucket(est);
    bucket[i] = b;
    atomicAdd(&h[b], 1);
  }
  __syncthreads();
  if (threadIdx.x < kCostBuckets && h[threadIdx.x] > 0) atomicAdd(&hist[threadIdx.x], h[threadIdx.x]);
}

// Tickets -> records: the first place of each bucket (the records in the buckets
// above, one wave's scan in every block) plus a place within it.
__global__ __launch_bounds__(256) void k_rec_scatter(const int* __restrict__ wctl, int n,
                                                     const int* __restrict__ bucket,
                                                     int* __restrict__ hist,
                                                     int* __restrict__ order) {
  __shared__ int h[kCostBuckets], base[kCostBuckets], first[kCostBuckets];
  constexpr int kPer = kOrderChunk / 256;
  static_assert(kCostBuckets == 64, "one wave scans the buckets");
  const int nrec = min(wctl[0], n);
  if (threadIdx.x < 64) {  // records in the buckets above
    const int b = kCostBuckets - 1 - threadIdx.x, v = hist[b];
    first[b] = wave_incl_scan(v) - v;
  }
  for (int c0 = blockIdx.x * kOrderChunk; c0 < nrec; c0 += gridDim.x * kOrderChunk) {
    if (threadIdx.x < kCostBuckets) h[threadIdx.x] = 0;
    __syncthreads();
    int bk[kPer], pos[kPer];
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
      const int i = c0 + k * 256 + threadIdx.x;
      bk[k] = i < nrec ? bucket[i] : -1;
      pos[k] = bk[k] >= 0 ? atomicAdd(&h[bk[k]], 1) : 0;
    }
    __syncthreads();
    if (threadIdx.x < kCostBuckets && h[threadIdx.x] > 0)
      base[threadIdx.x] =
          first[threadIdx.x] + atomicAdd(&hist[kCostBuckets + threadIdx.x], h[threadIdx.x]);
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
      const int at = bk[k] >= 0 ? base[bk[k]] + pos[k] : nrec;
      if (at < nrec) order[at] = c0 + k * 256 + threadIdx.x;
    }
    __syncthreads();
  }
}

__global__ void k_zero_u64(unsigned long long* p) {
  if (threadIdx.x == 0 && blockIdx.x == 0) *p = 0ull;
}

}  // namespace

void nb_bh_carve(nb_ctx* c, char* base, int upto) {
  nb_bh_state& b = c->bh;
  const nb_bh_layout L = nb_bh_layout_for(c->n);
  auto at = [&](int k) -> void* { return k < upto ? base + L.off[k] : nullptr; };
  b.bbox_part = (float*)at(kBhBbox);
  b.geom = (float*)at(kBhGeom);
  b.keys[0] = (uint32_t*)at(kBhKey0);
  b.keys[1] = (uint32_t*)at(kBhKey1);
  b.vals[0] = (uint32_t*)at(kBhVal0);
  b.vals[1] = (uint32_t*)at(kBhVal1);
  b.codes = (uint32_t*)at(kBhCodes);
  b.digit_hist = (int*)at(kBhHist);
  b.group_hist = (int*)at(kBhGroupHist);
  b.pms = (float4*)at(kBhPms);
  b.prefix = (double4*)at(kBhPrefix);
  b.scan_part = (double4*)at(kBhScanPart);
  b.nodes = (nb_node*)at(kBhNode);
  b.node_next = (int*)at(kBhNext);
  b.level_off = (int*)at(kBhLevel);
  b.marks = (unsigned char*)at(kBhMarks);
  b.node_end = (int*)at(kBhNodeEnd);
  b.level_cnt = (int*)at(kBhLevelCnt);
  b.counters = (int*)at(kBhCounters);
  b.waves = (int4*)at(kBhWaves);
  b.inter = (unsigned long long*)at(kBhInter);
  b.rec_cost = (float*)at(kBhRecCost);
  b.rec_bucket = (int*)at(kBhRecBucket);
  b.rec_order = (int*)at(kBhRecOrder);
  b.rec_hist = (int*)at(kBhRecHist);
  b.bbox_blocks = kBboxBlocks;
  b.sort_blocks = (int)L.sort_blocks;
  b.max_nodes = upto > kBhPms ? L.max_nodes : 0;
  int dev = 0, cus = 256;
  (void)hipGetDevice(&dev);
  (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
  b.persist_blocks = kListBlocksPerCU * cus;  // resident traversal blocks
}

int nb_sort_alloc(nb_ctx* c) {
  NB_TRY
  nb_bh_state& b = c->bh;
  if (b.keys[0]) return NB_OK;
  const nb_bh_layout L = nb_bh_layout_for(c->n);
  if (hipMalloc(&b.block, (size_t)L.off[kBhPms]) != hipSuccess) {
    b.block = nullptr;
    return nb_fail(NB_E_OOM, "device allocation failed (Morton sort)");
  }
  nb_bh_carve(c, (char*)b.block, kBhPms);
  if (hipMemset(b.geom, 0, sizeof(float) * 32) != hipSuccess)
    return nb_fail(NB_E_HIP, "hipMemset failed (Morton sort)");
  return NB_OK;
  NB_CATCH("nb_sort_alloc")
}

int nb_bh_alloc(nb_ctx* c) {
  NB_TRY
  nb_bh_state& b = c->bh;
  const nb_bh_layout L = nb_bh_layout_for(c->n);
  if (hipMalloc(&b.block, (size_t)L.off[kBhBufCount]) != hipSuccess) {
    b.block = nullptr;
    return nb_fail(NB_E_OOM, "nb_create: device allocation failed (octree)");
  }
  nb_bh_carve(c, (char*)b.block, kBhBufCount);
  if (hipMemset(b.geom, 0, sizeof(float) * 32) != hipSuccess ||
      hipMemset(b.rec_cost, 0, sizeof(float) * c->n) != hipSuccess)
    return nb_fail(NB_E_HIP, "nb_create: hipMemset failed (octree)");
  return NB_OK;
  NB_CATCH("nb_bh_alloc")
}

void nb_bh_free(nb_ctx* c) {
  nb_bh_state& b = c->bh;
  if (b.block) (void)hipFree(b.block);
  b = nb_bh_state{};
}

// Up to here each block takes bounds and counts from all bodies instead of from other
// launches' partial ones. Measured Barnes-Hut steps in us (Plummer sphere / uniform
// ball), partial and own:
//     4,000 bodies   96.4/ 80.8   84.9/ 69.9
//    10,000         113.9/ 96.2  106.9/ 87.9
//    20,011         121.0/105.4  118.9/100.5
//    30,011         145.9/118.3  145.0/116.4
//    40,000         157.1/130.1  162.5/131.3
//    65,536         204.9/158.0  217.3/161.9
constexpr int kSelfBodies = 3 << 13;

hipError_t nb_morton_sort(nb_ctx* c) {
  nb_bh_state& b = c->bh;
  const int n = c->n;
  hipStream_t s = c->stream;
  const int tiles = b.sort_blocks, groups = (tiles + kSortGroup - 1) / kSortGroup;
  const int cubic = (c->cfg.flags & NB_F_BH_AXIS_BOX) ? 0 : 1;
  const bool self = n <= kSelfBodies;
  // 1-2. bounding box and codes
  if (self) {
    hipLaunchKernelGGL(k_morton<true>, dim3(tiles), dim3(1024), 0, s, c->pm, n, cubic, nullptr, 0,
                       b.geom, b.codes, nullptr, nullptr);
  } else {
    const int parts = std::min(b.bbox_blocks, (n + 1023) / 1024);
    hipLaunchKernelGGL(k_bbox_partial, dim3(parts), dim3(1024), 0, s, c->pm, n, b.bbox_part,
                       b.group_hist, 4 * 256 * groups);
    hipLaunchKernelGGL(k_morton<false>, dim3(tiles), dim3(1024), 0, s, c->pm, n, cubic, b.bbox_part,
                       parts, b.geom, b.codes, b.digit_hist, b.group_hist);
  }
  // 3. sort: the last pass writes keys[0] and vals[0]
  const auto scatter = [&](auto kernel, const uint32_t* keys, const uint32_t* vals, int shift,
                           int* gh, int out) {
    const bool scan = gh && groups >= kScanGroups;
    if (scan) hipLaunchKernelGGL(k_radix_groups, dim3(1), dim3(1024), 0, s, gh, groups);
    hipLaunchKernelGGL(kernel, dim3(tiles), dim3(1024), 0, s, keys, vals, n, shift, b.digit_hist, gh,
                       scan ? 0 : groups, b.keys[out], b.vals[out]);
  };
  if (self) {
    scatter(k_radix_scatter<true, true>, b.codes, nullptr, 0, nullptr, 0);
    scatter(k_radix_scatter<false, true>, b.keys[0], b.vals[0], 10, nullptr, 1);
    scatter(k_radix_scatter<false, true>, b.keys[1], b.vals[1], 20, nullptr, 0);
  } else {
    scatter(k_radix_scatter<true, false>, b.codes, nullptr, 0, b.group_hist, 1);
    for (int pass = 1; pass < 4; ++pass) {
      const int in = pass & 1;
      int* gh = b.group_hist + pass * groups * 256;
      hipLaunchKernelGGL(k_radix_hist, dim3(tiles), dim3(1024), 0, s, b.keys[in], n, 8 * pass,
                         b.digit_hist, gh);
      scatter(k_radix_scatter<false, false>, b.keys[in], b.vals[in], 8 * pass, gh, in ^ 1);
    }
  }
  return hipGetLastError();
}

hipError_t nb_launch_permute_state(nb_ctx* c) {
  nb_bh_state& b = c->bh;
  const int n = c->n;
  hipStream_t s = c->stream;
  const int g256 = (n + 255) / 256;
  const uint32_t* perm = b.vals[0];
  double* arrays[4] = {c->pos, c->vel, c->acc, c->force};
  for (double* a : arrays) {
    hipLaunchKernelGGL(k_permute_d3, dim3(g256), dim3(256), 0, s, a, perm, n, c->tmp);
    hipError_t e = hipMemcpyAsync(a, c->tmp, sizeof(double) * 3 * n, hipMemcpyDeviceToDevice, s);
    if (e != hipSuccess) return e;
  }
  float* mtmp = reinterpret_cast<float*>(c->tmp);
  hipLaunchKernelGGL(k_permute_f32, dim3(g256), dim3(256), 0, s, c->mass, perm, n, mtmp);
  return hipMemcpyAsync(c->mass, mtmp, sizeof(float) * n, hipMemcpyDeviceToDevice, s);
}

hipError_t nb_bh_build(nb_ctx* c) {
  nb_bh_state& b = c->bh;
  const int n = c->n;
  hipStream_t s = c->stream;
  hipError_t es = nb_morton_sort(c);
  if (es != hipSuccess) return es;
  const uint32_t* codes_sorted = b.keys[0];
  const uint32_t* perm = b.vals[0];
  const int tiles = (n + kTreeTile - 1) / kTreeTile;
  const int leaf = c->cfg.leaf_size;
  const int pairs = nb_bh_pairs(n, c->cfg.flags) ? 1 : 0;
  // 4-6. bodies in sorted order, FP64 moment prefix, octree
  hipLaunchKernelGGL(k_tree_mark, dim3(tiles), dim3(kTreeTile), 0, s, codes_sorted, perm, c->pm,
                     n, leaf, b.pms, b.scan_part, b.marks, b.level_cnt);
  const Records records{b.waves, b.counters, b.rec_hist};
  const auto emit = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(tiles), dim3(kTreeTile), 0, s, b.pms, n, leaf, pairs,
                       b.scan_part, b.marks, b.level_cnt, b.counters, records, b.max_nodes,
                       b.prefix, b.nodes, b.node_next, b.node_end, b.level_off, c->flags);
  };
  if (tiles <= 64) {
    emit(k_tree_emit<true>);
  } else {
    hipLaunchKernelGGL(k_tree_scan, dim3(2 + kLevels), dim3(kScanThreads), 0, s, b.scan_part,
                       b.level_cnt, tiles, n, leaf, pairs, b.counters, records);
    emit(k_tree_emit<false>);
  }
  // 7. centre of mass, wave ranges
  const int cgrid = (int)std::max<int64_t>(1, std::min<int64_t>((b.max_nodes + 255) / 256, 8192));
  const int cubic = (c->cfg.flags & NB_F_BH_AXIS_BOX) ? 0 : 1;
  hipLaunchKernelGGL(k_tree_com, dim3(cgrid), dim3(256), 0, s, b.nodes, b.node_end, n,
                     b.max_nodes, b.level_off, b.prefix, b.pms, codes_sorted, b.geom, cubic,
                     c->cfg.theta, leaf, pairs, b.waves, b.counters);
  return hipGetLastError();
}

hipError_t nb_bh_traverse(nb_ctx* c, bool count_interactions) {
  nb_bh_state& b = c->bh;
  const int n = c->n;
  const int g256 = (n + 255) / 256;
  const bool group = !(c->cfg.flags & NB_F_BH_PER_BODY);
  if (count_interactions)
    hipLaunchKernelGGL(k_zero_u64, dim3(1), dim3(64), 0, c->stream, b.inter);
#define NB_TRAVERSE_ARGS                                                                       \
  b.pms, b.vals[0], n, b.nodes, b.node_next, b.level_off, b.max_nodes, b.geom, c->theta2, \
      c->cfg.eps2, c->G, c->force, b.inter, c->flags
  const bool guard = c->guard;
  const int gl = b.persist_blocks;  // persistent blocks pulling wave ranges
  // work costliest first from kOrderMinBodies on (and wherever pairs are
  // forced); smaller systems take their records in order and keep no times
  const bool ordered = group && (n >= kOrderMinBodies || (c->cfg.flags & NB_F_BH_PAIRS) != 0);
  if (ordered) {
    const int og = std::max(1, std::min((n + kOrderChunk - 1) / kOrderChunk, kOrderBlocks));
    hipLaunchKernelGGL(k_rec_bucket, dim3(og), dim3(256), 0, c->stream, b.waves, b.counters, n,
                       b.rec_cost, b.vals[0], b.rec_bucket, b.rec_hist);
    hipLaunchKernelGGL(k_rec_scatter, dim3(og), dim3(256), 0, c->stream, b.counters, n,
                       b.rec_bucket, b.rec_hist, b.rec_order);
  }
#define NB_LIST_ARGS                                                                     \
  b.pms, b.vals[0], n, b.nodes, b.level_off, b.max_nodes, c->cfg.eps2,     \
      c->G, c->force, b.inter, c->flags, b.waves, b.counters,                \
      ordered ? b.rec_order : nullptr, ordered ? b.rec_cost : nullptr, c->walk_stack
  if (group && count_interactions && guard)
    hipLaunchKernelGGL((k_traverse_list<true, true>), dim3(gl), dim3(64 * kListWaves), 0, c->stream,
                       NB_LIST_ARGS);
  else if (group && count_interactions)
    hipLaunchKernelGGL((k_traverse_list<true, false>), dim3(gl), dim3(64 * kListWaves), 0, c->stream,
                       NB_LIST_ARGS);
  else if (group && n < kBlockMaxBodies && !nb_bh_pairs(n, c->cfg.flags)) {
    const auto launch = [&](auto kernel, int waves) {
      const int blocks = b.persist_blocks / kListBlocksPerCU * (kBlockWavesPerCU / waves);
      hipLaunchKernelGGL(kernel, dim3(blocks), dim3(64 * waves), 0, c->stream, b.pms, b.vals[0], n,
                         b.nodes, b.level_off, b.max_nodes, c->cfg.eps2,
                         c->G, c->force, c->flags, b.waves, b.counters,
                         ordered ? b.rec_order : nullptr, ordered ? b.rec_cost : nullptr,
                         c->walk_stack);
    };
    if (n < kBlock8Bodies)
      guard ? launch(k_traverse_block<true, 8>, 8) : launch(k_traverse_block<false, 8>, 8);
    else
      guard ? launch(k_traverse_block<true, 4>, 4) : launch(k_traverse_block<false, 4>, 4);
  } else if (group && guard)
    hipLaunchKernelGGL((k_traverse_list<false, true>), dim3(gl), dim3(64 * kListWaves), 0, c->stream,
                       NB_LIST_ARGS);
  else if (group)
    hipLaunchKernelGGL((k_traverse_list<false, false>), dim3(gl), dim3(64 * kListWaves), 0, c->stream,
                       NB_LIST_ARGS);
#undef NB_LIST_ARGS
  else if (count_interactions)
    hipLaunchKernelGGL((k_traverse<true>), dim3(g256), dim3(256), 0, c->stream, NB_TRAVERSE_ARGS);
  else
    hipLaunchKernelGGL((k_traverse<false>), dim3(g256), dim3(256), 0, c->stream, NB_TRAVERSE_ARGS);
#undef NB_TRAVERSE_ARGS
  return hipGetLastError();
}

hipError_t nb_bh_count_per_body(nb_ctx* c) {
  nb_bh_state& b = c->bh;
  const int n = c->n;
  hipLaunchKernelGGL(k_zero_u64, dim3(1), dim3(64), 0, c->stream, b.inter);
  hipLaunchKernelGGL((k_traverse<true, true>), dim3((n + 255) / 256), dim3(256), 0, c->stream, b.pms,
                     b.vals[0], n, b.nodes, b.node_next, b.level_off, b.max_nodes, b.geom,
                     c->theta2, c->cfg.eps2, c->G, c->force, b.inter, c->flags);
  return hipGetLastError();
}

// ---- debug taps ---------------------------------------------------------------------------------
extern "C" int nb_debug_set_walk_stack(nb_ctx* c, int32_t entries) {
  NB_TRY
  if (!c) return nb_fail(NB_E_ARG, "nb_debug_set_walk_stack: null context");
  if (entries < 0 || entries > kStackCap)
    return nb_fail(NB_E_ARG, "nb_debug_set_walk_stack: entries must be 0..512");
  // a captured step holds the old value as a kernel argument
  nb_drop_graph(c->stream, c->graph_exec, c->graph);
  c->walk_stack = entries;
  return NB_OK;
  NB_CATCH("nb_debug_set_walk_stack")
}

extern "C" int nb_debug_morton(nb_ctx* c, uint32_t* codes, uint32_t* perm) {
  NB_TRY
  if (!c) return nb_fail(NB_E_ARG, "nb_debug_morton: null context");
  if (c->cfg.solver != NB_SOLVER_BH) return nb_fail(NB_E_ARG, "nb_debug_morton: not a BH context");
  if (!c->tree_valid) return nb_fail(NB_E_ARG, "nb_debug_morton: no BH force pass has run");
  NB_HIP(hipStreamSynchronize(c->stream));
  if (codes) NB_HIP(hipMemcpy(codes, c->bh.codes, sizeof(uint32_t) * c->n, hipMemcpyDeviceToHost));
  if (perm) NB_HIP(hipMemcpy(perm, c->bh.vals[0], sizeof(uint32_t) * c->n, hipMemcpyDeviceToHost));
  return NB_OK;
  NB_CATCH("nb_debug_morton")
}

extern "C" int nb_debug_tree(nb_ctx* c, nb_node_view* nodes, int64_t cap, int64_t* node_count,
                             float* bbox) {
  NB_TRY
  if (!c) return nb_fail(NB_E_ARG, "nb_debug_tree: null context");
  if (c->cfg.solver != NB_SOLVER_BH) return nb_fail(NB_E_ARG, "nb_debug_tree: not a BH context");
  if (!c->tree_valid) return nb_fail(NB_E_ARG, "nb_debug_tree: no BH force pass has run");
  NB_HIP(hipStreamSynchronize(c->stream));
  int off[kMaxLevel + 2];
  NB_HIP(hipMemcpy(off, c->bh.level_off, sizeof(off), hipMemcpyDeviceToHost));
  const int64_t total = off[kMaxLevel + 1];
  if (node_count) *node_count = total;
  if (bbox) NB_HIP(hipMemcpy(bbox, c->bh.geom, sizeof(float) * 6, hipMemcpyDeviceToHost));
  const int64_t m = std::min<int64_t>(cap, total);
  if (nodes && m > 0) {
    std::vector<nb_node> nd(m);
    std::vector<int> next(m);
    NB_HIP(hipMemcpy(nd.data(), c->bh.nodes, sizeof(nb_node) * m, hipMemcpyDeviceToHost));
    NB_HIP(hipMemcpy(next.data(), c->bh.node_next, sizeof(int) * m, hipMemcpyDeviceToHost));
    for (int64_t k = 0; k < m; ++k) {
      nb_node_view& v = nodes[k];
      v.com[0] = nd[k].com.x;
      v.com[1] = nd[k].com.y;
      v.com[2] = nd[k].com.z;
      v.mass = nd[k].com.w;
      v.first_child = nd[k].first;
      v.next = next[k];
      v.body_start = nd[k].start;
      v.body_count = nd[k].span >> 4;
      v.level = nd[k].span & 15;
      v.open_r2 = nd[k].r2;
    }
  }
  return NB_OK;
  NB_CATCH("nb_debug_tree")
}
