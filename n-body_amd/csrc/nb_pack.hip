// nb_pack.hip — between the caller's host arrays (one body after the other:
// float4 or double[3]) and the device state (FP64, one plane per component).
//
// The layouts are changed on the device. Results leave through a small pinned
// buffer that the kernel writes itself over the bus, so a small call is one
// kernel, one wait and one memcpy; a large one alternates the buffer's halves,
// the kernel filling one while the host empties the other. Measured into fresh
// host memory: 64 KB 16 us (kernel, pageable copy 44 us), 1 MB 66 us, 64 MB
// 14 GB/s (one hipMemcpy: 10 GB/s), 201 MB 38 GB/s with more threads copying.
// Converting on the host instead (three pageable copies and a transpose) took 84 us
// for the state of 1000 bodies and 92 ms at 4,194,304; now 12 us and 5.4 ms.
#include <algorithm>
#include <atomic>
#include <chrono>
#include <condition_variable>
#include <cstring>
#include <mutex>
#include <thread>

#include "nb_force_core.h"
#include "nb_internal.h"

namespace {

struct PackArgs {
  const double* src[3];  // first plane of each array
  int64_t stride;        // from one plane to the next
  int64_t part_first, part_stride;  // parts > 1: each value is G times a sum (nb_planes)
  double G;
  int parts;
  int n;               // bodies to pack
  int first;           // the first of them (caller's index)
  const int* slot_of;  // slot of each body, or null: body i is in slot i
  char* dst;           // array k at dst + k * n * (bytes per body)
  const int* flags;    // copied to flags_dst when not null
  int* flags_dst;
};

__device__ __forceinline__ double pack_value(const PackArgs& a, const double* src, int64_t k) {
  double f = src[k];
  if (a.parts > 1) {
    for (int p = 1; p < a.parts; ++p) f += src[a.part_first + (p - 1) * a.part_stride + k];
    f *= a.G;
  }
  return f;
}

// Thread per stored element, so that the stores over the bus are contiguous:
// a float4 body, or one double of an interleaved body.
template <int kLayout>
__global__ __launch_bounds__(256) void k_pack(PackArgs a) {
  const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (t == 0 && blockIdx.y == 0 && a.flags) *a.flags_dst = *a.flags;
  const double* src = a.src[blockIdx.y];
  if (kLayout == kPackD3) {
    if (t >= 3 * (int64_t)a.n) return;
    const int body = (int)(t / 3), comp = (int)(t - 3 * (int64_t)body);
    const int slot = a.slot_of ? a.slot_of[a.first + body] : a.first + body;
    double* dst = reinterpret_cast<double*>(a.dst) + blockIdx.y * 3 * (int64_t)a.n;
    dst[t] = pack_value(a, src, comp * a.stride + slot);
    return;
  }
  if (t >= a.n) return;
  const int slot = a.slot_of ? a.slot_of[a.first + t] : a.first + (int)t;
  float4 v;
  v.x = (float)pack_value(a, src, slot);
  v.y = (float)pack_value(a, src, a.stride + slot);
  v.z = (float)pack_value(a, src, 2 * a.stride + slot);
  v.w = 0.f;
  if (kLayout == kPackView) {  // |v|: the inputs of the reference's point shaders
                               // (vertexShader.glsl:3-9, fragmentShader.glsl)
    const double* vel = a.src[1];
    const double vx = vel[slot], vy = vel[a.stride + slot], vz = vel[2 * a.stride + slot];
    v.w = (float)sqrt(vx * vx + vy * vy + vz * vz);
  }
  reinterpret_cast<float4*>(a.dst)[blockIdx.y * (int64_t)a.n + t] = v;
}

hipError_t launch_pack(int layout, const PackArgs& a, int arrays, hipStream_t s) {
  const int64_t elems = layout == kPackD3 ? 3 * (int64_t)a.n : a.n;
  const dim3 grid((unsigned)((elems + 255) / 256), arrays);
  if (layout == kPackD3) hipLaunchKernelGGL((k_pack<kPackD3>), grid, dim3(256), 0, s, a);
  else if (layout == kPackF4) hipLaunchKernelGGL((k_pack<kPackF4>), grid, dim3(256), 0, s, a);
  else hipLaunchKernelGGL((k_pack<kPackView>), grid, dim3(256), 0, s, a);
  return hipGetLastError();
}

// 256 bodies per block. Interleaved doubles pass through LDS, so that the loads
// (over the bus in small calls) and the stores are both contiguous.
template <int kLayout>
__device__ __forceinline__ void unpack_array(const void* src, int64_t n, int64_t b0, double (&v)[3],
                                             double* lds) {
  const int64_t i = b0 + threadIdx.x;
  if (kLayout == kPackF4) {
    const float4 q = i < n ? static_cast<const float4*>(src)[i] : make_float4(0.f, 0.f, 0.f, 0.f);
    v[0] = q.x;
    v[1] = q.y;
    v[2] = q.z;
    return;
  }
  __syncthreads();  // the previous array has been read
#pragma unroll
  for (int r = 0; r < 3; ++r) {
    const int64_t k = 3 * b0 + r * 256 + threadIdx.x;
    lds[r * 256 + threadIdx.x] = k < 3 * n ? static_cast<const double*>(src)[k] : 0.0;
  }
  __syncthreads();
#pragma unroll
  for (int a = 0; a < 3; ++a) v[a] = lds[3 * threadIdx.x + a];
}

struct UnpackArgs {
  const void* src[3];  // positions, velocities, accelerations (null: zero), packed
  const float* mass;   // n masses
  double* dst[3];      // first plane of each array (null: the array is not part of this call)
  int64_t stride;
  int n, n_pad;        // bodies, and the entries of pm to fill (padding past n)
  float* mass_dst;     // null: the masses are in place
  float4* pm;          // written with the positions
  float scale;         // of the coordinates in pm
  int* flags;          // four words set to zero, or null
};

template <int kLayout>
__global__ __launch_bounds__(256) void k_unpack(UnpackArgs a) {
  __shared__ double lds[kLayout == kPackD3 ? 768 : 1];
  const int64_t b0 = (int64_t)blockIdx.x * 256, i = b0 + threadIdx.x;
  if (b0 == 0 && threadIdx.x < 4 && a.flags) a.flags[threadIdx.x] = 0;
  const bool body = i < a.n;
  float m = 0.f;
  if (a.pm && body) {
    m = a.mass[i];
    if (a.mass_dst) a.mass_dst[i] = m;
  }
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    if (!a.dst[k]) continue;
    double v[3] = {0.0, 0.0, 0.0};
    if (a.src[k]) unpack_array<kLayout>(a.src[k], a.n, b0, v, lds);
    if (body)
#pragma unroll
      for (int c = 0; c < 3; ++c) a.dst[k][c * a.stride + i] = v[c];
    if (k == 0 && a.pm && i < a.n_pad)
      a.pm[i] = body ? make_float4((float)v[0] * a.scale, (float)v[1] * a.scale,
                                   (float)v[2] * a.scale, m)
                     : nbcore::far_pad();
  }
}

hipError_t launch_unpack(int layout, const UnpackArgs& a, hipStream_t s) {
  const dim3 grid((unsigned)((a.n_pad + 255) / 256));
  if (layout == kPackD3) hipLaunchKernelGGL((k_unpack<kPackD3>), grid, dim3(256), 0, s, a);
  else hipLaunchKernelGGL((k_unpack<kPackF4>), grid, dim3(256), 0, s, a);
  return hipGetLastError();
}

// Copies between the stage and the caller's memory by a few threads that live as
// long as one call: one core moves 10 to 14 GB/s, fresh pages included, and the bus
// 50. The helpers only copy; every HIP call stays on the caller's thread. If none can
// be started the caller copies alone. Until the first chunk is there, behind all steps
// that are still queued, and in longer pauses they sleep.
class CopyTeam {
 public:
  explicit CopyTeam(int64_t bytes) {
    if (bytes < kMinBytes) return;
    const int want = (int)std::min<int64_t>(kHelpers, 1 + bytes / (8 << 20));
    try {
      for (; count_ < want; ++count_) helpers_[count_] = std::thread([this, k = count_] { help(k); });
    } catch (...) {
    }
  }
  ~CopyTeam() {
    {
      std::lock_guard<std::mutex> lk(mu_);
      stop_.store(true, std::memory_order_release);
    }
    cv_.notify_all();
    for (int k = 0; k < count_; ++k) helpers_[k].join();
  }
  CopyTeam(const CopyTeam&) = delete;
  CopyTeam& operator=(const CopyTeam&) = delete;

  void copy(void* dst, const void* src, size_t bytes) {
    if (count_ == 0 || bytes < (64 << 10)) {
      std::memcpy(dst, src, bytes);
      return;
    }
    dst_ = static_cast<char*>(dst);
    src_ = static_cast<const char*>(src);
    bytes_ = bytes;
    busy_.store(count_, std::memory_order_relaxed);
    {
      std::lock_guard<std::mutex> lk(mu_);
      job_.fetch_add(1, std::memory_order_release);
    }
    cv_.notify_all();
    slice(count_);
    while (busy_.load(std::memory_order_acquire) > 0) std::this_thread::yield();
  }

 private:
  static constexpr int64_t kMinBytes = 4 << 20;  // below: starting helpers costs what they save
  static constexpr int kHelpers = 5;  // 201 MB into fresh memory: none 14 GB/s, one 20, three 28,
                                      // five 38, seven 40; 12.6 MB: one 24, seven 23
  static constexpr std::chrono::microseconds kSpin{200};  // a chunk of 8 MB is 160 us on the bus

  void slice(int k) {  // of count_ + 1, whole pages each
    const size_t per = (bytes_ / (count_ + 1) + 4095) & ~size_t(4095);
    const size_t at = std::min(bytes_, per * k), end = k == count_ ? bytes_ : std::min(bytes_, at + per);
    std::memcpy(dst_ + at, src_ + at, end - at);
  }
  void help(int k) {
    using clock = std::chrono::steady_clock;
    for (int64_t seen = 0;; ++seen) {  // jobs follow each other only when all have done the last
      const auto idle = [&] {
        return job_.load(std::memory_order_acquire) == seen && !stop_.load(std::memory_order_acquire);
      };
      if (seen > 0)  // the next chunk is on its way
        for (const auto until = clock::now() + kSpin; idle() && clock::now() < until;) std::this_thread::yield();
      if (idle()) {
        std::unique_lock<std::mutex> lk(mu_);
        cv_.wait(lk, [&] { return !idle(); });
      }
      if (job_.load(std::memory_order_acquire) == seen) return;  // stopped
      slice(k);
      busy_.fetch_sub(1, std::memory_order_acq_rel);
    }
  }

  char* dst_ = nullptr;
  const char* src_ = nullptr;
  size_t bytes_ = 0;
  std::atomic<int64_t> job_{0};
  std::atomic<int> busy_{0};
  std::atomic<bool> stop_{false};
  std::mutex mu_;
  std::condition_variable cv_;
  int count_ = 0;  // helpers that started; they read it only after a job is posted
  std::thread helpers_[kHelpers];
};

int64_t body_bytes(int layout) { return layout == kPackD3 ? 24 : 16; }

}  // namespace

int nb_stage_ready(nb_stage& st, hipStream_t s, int64_t bytes) {
  if (st.busy) NB_HIP(hipStreamSynchronize(s));
  st.busy = false;
  if (st.bytes < bytes) {
    if (st.host) NB_HIP(hipHostFree(st.host));
    st.host = nullptr;
    st.bytes = 0;
    if (hipHostMalloc(reinterpret_cast<void**>(&st.host), bytes, hipHostMallocDefault) != hipSuccess) {
      st.host = nullptr;
      return nb_fail(NB_E_OOM, "pinned host allocation failed");
    }
    st.bytes = bytes;
    for (auto& e : st.done)
      if (!e) NB_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
  }
  return NB_OK;
}

void nb_stage_free(nb_stage& st) {
  if (st.host) (void)hipHostFree(st.host);
  for (auto& e : st.done)
    if (e) (void)hipEventDestroy(e);
  st = nb_stage{};
}

int nb_fetch(nb_stage& st, hipStream_t s, const nb_planes& p, int layout, int arrays,
             const double* const* src, void* const* dst, const int* flags, int* flags_out) {
  const int64_t per = body_bytes(layout);
  const int sources = layout == kPackView ? 1 : arrays;  // the view reads two arrays into one
  const int64_t all = sources * p.n * per;
  // the size of large calls lets every thread of the team fill pages of its own
  const int rc = nb_stage_ready(st, s, all >= 2 * kLargeStageBytes ? kLargeStageBytes : kStageBytes);
  if (rc) return rc;
  int* stage_flags = reinterpret_cast<int*>(st.host + st.bytes) - 1;
  PackArgs a{};
  a.stride = p.stride;
  a.part_first = p.part_first;
  a.part_stride = p.part_stride;
  a.parts = p.parts;
  a.G = p.G;
  a.slot_of = p.slot_of;
  a.flags_dst = stage_flags;
  if (all + 64 <= kStageBytes) {
    for (int k = 0; k < arrays; ++k) a.src[k] = src[k];
    a.n = (int)p.n;
    a.dst = st.host;
    a.flags = flags;
    NB_HIP(launch_pack(layout, a, sources, s));
    NB_HIP(hipStreamSynchronize(s));
    for (int k = 0; k < sources; ++k)
      std::memcpy(dst[k], st.host + k * p.n * per, p.n * per);
  } else {
    // halves of the stage in turn: the kernel fills one while the host empties the other
    CopyTeam team(all);
    const int64_t half = (st.bytes - 64) / 2 / 256 * 256, chunk = half / per;
    const int64_t chunks = (p.n + chunk - 1) / chunk, total = chunks * sources;
    const auto fill = [&](int64_t c) -> int {
      const int64_t i0 = c % chunks * chunk;
      for (int k = 0; k < arrays; ++k) a.src[k] = src[layout == kPackView ? k : c / chunks];
      a.first = (int)i0;
      a.n = (int)std::min(chunk, p.n - i0);
      a.dst = st.host + (c & 1) * half;
      a.flags = c + 1 == total ? flags : nullptr;
      NB_HIP(launch_pack(layout, a, 1, s));
      NB_HIP(hipEventRecord(st.done[c & 1], s));
      return NB_OK;
    };
    int e = fill(0);
    for (int64_t c = 0; !e && c < total; ++c) {
      if (c + 1 < total) e = fill(c + 1);
      if (e) break;
      NB_HIP(hipEventSynchronize(st.done[c & 1]));
      const int64_t i0 = c % chunks * chunk;
      team.copy(static_cast<char*>(dst[c / chunks]) + i0 * per, st.host + (c & 1) * half,
                std::min(chunk, p.n - i0) * per);
    }
    if (e) return e;
  }
  if (flags_out) *flags_out = flags ? *stage_flags : 0;
  return NB_OK;
}

int nb_put(nb_stage& st, hipStream_t s, void* dev_tmp, int layout, const nb_put_args& p) {
  UnpackArgs a{};
  a.stride = p.stride;
  a.n = (int)p.n;
  a.n_pad = (int)p.n_pad;
  a.scale = p.scale;
  const int64_t per = body_bytes(layout);
  const void* from[3] = {p.pos, p.vel, p.acc};
  if (3 * p.n * per + 4 * p.n <= kStageBytes) {
    // through the stage; nothing waits: the next use of the stage does
    const int rc = nb_stage_ready(st, s, kStageBytes);
    if (rc) return rc;
    char* at = st.host;
    for (int k = 0; k < 3; ++k) {
      a.dst[k] = p.dst[k];
      if (!from[k]) continue;
      std::memcpy(at, from[k], p.n * per);
      a.src[k] = at;
      at += p.n * per;
    }
    std::memcpy(at, p.mass, p.n * sizeof(float));
    a.mass = reinterpret_cast<const float*>(at);
    a.mass_dst = p.mass_dst;
    a.pm = p.pm;
    a.flags = p.flags;
    NB_HIP(launch_unpack(layout, a, s));
    st.busy = true;
    return NB_OK;
  }
  // array by array through device memory
  NB_HIP(hipMemcpyAsync(p.mass_dst, p.mass, p.n * sizeof(float), hipMemcpyHostToDevice, s));
  for (int k = 0; k < 3; ++k) {
    if (from[k]) NB_HIP(hipMemcpyAsync(dev_tmp, from[k], p.n * per, hipMemcpyHostToDevice, s));
    for (int j = 0; j < 3; ++j) {
      a.src[j] = j == k && from[k] ? dev_tmp : nullptr;
      a.dst[j] = j == k ? p.dst[k] : nullptr;
    }
    a.mass = k == 0 ? p.mass_dst : nullptr;
    a.pm = k == 0 ? p.pm : nullptr;
    a.flags = k == 0 ? p.flags : nullptr;
    NB_HIP(launch_unpack(layout, a, s));
  }
  NB_HIP(hipStreamSynchronize(s));  // the caller's arrays are free again
  return NB_OK;
}
