// What the GEMMs share when tiles are cut along K over several workgroups each: device memory for the partial tiles and
// tickets for the kernels whose last workgroup of a tile adds them, and, for the 16-bit tiles, the kernel that adds partial
// M x N planes up.
#include <algorithm>
#include <map>
#include <mutex>
#include <type_traits>
#include <utility>

#include "common.hpp"
#include "gemm_common.hpp"

namespace sarek_hip {
namespace {

// The sum of four columns' `splits` partial sums, up to nine of them asked for at once: one after the other, each waited a trip to the
// caches for the one before (us, with the products: 161 x 256 x 7182, 13 pieces, 14.2 and 12.4; 63 x 1130 x 7104, 14.4, 12.6; fused 98 x
// 576 x 2432 13.1, 11.4).  What is there is added in pairs, pairs of pairs and so on, the same for every run: 14 in a row were 38 x 2250 x
// 7680 1.03 of the few-rows kernel's error, so they are 0.96.  (In double 0.80, but a launch of 1.4 us more work: fused 67 x 4838 x 2885
// 18.6 to 20.1 us.)
template <int Count, class Vec>
__device__ __forceinline__ void add_next(f32x4_t &acc, const float *__restrict__ p, int64_t plane) {
  f32x4_t v[Count + 1];
  v[0] = acc;
#pragma unroll
  for (int u = 0; u < Count; ++u) v[u + 1] = *reinterpret_cast<const Vec *>(p + u * plane);
  // (without it the first pair is waited for before the other planes are asked for: fused 88 x 4928 x 3823 20.5 us, 18.5 with it)
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int w = 1; w <= Count; w *= 2)
#pragma unroll
    for (int u = 0; u + w <= Count; u += 2 * w) v[u] += v[u + w];
  acc = v[0];
}
template <class Vec>
__device__ __forceinline__ f32x4_t add_planes(const float *__restrict__ p, int64_t plane, int splits) {
  f32x4_t acc = *reinterpret_cast<const Vec *>(p);
  for (int s = 1; s < splits; s += 8) {
    const float *next = p + s * plane;
    switch (min(splits - s, 8)) {
      case 1: add_next<1, Vec>(acc, next, plane); break;
      case 2: add_next<2, Vec>(acc, next, plane); break;
      case 3: add_next<3, Vec>(acc, next, plane); break;
      case 4: add_next<4, Vec>(acc, next, plane); break;
      case 5: add_next<5, Vec>(acc, next, plane); break;
      case 6: add_next<6, Vec>(acc, next, plane); break;
      case 7: add_next<7, Vec>(acc, next, plane); break;
      default: add_next<8, Vec>(acc, next, plane);
    }
  }
  return acc;
}

// Adds the `splits` partial planes into C: a fixed order, so the result does not depend on which
// workgroup finished when.  C is 16-byte aligned (the callers' condition).
__global__ __launch_bounds__(256) void splitk_reduce_kernel(const float *__restrict__ partials, float *__restrict__ C,
                                                            int64_t mn, int64_t plane, int splits) {
  const int64_t i = (static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x) * 4;
  if (i >= mn) return;
  const f32x4_t acc = add_planes<f32x4_t>(partials + i, plane, splits);
  if (i + 4 <= mn) {
    *reinterpret_cast<f32x4_t *>(C + i) = acc;
  } else {
    for (int j = 0; i + j < mn; ++j) C[i + j] = acc[j];
  }
}

// The same for the fused product: y = relu(sum of the planes + bias), and the row's sum of y, in double, in a fixed order.  Waves
// of the four of a workgroup to a row.  Bound by the trips to the planes, which the products have left in the caches: a wave takes 256
// columns a turn, so of more it makes several trips where two or four waves make one.  Us, products with one wave to a row, two and four:
// 205 x 875 x 6932 20.2, 18.5, 17.3 (20.6 when such products were not cut), 133 x 958 x 4595 18.3, 16.3, 15.0 (17.5), 361 x 512 x 2112 12.2,
// 11.9, 13.6; with many rows the workgroups count: 2690 x 350 x 7071 in two pieces 41.4, 42.4, 43.3, 2000 x 1025 x 2000 31.4, 31.5, 32.8,
// 4642 x 583 x 6966 81 and 84.  The last one to three columns of an odd N are read four at a time too, with some of those before them: one by
// one they waited for every plane (205 x 875 x 6932 20.2, 17.3 now).
template <int Waves>
__global__ __launch_bounds__(256) void splitk_reduce_fused_kernel(const float *__restrict__ partials, const float *__restrict__ bias,
                                                                  float *__restrict__ y, float *__restrict__ rowsum, int m, int n,
                                                                  int64_t plane, int splits) {
  __shared__ double sums[4];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int row = static_cast<int>(blockIdx.x) * (4 / Waves) + wave / Waves;
  double sum = 0.0;
  if (row < m) {
    const float *p = partials + static_cast<int64_t>(row) * n;
    float *out = y + static_cast<int64_t>(row) * n;
    for (int c = (wave % Waves * 64 + lane) * 4; c < n; c += Waves * 256) {
      if (n >= 4) {
        const int at = min(c, n - 4);   // the last columns with some of those before them: one by one they wait for each plane
        const f32x4_t b = *reinterpret_cast<const f32x4_u *>(bias + at);
        f32x4_t acc = add_planes<f32x4_u>(p + at, plane, splits);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float v = acc[j] + b[j];
          acc[j] = v > 0.f ? v : 0.f;
          sum += at + j >= c ? static_cast<double>(acc[j]) : 0.0;
        }
        if (at == c) {
          *reinterpret_cast<f32x4_u *>(out + c) = acc;
        } else {
#pragma unroll
          for (int j = 1; j < 4; ++j)
            if (at + j >= c) out[at + j] = acc[j];
        }
      } else {
        for (int j = c; j < n; ++j) {
          float acc = p[j];
          for (int s = 1; s < splits; ++s) acc += p[s * plane + j];
          const float v = acc + bias[j];
          out[j] = v > 0.f ? v : 0.f;
          sum += static_cast<double>(v > 0.f ? v : 0.f);
        }
      }
    }
  }
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) sum += __shfl_xor(sum, o, 64);
  if constexpr (Waves > 1) {
    if (lane == 0) sums[wave] = sum;
    __syncthreads();
    if constexpr (Waves == 4) sum = (sums[0] + sums[1]) + (sums[2] + sums[3]);
    else sum = sums[wave] + sums[wave ^ 1];
  }
  if (lane == 0 && wave % Waves == 0 && row < m) rowsum[row] = static_cast<float>(sum);
}

__global__ __launch_bounds__(256) void zero_tickets_kernel(unsigned *tickets) {
  tickets[blockIdx.x * 256 + threadIdx.x] = 0;
}

}  // namespace

// One block of kSplitWorkspaceBytes and its tickets per (device, stream), allocated at the first call that wants one on
// that stream and kept until the process ends (never grown or freed, so a pointer handed out stays good whatever other threads do):
// calls on different streams never share one, calls on one stream are ordered by it and by the block's lock.  None (the caller then works
// without one: no K split, row sums by atomicAdd) for a stream under capture -- a recorded graph would carry the
// block's address to wherever it is replayed, next to eager calls or other replays that use the same block --, for
// hipStreamPerThread (one handle, a stream to each thread: their launches are not ordered by it), past 16 streams, or when
// the allocation fails.
Workspace splitk_workspace(hipStream_t st) {
  if (st == hipStreamPerThread) return {};
  struct Block {
    float *p;
    std::mutex issuing;
  };
  static std::mutex mu;
  static std::map<std::pair<int, hipStream_t>, Block> blocks;   // (their places do not change)
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return {};
  hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(st, &capturing) != hipSuccess || capturing != hipStreamCaptureStatusNone) {
    (void)hipGetLastError();
    return {};
  }
  std::unique_lock<std::mutex> lock(mu);
  auto it = blocks.find({dev, st});
  if (it != blocks.end()) {
    lock.unlock();   // nobody waits for another stream's call
    return {it->second.p, std::unique_lock<std::mutex>(it->second.issuing)};
  }
  if (blocks.size() >= 16) return {};
  void *p = nullptr;
  if (hipMalloc(&p, kSplitWorkspaceBytes + (kSplitTickets + kFoldTickets) * sizeof(unsigned)) != hipSuccess) {
    (void)hipGetLastError();
    return {};
  }
  hipLaunchKernelGGL(zero_tickets_kernel, dim3((kSplitTickets + kFoldTickets) / 256), dim3(256), 0, st, splitk_tickets(static_cast<float *>(p)));
  Block &block = blocks[{dev, st}];
  block.p = static_cast<float *>(p);
  return {block.p, std::unique_lock<std::mutex>(block.issuing)};
}

int compute_units() {
  static const int cus = [] {
    int dev = 0, v = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || v <= 0)
      v = 256;
    return v;
  }();
  return cus;
}

int launch_splitk_reduce(const float *partials, float *c, int m, int n, int splits, hipStream_t st) {
  const int64_t mn = static_cast<int64_t>(m) * n;
  hipLaunchKernelGGL(splitk_reduce_kernel, dim3(static_cast<unsigned>((mn + 1023) / 1024)), dim3(256), 0, st, partials, c,
                     mn, splitk_plane_floats(m, n), splits);
  return check_launch("split-K reduction launch");
}

int launch_splitk_reduce_fused(const float *partials, const float *bias, float *y, float *rowsum, int m, int n, int splits,
                               hipStream_t st) {
  const int64_t plane = splitk_plane_floats(m, n);
  auto launch = [&]<int Waves>(std::integral_constant<int, Waves>) {
    hipLaunchKernelGGL(splitk_reduce_fused_kernel<Waves>, dim3((m + 4 / Waves - 1) / (4 / Waves)), dim3(256), 0, st, partials, bias, y,
                       rowsum, m, n, plane, splits);
  };
  const int by_columns = n <= 256 ? 1 : n <= 512 ? 2 : 4, by_rows = m < 1280 ? 4 : m <= 2048 || n > 1024 ? 2 : 1;
  const int waves = std::min(by_columns, by_rows);
  if (waves == 4) launch(std::integral_constant<int, 4>{});
  else if (waves == 2) launch(std::integral_constant<int, 2>{});
  else launch(std::integral_constant<int, 1>{});
  return check_launch("split-K reduction launch");
}

}  // namespace sarek_hip
