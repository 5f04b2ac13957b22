// float32 products of up to 6 GFLOP: C[M x N] = A[M x K] . B[K x N] on v_mfma_f32_16x16x4_f32, operands straight from
// memory to registers.
//
// What bounds these products is latency, not a rate: with the 64 x 64 tile of gemm_f32_dma_kernel 512^3 is 64 workgroups
// on 256 CUs, each walking all of K through an LDS ring (two slab latencies before the first MFMA, a barrier per slab).
// Here a tile is 16 MT rows by 64 columns, four to two times as many of them, and the waves of a workgroup take the
// K = 16 steps of their tile in turn, so a wave has K / 16 / kWaves steps, nothing to share with the others and no
// barrier until they add their sums through LDS.  A step is 4 + MT 16-byte loads a lane, one step ahead of 16 MT MFMAs:
//   A: lane (l16, g) of row block t holds row 16 t + l16, k = 4 g .. 4 g + 3;
//   B: load j holds row 4 g + j at columns 4 l16 .. 4 l16 + 3, so that MFMA (j, t, c) multiplies k = 4 g + j, and
//      accumulator c holds columns 4 l16 + c: a lane owns four neighbouring columns of C.
// Against that, 16 MT rows share a load of B where 64 do in the LDS kernel: the operands of all tiles together pass the
// L2 at about 20 TB/s, which is what the larger products run into.  Measured, the LDS kernel against this one, us:
// 128^3 5.1 / 3.5, 256^3 7.1 / 4.0, 512^3 11.0 / 5.4, 640 x 107 x 640 14.5 / 5.7, 68 x 119 x 3328 14.2 / 7.5,
// 1391 x 936 x 1822 66.8 / 47.4, 1024^3 20.1 / 21.2.  Starting each tile at another step of
// K (which the few-rows 16-bit kernel gains from) lost 0 to 20 % here: the tiles that share rows of B then no longer
// read them at the same time.
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "common.hpp"
#include "gemm_common.hpp"

namespace sarek_hip {
namespace {

constexpr int kCols = 64, kStepK = 16;
constexpr int kRedPitch = kCols + 4;

// Workgroup -> (piece of K, tile): every XCD gets a contiguous run of the pieces' tiles, which it walks in bands of
// `band` tile rows, column by column, the band chosen so that the patch of a run is about as tall as wide: the tiles that
// one L2 serves then share their rows of A and columns of B.  Against tiles row by row over all XCDs (us):
// 153 x 1216 x 1920 15.2 to 11.6, 434 x 3952 x 3328 130 to 108.  The divisions are by
// numbers known at the launch, a multiplication by their reciprocals each (divided out they took 0.3 us of a 5 us
// kernel): n / d = floor(n r / 2^32), r = floor(2^32 / d) + 1, is exact while n d < 2^32, so blocks stay under 2^16.
constexpr int kMaxBlocks = 65535;
struct TileMap {
  int tiles_m, tiles_n, band;
  unsigned by_tiles, by_band, by_rows, by_last_rows;   // reciprocals; 0 for 1
};
unsigned reciprocal(int d) { return d == 1 ? 0 : static_cast<unsigned>((1ull << 32) / d + 1); }
__device__ __forceinline__ int divide(int n, unsigned r) {
  return r ? static_cast<int>(__umulhi(static_cast<unsigned>(n), r)) : n;
}

template <int MT, int kWaves>
__global__ __launch_bounds__(64 * kWaves) void gemm_f32_direct_kernel(const float *__restrict__ A, const float *__restrict__ B,
                                                                      float *__restrict__ C, int M, int N, int K, TileMap map,
                                                                      int splits, int steps_per_split,
                                                                      float *__restrict__ partials,
                                                                      unsigned *__restrict__ tickets) {
  __shared__ __attribute__((aligned(16))) float red[kWaves][16 * kRedPitch];
  __shared__ bool last;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l16 = lane & 15, g = lane >> 4;
  const int tiles = map.tiles_m * map.tiles_n, blocks = tiles * splits, xcd = blockIdx.x % NUM_XCD;
  const int id = xcd * (blocks / NUM_XCD) + min(xcd, blocks % NUM_XCD) + static_cast<int>(blockIdx.x / NUM_XCD);
  const int split = divide(id, map.by_tiles), tile = id - split * tiles;
  const int band = divide(tile, map.by_band), in_band = tile - band * map.band * map.tiles_n;
  const int rows = min(map.band, map.tiles_m - band * map.band);
  const int tn = divide(in_band, rows == map.band ? map.by_rows : map.by_last_rows);
  const int m0 = (band * map.band + in_band - tn * rows) * (16 * MT), n0 = tn * kCols;
  const int nsteps = (K + kStepK - 1) / kStepK;
  const int s_begin = split * steps_per_split, s_end = min(nsteps, s_begin + steps_per_split);

  const uint32_t row_bytes = static_cast<uint32_t>(N) * 4;
  const int64_t b_bytes = static_cast<int64_t>(K) * row_bytes;
  const uint32_t b_off = 4 * g * row_bytes + (n0 + 4 * l16) * 4u;
  uint32_t a_off[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) a_off[t] = (static_cast<uint32_t>(min(m0 + 16 * t + l16, M - 1)) * K + 4 * g) * 4u;

  // a step all of whose loads lie inside the matrices; without `ok` the range is empty and nothing is fetched
  auto load = [&](int s, bool ok, f32x4_t (&bf)[4], f32x4_t (&af)[MT]) {
    const uint32_t range = ok ? 0x80000000u : 0u;
    const __amdgpu_buffer_rsrc_t b_rsrc =
        make_rsrc(reinterpret_cast<const char *>(B) + static_cast<int64_t>(s) * kStepK * row_bytes, range);
    const __amdgpu_buffer_rsrc_t a_rsrc = make_rsrc(A + static_cast<int64_t>(s) * kStepK, range);
#pragma unroll
    for (int j = 0; j < 4; ++j)
      bf[j] = __builtin_bit_cast(f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(b_rsrc, b_off, j * row_bytes, 0));
#pragma unroll
    for (int t = 0; t < MT; ++t)
      af[t] = __builtin_bit_cast(f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(a_rsrc, a_off[t], 0, 0));
  };
  // a step at the end of K: B past its last element reads as zero, A's pieces past K are masked
  auto load_end = [&](int s, f32x4_t (&bf)[4], f32x4_t (&af)[MT]) {
    const int64_t at = static_cast<int64_t>(s) * kStepK * row_bytes;
    const __amdgpu_buffer_rsrc_t b_rsrc =
        make_rsrc(reinterpret_cast<const char *>(B) + at,
                  static_cast<uint32_t>(min(b_bytes - at, static_cast<int64_t>(0x7FFFFFFF))));
    const __amdgpu_buffer_rsrc_t a_rsrc =
        make_rsrc(A + static_cast<int64_t>(s) * kStepK, static_cast<uint32_t>((static_cast<int64_t>(M) * K - s * kStepK) * 4));
    const int left = K - s * kStepK - 4 * g;
#pragma unroll
    for (int j = 0; j < 4; ++j)
      bf[j] = __builtin_bit_cast(f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(b_rsrc, b_off + j * row_bytes, 0, 0));
#pragma unroll
    for (int t = 0; t < MT; ++t) {
      u32x4 v = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(a_rsrc, a_off[t], 0, 0));
#pragma unroll
      for (int d = 0; d < 4; ++d) v[d] = left > d ? v[d] : 0u;
      af[t] = __builtin_bit_cast(f32x4_t, v);
    }
  };

  f32x4_t acc[MT][4];
#pragma unroll
  for (int t = 0; t < MT; ++t)
#pragma unroll
    for (int c = 0; c < 4; ++c) acc[t][c] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  auto multiply = [&](f32x4_t (&bf)[4], f32x4_t (&af)[MT]) {
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int c = 0; c < 4; ++c) acc[t][c] = __builtin_amdgcn_mfma_f32_16x16x4f32(af[t][j], bf[j][c], acc[t][c], 0, 0, 0);
  };

  // The pieces of B past column N run into the rows below, so the last rows of B belong to the end.
  const int64_t plain_rows = K - (kCols + N - 1) / N;
  const int plain = max(min(s_end, plain_rows > 0 ? static_cast<int>(plain_rows / kStepK) : 0) - s_begin, 0);
  f32x4_t bf[2][4], af[2][MT];
  auto load_at = [&](int i, auto buffer) { load(s_begin + i, i < plain, bf[buffer], af[buffer]); };
  constexpr std::integral_constant<int, 0> b0{};
  constexpr std::integral_constant<int, 1> b1{};
  load_at(wave, b0);
  for (int i = wave; i < plain; i += 2 * kWaves) {
    load_at(i + kWaves, b1);
    multiply(bf[0], af[0]);
    load_at(i + 2 * kWaves, b0);
    multiply(bf[1], af[1]);
  }
  for (int s = s_begin + plain + wave; s < s_end; s += kWaves) {
    load_end(s, bf[0], af[0]);
    multiply(bf[0], af[0]);
  }

  const int row = (threadIdx.x & 255) >> 4, col = (threadIdx.x & 15) * 4;   // threads 0 .. 255
  static_assert(kWaves >= 4);
  auto put = [&](int t, f32x4_t v) {
    const int m = m0 + 16 * t + row, n = n0 + col;
    if (m >= M) return;
    float *dst = C + static_cast<int64_t>(m) * N + n;
    if (n + 4 <= N) {
      *reinterpret_cast<f32x4_u *>(dst) = v;
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (n + j < N) dst[j] = v[j];
    }
  };
  const int plane_bytes = tiles * (MT * 16 * kCols * 4);
  const __amdgpu_buffer_rsrc_t p_rsrc =
      make_rsrc(partials + static_cast<int64_t>(tile) * (MT * 16 * kCols), 0x80000000u);
  const int piece = (row * kCols + col) * 4;
  // The sums of the waves, added in the order of the waves; cut along K the tile goes to its plane instead of C, past
  // the XCD's L2, and the workgroup that draws a tile's last ticket adds the planes in their order: the same bits on
  // every run, and no second launch (5 us against 1 to 2).
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    if (t > 0) __syncthreads();
#pragma unroll
    for (int r = 0; r < 4; ++r)
      *reinterpret_cast<f32x4_t *>(&red[wave][(4 * g + r) * kRedPitch + 4 * l16]) =
          f32x4_t{acc[t][0][r], acc[t][1][r], acc[t][2][r], acc[t][3][r]};
    __syncthreads();
    if (threadIdx.x < 256) {
      f32x4_t v = *reinterpret_cast<const f32x4_t *>(&red[0][row * kRedPitch + col]);
#pragma unroll
      for (int w = 1; w < kWaves; ++w) v += *reinterpret_cast<const f32x4_t *>(&red[w][row * kRedPitch + col]);
      if (splits == 1) put(t, v);
      else
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), p_rsrc, piece + t * (16 * kCols * 4),
                                               split * plane_bytes, kDeviceScope);
    }
  }
  if (splits == 1) return;
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (threadIdx.x == 0)
    last = __hip_atomic_fetch_add(tickets + tile, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) ==
           static_cast<unsigned>(splits - 1);
  __syncthreads();
  if (!last) return;
  if (threadIdx.x < 256) {
    f32x4_t sum[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t) sum[t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    for (int q = 0; q < splits; q += 4) {
      f32x4_t v[4][MT];
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int t = 0; t < MT; ++t)
          v[u][t] = __builtin_bit_cast(
              f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(p_rsrc, piece + t * (16 * kCols * 4),
                                                             min(q + u, splits - 1) * plane_bytes, kDeviceScope));
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (q + u < splits) {
#pragma unroll
          for (int t = 0; t < MT; ++t) sum[t] += v[u][t];
        }
    }
#pragma unroll
    for (int t = 0; t < MT; ++t) put(t, sum[t]);
  }
  if (threadIdx.x == 0) __hip_atomic_store(tickets + tile, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

template <int MT, int W>
int launch(const float *a, const float *b, float *c, int m, int n, int k, int splits, float *partials, hipStream_t st) {
  const int tiles_m = (m + 16 * MT - 1) / (16 * MT), tiles_n = (n + kCols - 1) / kCols, steps = (k + kStepK - 1) / kStepK;
  if (!partials) splits = 1;
  const int per = (steps + splits - 1) / splits;
  const double run = std::min(1.0, splits / static_cast<double>(NUM_XCD)) * tiles_m * tiles_n;
  const int band = std::max(1, std::min(tiles_m, static_cast<int>(std::lround(std::sqrt(run * kCols / (16 * MT))))));
  const TileMap map{tiles_m, tiles_n, band, reciprocal(tiles_m * tiles_n), reciprocal(band * tiles_n), reciprocal(band),
                    reciprocal(tiles_m % band ? tiles_m % band : band)};
  hipLaunchKernelGGL((gemm_f32_direct_kernel<MT, W>), dim3(static_cast<unsigned>(tiles_m) * tiles_n * splits), dim3(64 * W),
                     0, st, a, b, c, m, n, k, map, splits, per, partials, partials ? splitk_tickets(partials) : nullptr);
  return check_launch("gemm_f32 direct kernel launch");
}

}  // namespace

// 16 rows of B and the whole of A lie within 32-bit offsets, and the tiles can be numbered.
bool gemm_f32_direct_serves(int m, int n, int k) {
  const int64_t tiles = static_cast<int64_t>((m + 15) / 16) * ((n + kCols - 1) / kCols);
  return tiles <= kMaxBlocks && static_cast<int64_t>(m) * k * 4 < 0x7FFFFFFF && static_cast<int64_t>(n) * 2 * kStepK * 4 < 0x7FFFFFFF;
}

// Up to 6 GFLOP: above, the LDS kernel with its last tiles cut is level or ahead (1280 x 1644 x 960, 4 GFLOP: 41 us here, 36
// there; 1500^3, 7: 62 and 57; 2049 x 4097 x 3000, 50: 408 and 388).  Up to 10 where tiles cannot be cut.
bool gemm_f32_direct_pays(int m, int n, int k, bool cuts) { return static_cast<double>(m) * n * k <= (cuts ? 3e9 : 5e9); }

// At most `splits` pieces of K: of whole steps, none empty, their planes within the workspace and a ticket per tile.
int gemm_f32_direct_pieces(int m, int n, int k, int row_blocks, int splits) {
  const int64_t tiles = static_cast<int64_t>((m + 16 * row_blocks - 1) / (16 * row_blocks)) * ((n + kCols - 1) / kCols);
  if (tiles > kSplitTickets) return 1;
  const int64_t fit = static_cast<int64_t>(kSplitWorkspaceBytes) / (tiles * (16 * row_blocks * kCols * 4));
  const int steps = (k + kStepK - 1) / kStepK;
  splits = static_cast<int>(std::max<int64_t>(1, std::min<int64_t>({splits, steps, fit, kMaxBlocks / tiles})));
  const int per = (steps + splits - 1) / splits;
  return (steps + per - 1) / per;
}

// Estimated time in us: of the terms below, with weights fitted to 135 drawn products of 0 to 80 GFLOP on which each
// variant was timed with 1 to 8 pieces (5 % rms).  A launch; the MFMAs of the CU with the most workgroups, against the
// chain of one wave (a step's loads take 0.28 us a row block to come, two steps in flight); the operands of all tiles
// through the L2s, at 24 TB/s; the sum over the waves; A and B once, and the stores of C; and, cut along K, the planes out and in and the
// wait for the last workgroup.
double gemm_f32_direct_estimate(int m, int n, int k, int row_blocks, int waves, int splits) {
  const double tiles = static_cast<double>((m + 16 * row_blocks - 1) / (16 * row_blocks)) * ((n + kCols - 1) / kCols);
  const int steps = (k + kStepK - 1) / kStepK, per = (steps + splits - 1) / splits;
  const double rounds = std::ceil(tiles * splits / compute_units()), wave_steps = (per + waves - 1) / waves;
  auto square = [](double x) { return x * x; };
  const double mfma = 0.0543 * rounds * per * row_blocks, chain = 0.28 * wave_steps * row_blocks;
  const double issue = std::sqrt(std::sqrt(square(square(mfma)) + square(square(chain))));
  const double operands = 0.0418 * tiles * k * (16 * row_blocks + kCols) * 4e-6;
  double us = 3.33 + std::cbrt(issue * issue * issue + operands * operands * operands) + 0.04 * wave_steps +
              0.06 * rounds * row_blocks * waves + 4e-6 * (0.018 * (static_cast<double>(m) + n) * k + 0.24 * m * n);
  if (splits > 1) us += 0.65 + 0.101 * tiles * splits * row_blocks * 8192e-6 + 0.131 * splits * row_blocks;
  return us;
}

int launch_gemm_f32_direct(const float *a, const float *b, float *c, int m, int n, int k, int row_blocks, int waves,
                           int splits, float *partials, hipStream_t st) {
  if (row_blocks == 2) return launch<2, 4>(a, b, c, m, n, k, splits, partials, st);
  if (waves == 8) return launch<1, 8>(a, b, c, m, n, k, splits, partials, st);
  return launch<1, 4>(a, b, c, m, n, k, splits, partials, st);
}

}  // namespace sarek_hip
