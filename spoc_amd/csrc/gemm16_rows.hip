// 16-bit-input (bf16 / fp16), f32-accumulate products in tiles of at most 64 rows:  C[M x N] = A[M x K] . B[K x N],
// row-major; for the fp16 product with bias, ReLU and row sums as well.
//
// What bounds it: B is read once and used M times, so the product is a read of B (16 x 8192 x 8192: 134 MB, 21 us at the
// 6.3 TB/s large streams reach here) and a CU draws at most about 39 GB/s of L2 misses, so every CU has to take its
// share.  The 128 x 128 tile of gemm16_m16_small_kernel fetches 128 rows of A whatever M is and adds its K pieces in a
// second launch.  Here:
//   - No LDS on the way in.  A wave takes steps of 32 k x 128 columns of B, 8 KiB in eight 16-byte loads per lane: lane
//     (l, g) = (lane % 16, lane / 16) gets rows 8g .. 8g+7 at columns 8l .. 8l+7.  v_perm_b32 turns that 8 x 8 block into
//     eight operands of v_mfma_f32_16x16x32 (column 8l + c over k = 8g .. 8g+7, c = 0 .. 7), four instructions each; A's
//     rows are the other operand, read as they lie.  The result puts 32 consecutive columns of one row of C in a lane.
//   - The eight waves of a workgroup take the steps of its piece of K in turn, two in flight each, and add up through LDS.
//   - K is cut over `splits` workgroups per column tile; each leaves its sums in a plane of the stream's workspace, past
//     the L2s, and the one that takes a tile's last ticket adds the planes in order.  The order of all additions is fixed:
//     the same bits on every run.
//   - Workgroups start at different places of their piece: A's rows are a power of two apart in the usual case, and in
//     step all workgroups would read them from the same L2 channels (64 x 8192 x 8192: 51 us in step, 38 rotated).
// Measured, before (the 128 x 128 tile, which then took the last column of an odd N in a launch of its own) and now, launches back to back on rotating operands:
//   16 x 8192 x 8192 34.5 -> 25.7 us (5.2 TB/s), 16 x 2048 x 2048 10.4 -> 6.8, 16 x 40000 x 1024 21.1 -> 19.6,
//   32 x 16384 x 4096 32.9 -> 27.4, 48 x 4096 x 4096 17.2 -> 13.8, 16 x 256 x 8192 12.8 -> 7.4; odd sizes:
//   10 x 4161 x 4221 80 -> 12.6, 64 x 4097 x 4103 74 -> 20.5, 8 x 50257 x 1024 34.5 -> 28.0.
// More rows are more row tiles.  Where all tiles find a CU of their own the product is bound by the latency of its steps,
// not by what is read, and the 128 x 128 tile has one wave per SIMD to hide it and, with the fused epilogue, no K pieces:
//   77 x 2332 x 1920 22.7 -> 10.0, 97 x 1633 x 1090 16.1 -> 11.0; fused 220 x 256 x 4444 47.8 -> 16.0,
//   537 x 259 x 3648 40.7 -> 18.0, 214 x 1088 x 3264 25.3 -> 17.1, 224 x 256 x 2368 18.9 -> 14.4.
// Tried: 4 waves with 2 to 4 steps in flight (5 to 10 % slower), tiles dealt so that neighbours share an XCD (no change),
// 64-bit atomic stores and loads for the planes (4 planes of 64 x 8192: 3 us more than the 16-byte accesses).
#include <algorithm>
#include <cmath>
#include <type_traits>
#include <utility>

#include "common.hpp"
#include "gemm_common.hpp"
#include "tunables.hpp"

namespace sarek_hip {
namespace {

constexpr int kTileRows = 64, kCols = 128, kStepK = 32, kWaves = 8;
constexpr int kRedPitch = kCols + 4;   // floats per row of the waves' sums in LDS: 16 rows on different banks
constexpr int kNonTemporal = 2;   // cache policy of a buffer access

template <bool Bf16, int MT, int BPolicy, bool Fused>
__global__ __launch_bounds__(64 * kWaves) void gemm16_rows_kernel(const uint16_t *__restrict__ A,
                                                                  const uint16_t *__restrict__ B, float *__restrict__ C,
                                                                  const float *__restrict__ bias,
                                                                  float *__restrict__ rowsum, int M, int N, int K,
                                                                  int row_tiles, int col_tiles, int splits,
                                                                  int steps_per_split, float *__restrict__ rs_planes,
                                                                  float *__restrict__ partials,
                                                                  unsigned *__restrict__ tickets, RowFold fold) {
  __shared__ __attribute__((aligned(16))) float red[kWaves][16 * kRedPitch];
  __shared__ bool last;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l16 = lane & 15, g = lane >> 4;
  // The row tiles of a column tile read the same piece of B: they are neighbours in an XCD's run of workgroups.
  int index = blockIdx.x;
  if (row_tiles > 1) {
    const int xcd = index % NUM_XCD, nb = gridDim.x;
    index = xcd * (nb / NUM_XCD) + min(xcd, nb % NUM_XCD) + index / NUM_XCD;
  }
  const int row_tile = index % row_tiles, col_tile = index / row_tiles % col_tiles;
  const int split = index / (row_tiles * col_tiles);
  const int tile = col_tile * row_tiles + row_tile, tiles = row_tiles * col_tiles;
  const int n0 = col_tile * kCols, m0 = row_tile * (16 * MT);
  A += static_cast<int64_t>(m0) * K;
  M -= m0;   // from here on rows count from the tile's first
  C += static_cast<int64_t>(m0) * N;

  const int nsteps = (K + kStepK - 1) / kStepK;
  const int s_begin = split * steps_per_split, s_end = min(nsteps, s_begin + steps_per_split);

  const uint32_t row_bytes = static_cast<uint32_t>(N) * 2;
  const int64_t b_bytes = (static_cast<int64_t>(K) * N - (N & 1)) * 2;   // see load_end
  const uint32_t b_off = 8 * g * row_bytes + (n0 + 8 * l16) * 2u;
  uint32_t a_off[MT];   // rows past M repeat the last one: what they produce is never stored
#pragma unroll
  for (int t = 0; t < MT; ++t) a_off[t] = (static_cast<uint32_t>(min(16 * t + l16, M - 1)) * K + 8 * g) * 2u;

  // A step whose loads all lie inside A and B (columns past N bring the next rows' elements, and are never stored).
  // !ok: the resources have no range, so every load returns zeros and fetches nothing; it keeps the count of loads in
  // flight the same in every turn of the loop.
  auto load = [&](int s, bool ok, u32x4 (&bf)[8], u32x4 (&af)[MT]) {
    const uint32_t range = ok ? 0x80000000u : 0u;
    const __amdgpu_buffer_rsrc_t b_rsrc =
        make_rsrc(reinterpret_cast<const char *>(B) + static_cast<int64_t>(s) * kStepK * row_bytes, range);
    const __amdgpu_buffer_rsrc_t a_rsrc = make_rsrc(A + static_cast<int64_t>(s) * kStepK, range);
#pragma unroll
    for (int i = 0; i < 8; ++i)
      bf[i] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(b_rsrc, b_off, i * row_bytes, BPolicy));
#pragma unroll
    for (int t = 0; t < MT; ++t)
      af[t] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(a_rsrc, a_off[t], 0, 0));
  };
  // A step at the end of B: B's range is exact, so what lies past it reads as zero; elements of A past K count as zero.
  auto load_end = [&](int s, u32x4 (&bf)[8], u32x4 (&af)[MT]) {
    const int64_t at = static_cast<int64_t>(s) * kStepK * row_bytes;
    const __amdgpu_buffer_rsrc_t b_rsrc =
        make_rsrc(reinterpret_cast<const char *>(B) + at,
                  static_cast<uint32_t>(min(b_bytes - at, static_cast<int64_t>(0x7FFFFFFF))));
#pragma unroll
    for (int i = 0; i < 8; ++i)
      bf[i] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(b_rsrc, b_off + i * row_bytes, 0, 0));
    const int left = K - s * kStepK - 8 * g;   // elements of A this lane has before the end of K
    const __amdgpu_buffer_rsrc_t a_rsrc =
        make_rsrc(A + static_cast<int64_t>(s) * kStepK,
                  static_cast<uint32_t>(min((static_cast<int64_t>(M) * K - (K & 1) - s * kStepK) * 2,
                                            static_cast<int64_t>(0x7FFFFFFF))));
#pragma unroll
    for (int t = 0; t < MT; ++t) {
      af[t] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(a_rsrc, a_off[t], 0, 0));
#pragma unroll
      for (int d = 0; d < 4; ++d) af[t][d] &= left >= 2 * d + 2 ? 0xFFFFFFFFu : left == 2 * d + 1 ? 0xFFFFu : 0u;
    }
    // with an odd K the dword that holds A[M-1][K-1] ends past A: the range ends in front of it, it read as zero ...
    if ((K & 1) != 0 && s == nsteps - 1) {
      const uint32_t v = A[static_cast<int64_t>(M) * K - 1];
#pragma unroll
      for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int d = 0; d < 4; ++d)
          if (16 * t + l16 >= M - 1 && left == 2 * d + 1) af[t][d] = v;
    }
    // ... and with an odd N the one that holds B[K-1][N-1] past B
    if ((N & 1) != 0 && s == nsteps - 1) {
      const int r = K - 1 - s * kStepK, c = N - 1 - n0;   // row in the step, column in the tile
      if (g == r / 8 && c >= 0 && l16 == c / 8) {
        const uint32_t v = B[static_cast<int64_t>(K - 1) * N + N - 1];
#pragma unroll
        for (int i = 0; i < 8; ++i)
#pragma unroll
          for (int d = 0; d < 4; ++d)
            if (i == r % 8 && d == (c % 8) / 2) bf[i][d] = v;
      }
    }
  };

  f32x4_t acc[8][MT];
#pragma unroll
  for (int c = 0; c < 8; ++c)
#pragma unroll
    for (int t = 0; t < MT; ++t) acc[c][t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  auto multiply = [&](u32x4 (&bf)[8], u32x4 (&af)[MT]) {
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      u32x4 op;
#pragma unroll
      for (int d = 0; d < 4; ++d)
        op[d] = __builtin_amdgcn_perm(bf[2 * d + 1][c / 2], bf[2 * d][c / 2], c % 2 ? 0x07060302u : 0x05040100u);
#pragma unroll
      for (int t = 0; t < MT; ++t) acc[c][t] = mfma16<Bf16>(op, af[t], acc[c][t]);
    }
  };

  // The piece's plain steps: whole K, and at least one tile's width of B behind their last row's first element
  const int64_t plain_rows = K - (kCols + N - 1) / N;
  const int plain = max(min(s_end, plain_rows > 0 ? static_cast<int>(plain_rows / kStepK) : 0) - s_begin, 0);
  const int first = plain > 0 ? (col_tile * kWaves) % plain : 0;
  u32x4 bf[2][8], af[2][MT];
  auto load_at = [&](int i, auto buffer) {
    const int at = i + first;
    load(s_begin + (at < plain ? at : at - plain), i < plain, bf[buffer], af[buffer]);
  };
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

  // Sums over the waves, 16 rows at a time: thread -> row `row`, columns col .. col + 3 of them
  const int row = threadIdx.x >> 5, col = (threadIdx.x & 31) * 4;
  // (Fused: bias, ReLU, and the row's sum over the tile's columns, added by the 32 lanes that hold it, to its plane)
  f32x4_t bias4 = {0.f, 0.f, 0.f, 0.f};
  if constexpr (Fused) {
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (n0 + col + j < N) bias4[j] = bias[n0 + col + j];
  }
  auto put = [&](int t, f32x4_t v) {
    const int m = 16 * t + row, n = n0 + col;
    if constexpr (Fused) {
      float sum = 0.f;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        v[j] += bias4[j];
        v[j] = v[j] > 0.f ? v[j] : 0.f;
        sum += n + j < N ? v[j] : 0.f;
      }
#pragma unroll
      for (int o = 16; o >= 1; o >>= 1) sum += __shfl_xor(sum, o, 64);
      if (m < M && (lane & 31) == 0) {
        if (rs_planes && !fold.tickets)
          rs_planes[static_cast<int64_t>(col_tile) * (M + m0) + m0 + m] = sum;
        else if (rs_planes)
          __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(sum), make_rsrc(rs_planes, 0x7FFFFFFFu),
                                                (col_tile * (M + m0) + m0 + m) * 4, 0, kDeviceScope);
        else
          atomicAdd(rowsum + m0 + m, sum);
      }
    }
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
  // plane `split`: per tile 16 MT rows of kCols
  const int plane_bytes = tiles * (MT * 16 * kCols * 4);
  const __amdgpu_buffer_rsrc_t p_rsrc =
      make_rsrc(partials + static_cast<int64_t>(tile) * (MT * 16 * kCols), 0x80000000u);
  const int piece = (row * kCols + col) * 4;
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    if (t > 0) __syncthreads();
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int h = 0; h < 2; ++h)
        *reinterpret_cast<f32x4_t *>(&red[wave][l16 * kRedPitch + 32 * g + 8 * r + 4 * h]) =
            f32x4_t{acc[4 * h][t][r], acc[4 * h + 1][t][r], acc[4 * h + 2][t][r], acc[4 * h + 3][t][r]};
    __syncthreads();
    f32x4_t v = *reinterpret_cast<const f32x4_t *>(&red[0][row * kRedPitch + col]);
#pragma unroll
    for (int w = 1; w < kWaves; ++w) v += *reinterpret_cast<const f32x4_t *>(&red[w][row * kRedPitch + col]);
    if (splits == 1) put(t, v);
    else
      __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), p_rsrc, piece + t * (16 * kCols * 4),
                                             split * plane_bytes, kDeviceScope);
  }
  auto fold_here = [&] {
    if constexpr (Fused) {
      if (fold.tickets) fold_rows<64 * kWaves, kTileRows>(fold, M + m0, m0, 16 * MT, rowsum, row_tile, col_tiles, &red[0][0]);
    }
  };
  if (splits == 1) {
    fold_here();
    return;
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // every wave's pieces are where the other XCDs read them
  __syncthreads();
  if (threadIdx.x == 0)
    last = __hip_atomic_fetch_add(tickets + tile, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) ==
           static_cast<unsigned>(splits - 1);
  __syncthreads();
  if (!last) return;
  f32x4_t sum[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) sum[t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  for (int q = 0; q < splits; q += 4) {   // four planes asked for before the first is added
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
  if (threadIdx.x == 0) __hip_atomic_store(tickets + tile, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  fold_here();
}

// Rows per tile: as few tiles of at most 64 as there can be, of equal height, in blocks of 16.
inline int row_blocks_for(int m) {
  const int tiles = (m + kTileRows - 1) / kTileRows;
  return ((m + tiles - 1) / tiles + 15) / 16;
}

struct Shape {
  int mt, row_tiles, col_tiles, steps;
  int64_t tiles, plane, rs_floats;   // bytes of a partial plane; floats of the row sums' planes, whole 256-byte pieces
};
inline Shape shape_of(int m, int n, int k, bool fused) {
  Shape s;
  s.mt = row_blocks_for(m);
  s.row_tiles = (m + 16 * s.mt - 1) / (16 * s.mt);
  s.col_tiles = (n + kCols - 1) / kCols;
  s.steps = (k + kStepK - 1) / kStepK;
  s.tiles = static_cast<int64_t>(s.row_tiles) * s.col_tiles;
  s.plane = s.tiles * s.mt * 16 * kCols * 4;
  s.rs_floats = fused ? (static_cast<int64_t>(s.col_tiles) * m + 63) / 64 * 64 : 0;
  return s;
}

double rows_time(const Shape &s, int n, int k, int64_t splits) {
  const int cus = compute_units();
  const double memory = static_cast<double>(k) * n * 2 / 6.3e6;
  const double cu = static_cast<double>((s.tiles * splits + cus - 1) / cus) * s.steps / splits * (8192 + 1024 * s.mt) / 39e3;
  return std::cbrt(cu * cu * cu + memory * memory * memory) +
         (splits > 1 ? 1.0 + 0.15 * splits + 2.0 * static_cast<double>(splits * s.plane) / 2.7e6 : 0.0);
}

// Pieces of K per tile, by an estimate in microseconds whose constants were fitted to sweeps of 1 to 31 pieces
// over 12 shapes (within 1 us on those of 10 us and more): a CU's share of B and A at 39 GB/s in whole rounds of
// workgroups, B from memory at 6.3 TB/s, the two merged smoothly; a split adds its planes, written and read at 2.7 TB/s,
// a ticket, and a little per piece.  A wave keeps at least one step.  gemm16.rows_splits: 0 = this rule, n forces n.
int rows_splits_for(const Shape &s, int n, int k) {
  const int64_t fit = s.tiles > kSplitTickets
                          ? 1
                          : (static_cast<int64_t>(kSplitWorkspaceBytes) - s.rs_floats * 4) / s.plane;
  const int64_t forced = tunable("gemm16.rows_splits", 0);
  int64_t splits = 1;
  if (forced > 0) {
    splits = std::max<int64_t>(1, std::min<int64_t>({forced, s.steps, fit}));
  } else {
    double best = rows_time(s, n, k, 1);
    for (int64_t t = 2; t <= 64 && t <= fit && t * kWaves <= s.steps; ++t)
      if (rows_time(s, n, k, t) < best) best = rows_time(s, n, k, t), splits = t;
  }
  const int64_t per = (s.steps + splits - 1) / splits;   // the count follows from the piece so that none is empty
  return static_cast<int>((s.steps + per - 1) / per);
}

struct Call {
  const uint16_t *a, *b;
  float *c;
  const float *bias;
  float *rowsum;
  int m, n, k;
  hipStream_t st;
};

template <bool Bf16, bool Fused, int MT>
int launch(const Call &q, const Shape &s) {
  int splits = rows_splits_for(s, q.n, q.k);
  Workspace workspace;
  if (Fused || splits > 1) workspace = splitk_workspace(q.st);
  float *const block = workspace.block;
  if (!block) splits = 1;
  const int per = (s.steps + splits - 1) / splits;
  float *rs_planes = nullptr;
  if constexpr (Fused) {
    if (s.rs_floats * 4 <= static_cast<int64_t>(kSplitWorkspaceBytes)) rs_planes = block;
    if (!rs_planes) {
      const int rc = launch_zero_f32(q.rowsum, q.m, q.st);
      if (rc != SAREK_HIP_OK) return rc;
    }
  }
  RowFold fold{rs_planes, s.col_tiles, nullptr};
  // The last workgroup of a row of tiles adds the planes (fold_rows) while the tiles are few: the more, the longer their shares and
  // counts take to come together, the longer with more rows (us, rowsum_fold_kernel's launch and here, K of 512: 4 x 512 10.5 and
  // 7.3, 4 x 16384 9.7 and 8.2, 4 x 32768 10.4 and 11.9, 128 x 2048 11.4 and 11.3, 128 x 8192 11.8 and 12.8, 2000 x 512 12.3 and
  // 12.2, 1000 x 1024 12.3 and 12.8).  gemm16.fold: 0 = this rule, 1 = never, 2 = always.
  const int64_t asked = Fused ? tunable("gemm16.fold", 0) : 1;
  if (rs_planes && s.row_tiles <= kFoldTickets && asked != 1 &&
      (asked == 2 || s.tiles <= (s.mt <= 2 ? 128 : 64) || s.tiles * s.col_tiles <= 512))
    fold.tickets = fold_tickets(block);
  float *partials = splits > 1 ? block + s.rs_floats : nullptr;
  unsigned *tickets = splits > 1 ? splitk_tickets(block) : nullptr;
  // B past the caches from 64 MiB on where its rows are whole 128-byte lines (100 MB: 20.2 us against 22.8, 134 MB: 26.4
  // against 28.0, 34 MB: 15.8 against 13.2); rows at other offsets share lines between neighbouring loads, and lose
  // (16 x 30000 x 4096 53.1 against 49.9, 8 x 24632 x 3072 35.2 and 33.4, 16 x 22000 x 1536 18.2 and 17.5, operands new to the
  // caches), and so does what several row tiles read
  const bool nt = s.row_tiles == 1 && q.n % 64 == 0 && static_cast<int64_t>(q.k) * q.n * 2 > (int64_t{64} << 20);
  const dim3 grid(static_cast<unsigned>(s.tiles * splits)), block_dim(64 * kWaves);
  if (nt)
    hipLaunchKernelGGL((gemm16_rows_kernel<Bf16, MT, kNonTemporal, Fused>), grid, block_dim, 0, q.st, q.a, q.b, q.c, q.bias,
                       q.rowsum, q.m, q.n, q.k, s.row_tiles, s.col_tiles, splits, per, rs_planes, partials, tickets, fold);
  else
    hipLaunchKernelGGL((gemm16_rows_kernel<Bf16, MT, 0, Fused>), grid, block_dim, 0, q.st, q.a, q.b, q.c, q.bias,
                       q.rowsum, q.m, q.n, q.k, s.row_tiles, s.col_tiles, splits, per, rs_planes, partials, tickets, fold);
  const int rc = check_launch("gemm16 few-rows kernel launch");
  if (!rs_planes || fold.tickets || rc != SAREK_HIP_OK) return rc;
  return launch_rowsum_fold(rs_planes, s.col_tiles, q.m, q.rowsum, q.st);
}

template <bool Bf16, bool Fused>
int launch_rows(const Call &q) {
  const Shape s = shape_of(q.m, q.n, q.k, Fused);
  switch (s.mt) {
    case 1: return launch<Bf16, Fused, 1>(q, s);
    case 2: return launch<Bf16, Fused, 2>(q, s);
    case 3: return launch<Bf16, Fused, 3>(q, s);
    default: return launch<Bf16, Fused, 4>(q, s);
  }
}

}  // namespace

// Whether this kernel can take a product: rows of B of at least a pair of elements (load_end counts on it), K of at least
// one step, 32 rows of B and 64 of A within the 32-bit load offsets.
bool gemm16_rows_serves(int m, int n, int k) {
  return m >= 1 && n >= 2 && k >= kStepK && static_cast<int64_t>(n + kCols) * 2 * kStepK < 0x7FFFFFFF &&
         static_cast<int64_t>(kTileRows) * k * 2 < 0x7FFFFFFF && shape_of(m, n, k, false).tiles * 64 < 0x7FFFFFFF;
}

// Microseconds of a product of 17 to 64 rows whose B is new to the caches, by an estimate read off 800 drawn ones (9 % rms): the steps of the CU with the
// most workgroups by how A's and B's rows lie, against B from memory (whose stream the registers of more row blocks leave
// fewer loads in flight), and the sums.  coarse: B's share by how A's rows lie too.
double narrow_time(const Shape &s, int n, int k, int splits, bool coarse = false) {
  const int align = k % 8 == 0 && n % 8 == 0 ? 0 : k % 2 == 0 && n % 2 == 0 ? 1 : 2, b_align = coarse ? align : n % 8 == 0 ? 0 : 1 + n % 2;
  constexpr double kStep[] = {0.0125, 0.0147, 0.0288}, kMegabyte[] = {0.124, 0.147, 0.164};
  const double rounds = static_cast<double>((s.tiles * splits + compute_units() - 1) / compute_units());
  const double steps = rounds * s.steps / splits * kStep[align] * (4.0 + s.mt);
  const double memory = static_cast<double>(k) * n * 2e-6 * kMegabyte[b_align] * (1 + 0.182 * s.mt);
  return 2.94 + 0.97 * s.mt * rounds + std::cbrt(steps * steps * steps + memory * memory * memory) +
         (splits > 1 ? 1.17 + 0.31 * splits : 0.0);
}

// What does not go by estimates.  Up to 16 rows always here, but for more than 128 MiB of B in one piece of K whose rows, of an even N, share
// lines: there the tile's transfers into LDS come in better (16 x 30000 x 4096 43.2 on the tile, 49.9 here; elsewhere the tile was
// the faster by 4 % on 4 of 400 drawn products, operands new to the caches, this kernel by a quarter on average).  To 64 a workgroup's
// sums through LDS cost it 0.5 us per 16 rows and its registers leave room for one workgroup per CU, so short K and more
// column tiles than CUs belong to the 128 x 128 tile unless N is odd (us, 128 tile / here):
//   32 x 512 x 64 4.8 / 4.0, 32 x 4096 x 4096 15.7 / 12.0, 32 x 40000 x 1024 22.0 / 23.8, 32 x 40001 x 1024 34.5 / 29.9
//   48 x 4096 x 256 6.2 / 6.1, 48 x 4096 x 1024 10.2 / 9.4, 48 x 40000 x 1024 23.0 / 26.4, 48 x 40001 x 1024 35.3 / 33.4
//   64 x 4096 x 256 6.4 / 7.2, 64 x 4096 x 1024 10.5 / 10.5, 64 x 4096 x 4096 17.3 / 15.6, 64 x 40001 x 1024 36.3 / 37.0
// An odd N of up to 8 column tiles stays here (49 x 255 x 4129 13.5 / 15.1, 64 x 1001 x 1001 15.7 / 11.4), 17 to 32 rows against up to 96
// column tiles do (one of 576 more than 10 % slower), and so does a product whose pieces gemm16.rows_splits sets.  Beyond 64 rows, and with
// the fused epilogue at any number, its tiles have to fit the CUs in one round (882 x 2401 x 4259, 266 tiles: 50 us on the other tile, 108
// here) and half of the waves to have a step at least (in tiles of 64 rows some wave two: 256 x 1280 x 191 6.8 / 8.4, 723 x 1702 x 256 7.2 /
// 7.9, as 21 of 118 drawn products, all but 3 of them so short).
enum class Kernel { rows, tile, by_estimate };
bool narrow_counts(const Shape &s, int m, int n) {
  return m > 16 && m <= kTileRows && s.col_tiles > (s.mt == 2 ? 96 : n % 2 != 0 ? 8 : 0) && tunable("gemm16.rows_splits", 0) == 0;
}
Kernel outright(const Shape &s, int m, int n, int k, bool fused) {
  if (m > kTileRows || fused)
    return s.tiles > compute_units() || 2 * s.steps < kWaves || (s.mt == 4 && s.steps <= kWaves) ? Kernel::tile : Kernel::by_estimate;
  const bool odd = n % 2 != 0, one_round = s.col_tiles <= compute_units();
  bool here = true;
  switch (s.mt) {
    case 1:
      here = n % 64 == 0 || odd || static_cast<int64_t>(k) * n * 2 <= (int64_t{128} << 20) || rows_splits_for(s, n, k) > 1 ||
             tunable("gemm16.rows_splits", 0) != 0;
      return here ? Kernel::rows : Kernel::tile;
    case 2: here = odd || one_round; break;
    case 3: here = one_round ? odd || k >= 512 : odd && k >= 1024; break;
    default: here = one_round && (odd || k >= 1024);
  }
  return !here ? Kernel::tile : narrow_counts(s, m, n) ? Kernel::by_estimate : Kernel::rows;
}

// The same by coarser estimates of both kernels, that put this one up to 2 us too low, of the tile in 1 to 16 pieces of a plain product,
// powers of two: what decides where the tile would be the less exact, and where a product cannot be cut.  pieces_asked: it is about pieces
// of more than 2048 of K, for which this kernel is not left where its finer estimate of 17 to 64 rows has it ahead.
bool coarsely_on_the_tile(const Shape &s, int m, int n, int k, bool fused, int splits, bool pieces_asked = false) {
  const bool on16 = k % 8 == 0 && n % 8 == 0, on4 = k % 2 == 0 && n % 2 == 0, narrow = narrow_counts(s, m, n);
  const int align = k % 64 == 0 && n % 8 == 0 ? 0 : on16 ? 1 : on4 ? 2 : 3, cus = compute_units();
  constexpr double kSlab[] = {0.19, 0.19, 0.24, 0.33}, kNarrowSlab[] = {0.172, 0.257, 0.272, 0.334}, kMegabyte[] = {0.156, 0.125, 0.134, 0.155};
  const int64_t tiles = static_cast<int64_t>((m + 127) / 128) * s.col_tiles;
  const double c_mb = static_cast<double>(m) * n * 4e-6, memory = static_cast<double>(k) * n * 2e-6 * kMegabyte[align];
  // its pieces: of 256 at least, for a tenth of the time
  auto cut_time = [&](int64_t pieces) {
    return 8.0 + k / 32.0 / static_cast<double>(pieces) * 0.19 * (tiles * pieces > cus ? 1.15 : 1.0) +
           (pieces > 1 ? 5.0 + static_cast<double>(pieces) * c_mb * 0.62 : 0.0);
  };
  int64_t pieces = 1;
  double lowest = 0.9 * cut_time(1);
  for (int64_t t = 2; !fused && t <= 16 && tiles * t <= 2 * cus && k / t >= 256; t *= 2)
    if (cut_time(t) < lowest) lowest = cut_time(t), pieces = t;
  pieces = splitk_pieces(k, 64, pieces);
  const double slabs = k / 32.0 / static_cast<double>(pieces), planes = pieces > 1 ? static_cast<double>(pieces) * c_mb : 0.0;
  if (narrow) {
    const double chain = slabs * kNarrowSlab[align] * static_cast<double>((tiles * pieces + cus - 1) / cus);
    const double tile = 5.17 + std::cbrt(chain * chain * chain + memory * memory * memory) + 0.28 * c_mb + 0.38 * planes + (pieces == 1 ? 0.0 : 4.0);
    const bool behind = narrow_time(s, n, k, splits, !pieces_asked) >= 1.05 * tile;
    if (behind || !fused) return behind;
  }
  const double rounds = static_cast<double>((s.tiles * splits + cus - 1) / cus);
  const double here = (on16 ? 6.0 : 4.5) + rounds * s.steps / splits * (on16 ? 0.055 : on4 ? 0.07 : 0.12) * s.mt +
                      (splits > 1 ? 2.5 + 0.15 * splits + 2.0 * static_cast<double>(splits * s.plane) / 2.7e6 : 0.0);
  return here >= 5.5 + slabs * kSlab[align] + 0.62 * planes + (pieces == 1 ? 0.0 : 3.0);
}

// An element is one sum on the 128 x 128 tile with K whole and eight or more here, and its error there up to 2.8 times as large
// (1280 x 1134 x 566 1.8); in pieces the tile's sums are chunked and as exact as here, up to 2048 of K (37 x 9856 x 7744, 3 pieces, 1.12).
bool less_exact(int k, int tile_splits) { return tile_splits == 1 || k > 2048 * static_cast<int64_t>(tile_splits); }

// Whether a product goes here: by what both kernels are estimated to take, B being new to the caches as in a program's loop over its
// weights (again and again the same B favours the tile more).  17 to 64 rows, us, tile and here: 64 x 29028 x 2725 45.2, 51.8, 51 x 7969 x
// 5857 29.5, 34.4, 63 x 17239 x 320 7.6, 9.5, 42 x 17830 x 3328 32.4, 40.0 (4 % to this kernel's favour, 25 % of up to 8 column tiles:
// profiles/gemm16_rows_vs_tile.txt).  Beyond, and fused, a step costs by how A's and B's rows lie: read off 292 plain and 704 fused drawn
// products run on both (5 % rms, the same on 4000 drawn later; from three quarters of the CUs on 178 of those took 5 % longer): 139 x 2432 x
// 1416 12.0 on the tile, 9.5 here, 114 x 5824 x 2687 15.9, 27.2, fused 419 x 1472 x 2504 25.5, 17.4, 180 x 256 x 2240 10.0, 13.9.  Where
// that moved a product it is 9 % (plain) and 16 % (fused) faster on the average, 3 % of the 6000 looked at are more than 5 % slower.  Fitting it
// all again to those 6000 moves as many the wrong way as the right one.  `other`: what the tiled kernel is estimated at.
bool gemm16_rows_pays(int m, int n, int k, bool fused, Gemm16Estimate other) {
  const Shape s = shape_of(m, n, k, fused);
  const Kernel kernel = outright(s, m, n, k, fused);
  if (kernel != Kernel::by_estimate) return kernel == Kernel::rows;
  const Gemm16Time tile = other(m, n, k, fused);
  const int splits = rows_splits_for(s, n, k);
  double ratio = 0.0;   // this kernel's time over the tile's
  if (narrow_counts(s, m, n)) ratio = narrow_time(s, n, k, splits) / (s.col_tiles > 8 ? 1.04 : 1.25) / tile.us;
  if (m > kTileRows || fused) {
    struct Fit { double step[5], memory[2], base, rows, sums, piece, plane; };
    constexpr Fit kPlain = {{0.0479, 0.0501, 0.0657, 0.0895, 0.105}, {0.091, 0.132}, 2.34, 0.878, 1.01, 0.285, 0.246};
    constexpr Fit kFused = {{0.0489, 0.0487, 0.0638, 0.0884, 0.11}, {0.133, 0.193}, 4.4, 1.186, 0.51, 0.228, 0.335};
    const Fit &f = fused ? kFused : kPlain;
    const int align = k % 8 == 0 && n % 8 == 0 ? 0 : 1 + 2 * (k % 2) + n % 2;
    const double rounds = static_cast<double>((s.tiles * splits + compute_units() - 1) / compute_units());
    const double steps = rounds * s.steps / splits * s.mt * f.step[align], memory = static_cast<double>(k) * n * 2e-6 * f.memory[n % 8 != 0];
    const double here = f.base + f.rows * s.mt + std::sqrt(steps * steps + memory * memory) +
                        (splits > 1 ? f.sums + splits * (f.piece + f.plane * 1e-6 * static_cast<double>(s.plane)) : 0.0);
    ratio = std::max(ratio, here * (4 * s.tiles > 3 * compute_units() ? 1.06 : 1.0) / tile.us);
  }
  return ratio < 1.0 || (less_exact(k, tile.splits) && !coarsely_on_the_tile(s, m, n, k, fused, splits, tile.splits > 1));
}

bool gemm16_rows_more_exact(int m, int n, int k, bool fused) {
  const Shape s = shape_of(m, n, k, fused);
  const Kernel kernel = outright(s, m, n, k, fused);
  if (kernel != Kernel::by_estimate) return kernel == Kernel::rows;
  return !coarsely_on_the_tile(s, m, n, k, fused, rows_splits_for(s, n, k));
}

int gemm16_rows_k_splits(int m, int n, int k) { return rows_splits_for(shape_of(m, n, k, false), n, k); }

int launch_gemm16_rows(bool bf16, const uint16_t *a, const uint16_t *b, float *c, int m, int n, int k, hipStream_t st) {
  const Call q{a, b, c, nullptr, nullptr, m, n, k, st};
  return bf16 ? launch_rows<true, false>(q) : launch_rows<false, false>(q);
}

int launch_gemm16_rows_fused(const uint16_t *a, const uint16_t *b, const float *bias, float *c, float *rowsum, int m, int n,
                             int k, hipStream_t st) {
  return launch_rows<false, true>({a, b, c, bias, rowsum, m, n, k, st});
}

}  // namespace sarek_hip
