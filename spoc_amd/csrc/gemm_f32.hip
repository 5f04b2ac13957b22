// f32 GEMM for gfx950 on v_mfma_f32_32x32x2_f32 (f32 in, f32 accumulate).
//
// C[M x N] = A[M x K] . B[K x N], all row-major.  Replaces the 16x16 LDS-tiled kernel
// Sarek generates for its tiled matrix multiply: same result up to f32 summation
// order, computed on the matrix cores.
//
// Tiling: one workgroup (512 threads = 8 waves, 2 along M x 4 along N) owns a
// 256 x 256 tile of C and walks K in slabs of 32.  Each wave owns 128 x 64 = 4 x 2
// MFMA tiles of 32 x 32.  LDS holds two stages of (A slab [256][32], rows padded to
// 36 floats; B slab [32][256]).
//
// Operand fetch: the MFMA consumes, per step, k = {k_lo, k_hi} with lanes 0-31 feeding
// k_lo and lanes 32-63 feeding k_hi.  Any assignment of real k indices to (step, half)
// is valid as long as A and B agree, so each lane (m, h) reads FOUR consecutive k of
// its A row with one ds_read_b128 (k = 8*kk + 4h + j, j = 0..3) and uses them over
// four MFMA steps; the matching B values are row 8*kk + 4h + j, column n (ds_read_b32,
// bank-conflict free because n is contiguous).
#include <type_traits>
#include <utility>

#include <algorithm>
#include <cmath>

#include "common.hpp"
#include "gemm_common.hpp"
#include "tunables.hpp"

namespace sarek_hip {
namespace {

typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(4))) float f32x4;

constexpr int BM = 256, BN = 256, BK = 32;
constexpr int THREADS = 512;
constexpr int A_STRIDE = BK + 4;            // floats per A row in LDS (36)
constexpr int B_STRIDE = BN;                // floats per B row in LDS
constexpr int A_FLOATS = BM * A_STRIDE;     // 9216
constexpr int B_FLOATS = BK * B_STRIDE;     // 8192
constexpr int STAGE_FLOATS = A_FLOATS + B_FLOATS;
constexpr int LDS_BYTES = 2 * STAGE_FLOATS * 4;  // 139264

__global__ __launch_bounds__(THREADS) void gemm_f32_staged_kernel(const float *__restrict__ A,
                                                           const float *__restrict__ B,
                                                           float *__restrict__ C, int M, int N,
                                                           int K, int tiles_m, int tiles_n, int xcd_remap) {
  extern __shared__ __attribute__((aligned(16))) float lds_f[];
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 2, wn = wave & 3;
  const int lm = lane & 31, lh = lane >> 5;

  int tm, tn;
  tile_of_block(tiles_m, tiles_n, xcd_remap, tm, tn);
  const int m0 = tm * BM, n0 = tn * BN;

  f32x4 ra[4], rb[4];
  const f32x4 zero4 = {0.f, 0.f, 0.f, 0.f};
  // A slab: 256 rows x 8 chunks of 4 floats; B slab: 32 rows x 64 chunks of 4 floats.
  auto load_slab = [&](int k0) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int c = tid + THREADS * i;
      const int row = c >> 3, kc = (c & 7) * 4;
      const int gr = m0 + row, gk = k0 + kc;
      ra[i] = (gr < M && gk < K)
                  ? *reinterpret_cast<const f32x4 *>(A + static_cast<int64_t>(gr) * K + gk)
                  : zero4;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int c = tid + THREADS * i;
      const int kr = c >> 6, nc = (c & 63) * 4;
      const int gk = k0 + kr, gn = n0 + nc;
      rb[i] = (gk < K && gn < N)
                  ? *reinterpret_cast<const f32x4 *>(B + static_cast<int64_t>(gk) * N + gn)
                  : zero4;
    }
  };
  auto store_slab = [&](int stage) {
    float *sa = lds_f + stage * STAGE_FLOATS;
    float *sb = sa + A_FLOATS;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int c = tid + THREADS * i;
      *reinterpret_cast<f32x4 *>(sa + (c >> 3) * A_STRIDE + (c & 7) * 4) = ra[i];
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int c = tid + THREADS * i;
      *reinterpret_cast<f32x4 *>(sb + (c >> 6) * B_STRIDE + (c & 63) * 4) = rb[i];
    }
  };

  f32x16 acc[4][2];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

  const int a_off = (wm * 128 + lm) * A_STRIDE + lh * 4;   // + i*32*A_STRIDE + kk*8
  const int b_off = (lh * 4) * B_STRIDE + wn * 64 + lm;     // + (kk*8 + j)*B_STRIDE + jn*32

  const int nslabs = (K + BK - 1) / BK;
  load_slab(0);
  store_slab(0);
  __syncthreads();

  for (int s = 0; s < nslabs; ++s) {
    const int cur = s & 1;
    if (s + 1 < nslabs) load_slab((s + 1) * BK);
    const float *sa = lds_f + cur * STAGE_FLOATS;
    const float *sb = sa + A_FLOATS;
#pragma unroll
    for (int kk = 0; kk < BK / 8; ++kk) {
      f32x4 af[4];
#pragma unroll
      for (int i = 0; i < 4; ++i)
        af[i] = *reinterpret_cast<const f32x4 *>(sa + a_off + i * 32 * A_STRIDE + kk * 8);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        float bf[2];
#pragma unroll
        for (int jn = 0; jn < 2; ++jn) bf[jn] = sb[b_off + (kk * 8 + j) * B_STRIDE + jn * 32];
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int jn = 0; jn < 2; ++jn)
            acc[i][jn] = __builtin_amdgcn_mfma_f32_32x32x2f32(af[i][j], bf[jn], acc[i][jn], 0, 0, 0);
      }
    }
    if (s + 1 < nslabs) store_slab(cur ^ 1);
    __syncthreads();
  }

  // Accumulator layout: register r of lane l holds row 8*(r/4) + 4*(l/32) + r%4,
  // column l%32 of its 32 x 32 tile.
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int row = m0 + wm * 128 + i * 32 + 8 * (r >> 2) + 4 * lh + (r & 3);
#pragma unroll
      for (int jn = 0; jn < 2; ++jn) {
        const int col = n0 + wn * 64 + jn * 32 + lm;
        if (row < M && col < N) C[static_cast<int64_t>(row) * N + col] = acc[i][jn][r];
      }
    }
}

// ---- direct-to-LDS ring kernel ------------------------------------------------------
// Tile = (32*TI*WMW) x (32*TJ*WNW), WMW x WNW waves, each wave TI x TJ MFMA tiles of 32 x 32.
// K slabs of BKT stream through NS LDS stages by global_load_lds_dwordx4 (no staging
// registers, no ds_write); the pipeline is the one of the 16-bit GEMM: DMA of slab s+NS
// issued after the barrier inside slab s, barrier before the last k-step of a slab, next
// slab's first fragments fetched under that step's MFMAs.
//
// k-step = 8 k.  A: lane (m, h) reads k = 8kk+4h .. +3 of its row with one ds_read_b128 and
// feeds them to four MFMA steps j; B: for step j the lane reads row 8kk+4h+j at columns
// TJ*lane .. TJ*lane+TJ-1 of the wave's span (one ds_read of TJ floats): MFMA tile jn of the
// wave therefore holds columns {TJ*l + jn}, and in the epilogue every lane owns TJ adjacent
// columns of C, stored as one vector.
//
// LDS (64 banks x 4 B): A rows of 64 B: slot ^= (row>>2)&3, rows of 128 B: slot ^= (row>>1)&7
// (16-lane phases of ds_read_b128).  B reads are contiguous across lanes; only for TJ = 1
// the two half-waves (rows r, r+4) would meet modulo 256 B, so rows with bit 2 set are
// stored with their 128-byte halves swapped.
//
// Ragged = false: N % 4 == 0, K % BKT == 0, A, B and C 16-byte aligned.  Ragged = true: any N, any K >= BKT (or a multiple of
// 4 below it), any alignment.  A lane whose offset lies outside the buffer resource's range brings zeros into LDS, the range
// is checked per dword and the address needs no alignment beyond the element's, so B's range ends with its last element,
// pieces past column N bring the next row's elements into columns that are never stored, and C is stored element by element.
// What K is over whole slabs is at its start, outside the K loop: with it in a slab at the end, moved back over the one
// before, every turn of the loop chose its offsets by masks (64 x 64 tile: 2049 x 4097 x 3000 428 us, now 404; 2031 x 1792 x
// 2211 143, 135; 1500^3 77, 72).
template <int TI, int TJ, int WMW, int WNW, int BKT, int NS, bool Ragged, int Chains>
__global__ __launch_bounds__(64 * WMW * WNW, 2) void gemm_f32_dma_kernel(
    const float *__restrict__ A, const float *__restrict__ B, float *__restrict__ C, int M, int N,
    int K, int tiles_m, int tiles_n, int xcd_remap, unsigned long long *probe, int columns, int cut_tiles, int pieces, int k_chunk,
    float *__restrict__ partials, unsigned *__restrict__ tickets) {
  typedef __attribute__((ext_vector_type(TJ))) float bvec_t;
  constexpr int BMT = 32 * TI * WMW, BNT = 32 * TJ * WNW, NWAVES = WMW * WNW;
  constexpr int KK = BKT / 8;
  constexpr int A_ROW = BKT * 4, A_CHUNKS = A_ROW / 16, A_ROWS_PER_DMA = 1024 / A_ROW;
  constexpr int B_ROW = BNT * 4, B_CHUNKS = B_ROW / 16, B_ROWS_PER_DMA = 1024 / B_ROW;
  constexpr int A_BYTES_S = BMT * A_ROW, B_BYTES_S = BKT * B_ROW;
  constexpr int A_DMA = A_BYTES_S / 1024 / NWAVES, B_DMA = B_BYTES_S / 1024 / NWAVES;
  static_assert(A_DMA >= 1 && B_DMA >= 1 && A_DMA * 1024 * NWAVES == A_BYTES_S &&
                    B_DMA * 1024 * NWAVES == B_BYTES_S, "slab does not split over the waves");
  static_assert(A_ROW == 64 || A_ROW == 128, "BKT must be 16 or 32");
  static_assert(B_ROW <= 1024 && NS * (A_BYTES_S + B_BYTES_S) <= 160 * 1024, "LDS layout");
  static_assert((NS - 1) * (A_DMA + B_DMA) < 64, "vmcnt range");

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WNW, wn = wave % WNW;
  const int lm = lane & 31, lh = lane >> 5;
  // The work: the last cut_tiles of the tiles in `pieces` pieces of K each, then the other tiles, dealt to `columns` (the
  // CUs) in turns of one each.  A column has one or two workgroups that take its turns alternately: workgroups go to the
  // CUs one each and then a second one each, so that what a CU has is even to a turn.  Left to the order in which slots
  // come free it is not: a whole tile and a piece that end together make room for two whole tiles on one CU (634 x 3456 x 1408,
  // 540 tiles of 64 x 64, 28 of them in two pieces, 74.5 us, dealt 55.8).  Beside another stream's kernels a workgroup that starts
  // late keeps its share; 16 products beside the same product took 0.977 of the time of tiles that go to free slots (0.94 to 1.04),
  // beside bf16 4096^3 0.970, alone 0.911, and with fixed turns for launches of cut tiles alone no other.
  // Tiles past whole turns as they are, and cut: 2049 x 4097 x 3000 404 us and 388, 2376 x 2140 x 4096 357 and 299, 1500^3 72 and 57,
  // 896 x 2816 x 2981 138 and 119.
  const int cut_blocks = cut_tiles * pieces, cut_turns = (cut_blocks + columns - 1) / columns;
  const int whole = tiles_m * tiles_n - cut_tiles, turns = cut_turns + (whole + columns - 1) / columns;
  const int column = blockIdx.x % columns, abreast = (gridDim.x + columns - 1) / columns;
  long long probe_c0 = 0, probe_t0 = 0;
  if (kMeasureBuild && probe) {
    probe_c0 = clock64();
    probe_t0 = wall_clock64();
  }
  for (int turn = blockIdx.x / columns; turn < turns; turn += abreast) {
    const bool cut = turn < cut_turns;
    const int item = (cut ? turn : turn - cut_turns) * columns + column;
    if (item >= (cut ? cut_blocks : whole)) continue;
    wait_lds();
    barrier_no_fence();   // the LDS is free again
    const int piece = cut ? item / cut_tiles : 0, cut_tile = item - piece * cut_tiles;
    int tm, tn;
    tile_of_block(tiles_m, tiles_n, xcd_remap, tm, tn, cut ? whole + cut_tile : item);
    const int m0 = tm * BMT, n0 = tn * BNT;
    auto a_swz = [](int row) { return A_CHUNKS == 8 ? ((row >> 1) & 7) : ((row >> 2) & 3); };
    auto b_swz = [](int row) { return TJ == 1 ? (((row >> 2) & 1) << 3) : 0; };

    // DMA sources: uniform 64-bit base + per-lane 32-bit byte offset.  Rows past M and columns
    // past N are clamped to valid addresses; what they produce is never stored.
    uint32_t a_off[A_DMA], b_off[B_DMA];
#pragma unroll
    for (int i = 0; i < A_DMA; ++i) {
      const int q = wave + NWAVES * i;
      const int row_t = q * A_ROWS_PER_DMA + lane / A_CHUNKS;
      const int row = min(row_t, M - 1 - m0);
      a_off[i] = (static_cast<uint32_t>(row) * K + (((lane % A_CHUNKS) ^ a_swz(row_t)) << 2)) * 4u;
    }
#pragma unroll
    for (int i = 0; i < B_DMA; ++i) {
      const int q = wave + NWAVES * i;
      const int brow = q * B_ROWS_PER_DMA + lane / B_CHUNKS;
      const int chunk = (lane % B_CHUNKS) ^ b_swz(brow);
      const int col = Ragged ? n0 + chunk * 4 : min(n0 + chunk * 4, N - 4);
      b_off[i] = (static_cast<uint32_t>(brow) * N + col) * 4u;
    }
    // this workgroup's k: k0 .. k0 + k_len - 1, a last piece what is left of K (at least a slab)
    const int k0 = piece * k_chunk;
    const int k_len = !cut ? K : piece == pieces - 1 ? K - k0 : k_chunk;
    const char *a_base = reinterpret_cast<const char *>(A + static_cast<int64_t>(m0) * K + k0);
    const int64_t b_slab_bytes = static_cast<int64_t>(BKT) * N * 4;
    const int nslabs = (k_len + BKT - 1) / BKT;
    // Ragged: K need not be whole slabs.  What is over them, the first `head` elements, is a slab of its own in front of the
    // others, which then end at K (their A pieces hold nothing but elements of their own rows, at whatever alignment), and
    // the K loop is the aligned form's.  Pieces of A and rows of B past `head` are sent out of range, in A as in B (they belong
    // to the next slab, and an infinity times the other's zero would be NaN); the rest of a piece of A that holds k on both
    // sides of `head` is zeroed in LDS by the lane that brought it (keep).  A lane's k piece is the same for all its A
    // transfers: rows NWAVES * A_ROWS_PER_DMA apart share the swizzle.
    const int head = Ragged ? k_len - (nslabs - 1) * BKT : BKT;
    const int a_lane_k = ((lane % A_CHUNKS) ^ a_swz(wave * A_ROWS_PER_DMA + lane / A_CHUNKS)) << 2;
    const int keep = Ragged && a_lane_k < head && head < a_lane_k + 4 ? head - a_lane_k : 0;
    constexpr uint32_t kOutOfRange = 0x80000000u;

    // Chains: accumulators to an element, for the MFMA steps in turn, added at the end.  Shorter sums are closer to the product
    // (2049 x 4097 x 3000 on the 64 x 64 tile: 6.9e-7 of the result with two, 4.8e-7 with four, 3.4e-7 with eight, which cost 0 to
    // 2 % of the time), and a wave with a single MFMA tile does not feed every MFMA the result of the one before.
    f32x16 acc[Chains][TI][TJ];
#pragma unroll
    for (int h = 0; h < Chains; ++h)
#pragma unroll
      for (int i = 0; i < TI; ++i)
#pragma unroll
        for (int j = 0; j < TJ; ++j)
#pragma unroll
          for (int r = 0; r < 16; ++r) acc[h][i][j][r] = 0.f;

    const int a_row = wm * 32 * TI + lm;
    int a_addr0 = a_row * A_ROW + ((lh ^ a_swz(a_row)) << 4);           // ^ (kk << 5), + i*32*A_ROW
    int b_addr0 = (4 * lh) * B_ROW + (((wn * 32 * TJ + TJ * lm) * 4) ^ (TJ == 1 ? (lh << 7) : 0));

    // A: one resource for the tile's row panel, the slab selects a scalar byte offset.
    // B: the resource is rebased to the slab's first row (keeps every offset below 2^31).
    // Past the last slab a transfer has an empty range: it fetches nothing, and the count of transfers in flight keeps its
    // pattern.  Slabs are issued in order; `at` is 0 for the first.
    const char *b_src = reinterpret_cast<const char *>(B + static_cast<int64_t>(k0) * N);
    int64_t b_left = static_cast<int64_t>(K - k0) * N * 4;
    uint32_t a_so = 0;
    int to_issue = nslabs;
    auto issue = [&](auto at, char *sa, char *sb) {
      constexpr bool first = Ragged && decltype(at)::value == 0;
      const int32_t left_hi = static_cast<int32_t>(b_left >> 32);
      const uint32_t left = left_hi > 0 ? kOutOfRange : left_hi < 0 ? 0u : min(static_cast<uint32_t>(b_left), kOutOfRange);
      const __amdgpu_buffer_rsrc_t a_rsrc = make_rsrc(a_base, to_issue > 0 ? kOutOfRange : 0u);
      const __amdgpu_buffer_rsrc_t b_rsrc = make_rsrc(b_src, Ragged ? left : to_issue > 0 ? kOutOfRange : 0u);
#pragma unroll
      for (int i = 0; i < A_DMA; ++i)
        dma16(a_rsrc, first && a_lane_k >= head ? kOutOfRange : a_off[i], a_so, sa + (wave + NWAVES * i) * 1024);
#pragma unroll
      for (int i = 0; i < B_DMA; ++i)
        dma16(b_rsrc, first && (wave + NWAVES * i) * B_ROWS_PER_DMA + lane / B_CHUNKS >= head ? kOutOfRange : b_off[i], 0u,
              sb + (wave + NWAVES * i) * 1024);
      --to_issue;
      const int64_t step = first ? static_cast<int64_t>(head) * N * 4 : b_slab_bytes;
      b_src += step;
      b_left -= step;
      a_so += first ? head * 4u : BKT * 4u;
    };
    auto load_frags = [&](const char *sa, const char *sb, int kk, f32x4 (&af)[TI], bvec_t (&bf)[4]) {
      const char *pa = sa + (a_addr0 ^ (kk << 5));
#pragma unroll
      for (int i = 0; i < TI; ++i) af[i] = *reinterpret_cast<const f32x4 *>(pa + i * 32 * A_ROW);
#pragma unroll
      for (int j = 0; j < 4; ++j)
        bf[j] = *reinterpret_cast<const bvec_t *>(sb + b_addr0 + (kk * 8 + j) * B_ROW);
    };
    auto mfma_step = [&](int kk, f32x4 (&af)[TI], bvec_t (&bf)[4]) {
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int i = 0; i < TI; ++i)
#pragma unroll
          for (int jn = 0; jn < TJ; ++jn) {
            f32x16 &chain = acc[(4 * kk + j) % Chains][i][jn];
            chain = __builtin_amdgcn_mfma_f32_32x32x2f32(af[i][j], bf[j][jn], chain, 0, 0, 0);
          }
    };
    // Issue order inside one k-step: behind each of the first MFMAs go the DMA instructions
    // of this k-step (NV of them; unpinned, the compiler bunches them in front of the first
    // MFMA, where their issue time leaves the pipe idle) and the LDS reads of the next
    // step's fragments.
    auto interleave = [](auto nv_c) {
      constexpr int NV = decltype(nv_c)::value;
      constexpr int READS = TI + 4, MFMAS = 4 * TI * TJ;
      constexpr int GROUPS = READS < MFMAS ? READS : MFMAS;
      constexpr int PER = (READS + GROUPS - 1) / GROUPS, VPER = (NV + GROUPS - 1) / GROUPS;
      [&]<int... Gs>(std::integer_sequence<int, Gs...>) {
        (([] {
           __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);    // 1 MFMA
           if constexpr (Gs * VPER < NV)                         // DMA instructions
             __builtin_amdgcn_sched_group_barrier(0x020, (NV - Gs * VPER) < VPER ? (NV - Gs * VPER) : VPER, 0);
           __builtin_amdgcn_sched_group_barrier(0x100, PER, 0);  // DS reads
         }()),
         ...);
      }(std::make_integer_sequence<int, GROUPS>{});
      if (MFMAS > GROUPS) __builtin_amdgcn_sched_group_barrier(0x008, MFMAS - GROUPS, 0);
      __builtin_amdgcn_sched_barrier(0);
    };

    f32x4 af[2][TI];
    bvec_t bf[2][4];

    auto slab = [&](char *ca, char *cb, char *na, const char *nb) {
      asm volatile("" : "+v"(a_addr0), "+v"(b_addr0));   // keep per-stage addresses out of registers
#pragma unroll
      for (int kk = 0; kk + 1 < KK; ++kk) {
        load_frags(ca, cb, kk + 1, af[(kk + 1) & 1], bf[(kk + 1) & 1]);
        mfma_step(kk, af[kk & 1], bf[kk & 1]);
        interleave(std::integral_constant<int, 0>{});
      }
      __builtin_amdgcn_s_waitcnt(waitcnt_vm_lgkm0((NS - 2) * (A_DMA + B_DMA)));
      barrier_no_fence();
      issue(std::integral_constant<int, -1>{}, ca, cb);
      load_frags(na, nb, 0, af[0], bf[0]);
      mfma_step(KK - 1, af[(KK - 1) & 1], bf[(KK - 1) & 1]);
      interleave(std::integral_constant<int, A_DMA + B_DMA>{});
    };

    [&]<int... Is>(std::integer_sequence<int, Is...>) {
      (issue(std::integral_constant<int, Is>{}, lds_ring<2 * Is, A_BYTES_S>, lds_ring<2 * Is + 1, B_BYTES_S>), ...);
    }(std::make_integer_sequence<int, NS>{});
    __builtin_amdgcn_s_waitcnt(waitcnt_vm_lgkm0((NS - 1) * (A_DMA + B_DMA)));
    if (keep > 0) {
#pragma unroll
      for (int i = 0; i < A_DMA; ++i) {
        float *piece = reinterpret_cast<float *>(lds_ring<0, A_BYTES_S> + (wave + NWAVES * i) * 1024 + lane * 16);
#pragma unroll
        for (int d = 1; d < 4; ++d)
          if (d >= keep) piece[d] = 0.f;
      }
      wait_lds();
    }
    barrier_no_fence();
    load_frags(lds_ring<0, A_BYTES_S>, lds_ring<1, B_BYTES_S>, 0, af[0], bf[0]);
    __builtin_amdgcn_sched_barrier(0);

    auto ring_slab = [&](auto st_c) {
      constexpr int st = decltype(st_c)::value;
      constexpr int nx = (st + 1) % NS;
      slab(lds_ring<2 * st, A_BYTES_S>, lds_ring<2 * st + 1, B_BYTES_S>, lds_ring<2 * nx, A_BYTES_S>,
           lds_ring<2 * nx + 1, B_BYTES_S>);
    };
    using I0 = std::integral_constant<int, 0>;
    using I1 = std::integral_constant<int, 1>;
    using I2 = std::integral_constant<int, 2>;
    using I3 = std::integral_constant<int, 3>;
    const int full = nslabs - nslabs % NS;
    for (int s = 0; s < full; s += NS) {
      ring_slab(I0{});
      ring_slab(I1{});
      if constexpr (NS == 4) {
        ring_slab(I2{});
        ring_slab(I3{});
      }
    }
    if (full < nslabs) ring_slab(I0{});
    if constexpr (NS == 4) {
      if (full + 1 < nslabs) ring_slab(I1{});
      if (full + 2 < nslabs) ring_slab(I2{});
    }
    __builtin_amdgcn_s_waitcnt(waitcnt_vm_lgkm0(0));   // drain the tail's (empty) transfers
    f32x16 sum[TI][TJ];
#pragma unroll
    for (int i = 0; i < TI; ++i)
#pragma unroll
      for (int j = 0; j < TJ; ++j) {
#pragma unroll
        for (int h = 1; h < Chains; h *= 2)
#pragma unroll
          for (int c = 0; c + h < Chains; c += 2 * h) acc[c][i][j] += acc[c + h][i][j];
        sum[i][j] = acc[0][i][j];
      }

    // A piece's sums go to its plane, past the XCD's L2, in the order its threads hold them; the workgroup that draws a
    // tile's last ticket adds the planes in the order of k and stores the tile: the same bits on every run.
    if (TI * TJ <= 4 && cut) {
      constexpr int kThreads = 64 * NWAVES, kGroups = TI * TJ * 4, kPlane = BMT * BNT * 4, kAtOnce = 8 / (TI * TJ);
      const __amdgpu_buffer_rsrc_t rsrc =
          make_rsrc(reinterpret_cast<char *>(partials) + static_cast<int64_t>(cut_tile) * pieces * kPlane, 0x80000000u);
#pragma unroll
      for (int u = 0; u < kGroups; ++u) {
        const f32x16 &t = sum[u / 4 / TJ][u / 4 % TJ];
        const int r = u % 4 * 4;
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, f32x4{t[r], t[r + 1], t[r + 2], t[r + 3]}), rsrc,
                                               tid * 16, piece * kPlane + u * (kThreads * 16), kDeviceScope);
      }
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
      unsigned *const drawn = reinterpret_cast<unsigned *>(lds_ring<0, A_BYTES_S>);
      if (tid == 0) *drawn = __hip_atomic_fetch_add(tickets + cut_tile, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __syncthreads();
      if (*drawn != static_cast<unsigned>(pieces - 1)) continue;
      if (tid == 0) __hip_atomic_store(tickets + cut_tile, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
      for (int i = 0; i < TI; ++i)
#pragma unroll
        for (int j = 0; j < TJ; ++j)
#pragma unroll
          for (int r = 0; r < 16; ++r) sum[i][j][r] = 0.f;
      for (int q = 0; q < pieces; q += kAtOnce) {
        f32x4 v[kAtOnce][kGroups];
#pragma unroll
        for (int p = 0; p < kAtOnce; ++p)
#pragma unroll
          for (int u = 0; u < kGroups; ++u)
            v[p][u] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(
                                                    rsrc, tid * 16, min(q + p, pieces - 1) * kPlane + u * (kThreads * 16),
                                                    kDeviceScope));
#pragma unroll
        for (int p = 0; p < kAtOnce; ++p)
          if (q + p < pieces) {
#pragma unroll
            for (int u = 0; u < kGroups; ++u)
#pragma unroll
              for (int e = 0; e < 4; ++e) sum[u / 4 / TJ][u / 4 % TJ][u % 4 * 4 + e] += v[p][u][e];
          }
      }
    }

    // Epilogue: register r of lane l holds row 8*(r/4) + 4*(l/32) + r%4 of its 32-row tile and
    // columns TJ*(l%32) .. +TJ-1 of the wave's span (one per MFMA tile jn).
#pragma unroll
    for (int i = 0; i < TI; ++i)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int row = m0 + wm * 32 * TI + i * 32 + 8 * (r >> 2) + 4 * lh + (r & 3);
        const int col = n0 + wn * 32 * TJ + TJ * lm;
        if constexpr (Ragged) {
#pragma unroll
          for (int jn = 0; jn < TJ; ++jn)
            if (row < M && col + jn < N) C[static_cast<int64_t>(row) * N + col + jn] = sum[i][jn][r];
        } else if (row < M && col < N) {
          bvec_t v;
#pragma unroll
          for (int jn = 0; jn < TJ; ++jn) v[jn] = sum[i][jn][r];
          *reinterpret_cast<bvec_t *>(C + static_cast<int64_t>(row) * N + col) = v;
        }
      }
  }
  if (kMeasureBuild && probe && tid == 0) {
    probe[2 * blockIdx.x] = static_cast<unsigned long long>(clock64() - probe_c0);
    probe[2 * blockIdx.x + 1] = static_cast<unsigned long long>(wall_clock64() - probe_t0);
  }
}

// Any shape, any alignment: one thread per C element, f32 FMA in k order.
__global__ __launch_bounds__(256) void gemm_f32_simple_kernel(const float *__restrict__ A,
                                                              const float *__restrict__ B,
                                                              float *__restrict__ C, int M, int N,
                                                              int K) {
  const int col = blockIdx.x * 64 + (threadIdx.x & 63);
  const int row = blockIdx.y * 4 + (threadIdx.x >> 6);
  if (row >= M || col >= N) return;
  float acc = 0.f;
  for (int k = 0; k < K; ++k)
    acc = fmaf(A[static_cast<int64_t>(row) * K + k], B[static_cast<int64_t>(k) * N + col], acc);
  C[static_cast<int64_t>(row) * N + col] = acc;
}

}  // namespace
}  // namespace sarek_hip

using namespace sarek_hip;

namespace {
// How a product is computed: straight from memory (row_blocks > 0; gemm_f32_direct.hip) or through the LDS ring in tiles
// of `tile`, and into how many pieces K is cut (the 64 x 64 tile and the direct kernel).
struct Plan {
  int row_blocks, waves, tile, splits;
  int cut_tiles;   // of the LDS tiles, how many are cut into `splits` pieces of K: the last ones
  int chains;      // sums an element and piece on an LDS tile
};

int64_t tiles_of(int m, int n, int tile) { return ceil_div(m, tile) * ceil_div(n, tile); }
int slab_of(int tile) { return tile == 64 ? 32 : 16; }   // k of an LDS slab

// At most `splits` pieces of K for `cut` tiles: of whole slabs, a ticket per tile, planes within the workspace.
int ring_pieces(int64_t cut, int k, int tile, int64_t splits) {
  if (cut < 1 || cut > kSplitTickets || tile == 256) return 1;
  const int64_t fit = static_cast<int64_t>(kSplitWorkspaceBytes) / (cut * tile * tile * 4);
  return splitk_pieces(k, slab_of(tile), std::max<int64_t>(1, std::min<int64_t>({splits, static_cast<int64_t>(k / 32), fit})));
}

// Estimated time in us of the LDS kernels, fitted to 300 drawn products of 0.2 to 50 GFLOP.  On 440 others, drawn over 64 ..
// 4100 a side from 20 MFLOP on, the plan with the lowest estimate takes 1.2 % more than the fastest of those that were timed; 34
// take more than 5 % and 10 more than 10 %, the worst 21 % (profiles/gemm_f32_plans.txt).  A 64 x 64 tile takes 0.46 us per K = 32
// slab alone on its CU, and two on a CU share its matrix cores, so tiles count in turns of CUs; the larger ones take four and
// sixteen times as long less the operand traffic they save.  A turn's start and stores are 6 us on the 256 x 256 tile, whose
// launch has one workgroup to a CU (2816 x 4096 x 90 36.2 us on it, 31.0 on 128 x 128; counted as 3 us it was taken).  Tiles that
// are cut come on top, in turns of their pieces, with the planes to write and to add.  splits = 0: no less than that with any
// number of pieces.
double ring_estimate(int m, int n, int k, int tile, int64_t cut, int splits) {
  const int64_t tiles = tiles_of(m, n, tile), cus = compute_units();
  const double slabs = k / 32.0, c_mb = 4e-6 * m * n;
  const double slab = tile == 64 ? 0.458 : tile == 128 ? 1.807 : 7.38, each = tile == 64 ? 1.06 : tile == 128 ? 2.96 : 6.0;
  double us = 3.89 + static_cast<double>(ceil_div(tiles - cut, cus)) * (slabs * slab + each) + 0.141 * c_mb;
  if (cut > 0 && splits == 0)
    us += static_cast<double>(cut) / static_cast<double>(cus) * slabs * slab + each + 3.44;
  else if (cut > 0)
    us += static_cast<double>(ceil_div(cut * splits, cus)) * (slabs / splits * slab + each) + 3.44 +
          0.037 * 4e-6 * static_cast<double>(cut) * splits * tile * tile;
  return us;
}

// The variant and the pieces with the lowest estimate.  Pieces are tried only while they leave every wave a step (direct) or
// three slabs (LDS).  Of the LDS tiles those past whole turns of CUs are cut: all of them where there is no whole turn, which
// pays for the 64 x 64 tile alone.
// An element is the sum of shorter ones, of the waves, the chains and the pieces, and its error grows with their length, so a
// plan is not left for a faster one with fewer sums: of the LDS tiles that are cut and of all 64 x 64 ones only those count
// that have as many as the direct variant which would be taken up to 10 GFLOP (four to eight a piece).  The 64 x 64 tile has
// eight chains where it would have fewer otherwise, and where products of under two turns are cut (they were all cut, into
// three pieces or more, before their last tiles alone were).  K = 4000, some 300 tiles: eight waves 4.0e-7 of the result, four
// chains 5.5e-7, eight 3.8e-7 (640 x 1770 x 3844: 99 us, 75.3 and 75.6).  Of 40000 products drawn over 64 .. 4100 a side one has
// fewer sums than before there were cuts (24 for 30).  Tiles that are all cut weigh a 26th less than they are estimated at
// against four sums of the direct kernel, for the same reason.
// block: whether there is one for the pieces' sums.  Without (stream capture, hipStreamPerThread, the seventeenth stream)
// nothing is cut, and a tile that was chosen for its cut is not the one to run whole: in a graph 247 x 1600 x 2884 took 48 us,
// 26 as planned here, 1380 x 3328 x 2112 236 and 156.
// Six workgroups of two row blocks share a CU (their registers), and what is over six to a CU waits for a place: from there to
// eight the direct kernel's estimate is 5 to 24 % short (877 x 3886 x 436, 6.7 to a CU, 39.4 us, 64 x 64 tiles 34).  On 100
// products round there, drawn apart, the chosen plan was 5.4 % above the fastest without the factor, 2.5 with it.
// gemm_f32.direct: 1 = never, 18 / 14 / 24 = always, with (row_blocks, waves) these digits, any other value as 0;
// gemm_f32.tile forces a tile, gemm_f32.split_k the pieces (1 = whole) of all 64 x 64 tiles or of a forced direct variant;
// gemm_f32.cut: 1 = no tile is cut by the rule, n >= 2 = the tiles past whole rounds into n.  0 leaves the choice here.
Plan plan_for(int m, int n, int k, bool ring_ok, bool block) {
  constexpr int kPieces[] = {1, 2, 3, 4, 6, 8, 12, 16};
  const int64_t asked = tunable("gemm_f32.direct", 0);
  const int direct = asked == 1 || asked == 18 || asked == 14 || asked == 24 ? static_cast<int>(asked) : 0;
  const int forced = static_cast<int>(tunable("gemm_f32.tile", 0));
  const int tile = forced == 0 || forced == 256 || forced == 128 ? forced : 64;
  int64_t split = tunable("gemm_f32.split_k", 0), cutting = tunable("gemm_f32.cut", 0);
  if (!block) split = std::min<int64_t>(split, 1), cutting = 1;
  const bool direct_ok = gemm_f32_direct_serves(m, n, k);
  if (direct > 1 && direct_ok)
    return {direct / 10, direct % 10, 0, gemm_f32_direct_pieces(m, n, k, direct / 10, static_cast<int>(std::min<int64_t>(split, 64))), 0, 0};
  const int64_t cus = compute_units();
  Plan best{0, 0, 0, 1, 0, 0}, best_direct = best;
  double best_us = 1e300, direct_us = 1e300, uncrowded_us = 1e300;
  // (the clock probe of the measurement build is the ring kernels': a launch that it watches goes to them)
  const bool probed = kMeasureBuild && clock_probe(1) != nullptr;
  if (direct == 0 && direct_ok && !(probed && ring_ok) && (!ring_ok || (tile == 0 && split == 0 && gemm_f32_direct_pays(m, n, k, false))))
    for (const auto [row_blocks, waves] : {std::pair{1, 8}, std::pair{1, 4}, std::pair{2, 4}}) {
      const int64_t tiles = ceil_div(m, 16 * row_blocks) * ceil_div(n, 64);
      for (const int pieces : kPieces) {
        if (pieces > 1 && (!block || k / 16 / pieces < waves || tiles * pieces > 4 * cus)) break;
        const int splits = gemm_f32_direct_pieces(m, n, k, row_blocks, pieces);
        double us = 1.01 * gemm_f32_direct_estimate(m, n, k, row_blocks, waves, splits);
        uncrowded_us = std::min(uncrowded_us, us);
        if (row_blocks == 2 && tiles * splits > 6 * cus && tiles * splits <= 8 * cus) us *= 1.15;
        if (us < direct_us) direct_us = us, best_direct = {row_blocks, waves, 0, splits, 0, 0};
      }
    }
  if (!ring_ok || gemm_f32_direct_pays(m, n, k, block)) best_us = direct_us, best = best_direct;
  if (!ring_ok) return best;
  const int direct_sums = best_direct.waves * best_direct.splits;
  for (const int t : {64, 128, 256}) {
    if (tile != 0 && tile != t) continue;
    const int64_t tiles = tiles_of(m, n, t), over = tiles % cus;
    auto consider = [&](int64_t cut, int splits) {
      if (splits < 2) cut = 0, splits = 1;
      const int pieces = cut == tiles ? splits : 1;   // of every element
      double us = ring_estimate(m, n, k, t, cut, splits);
      if (cut == tiles && direct_sums == 4) us /= 1.04;
      int chains = t == 256 ? 1 : t == 128 ? 2 : 4;
      if (t == 64 && (chains * pieces < direct_sums || (cut > 0 && tiles < 2 * cus))) chains = 8;
      if (chains * pieces < direct_sums && (t == 64 || cut > 0 || us >= uncrowded_us)) return;
      if (us < best_us) best_us = us, best = {0, 0, t, splits, static_cast<int>(cut), chains};
    };
    if (t == 64 && split >= 2) {
      consider(tiles, ring_pieces(tiles, k, t, split));
      continue;
    }
    const bool may_cut = split == 0 && cutting != 1 && !probed && t != 256;
    if (!may_cut || cutting < 2) consider(0, 1);
    if (!may_cut) continue;
    if (cutting >= 2) {
      consider(over ? over : std::min(tiles, cus), ring_pieces(over ? over : std::min(tiles, cus), k, t, cutting));
      continue;
    }
    // (where no number of pieces can be ahead they are not gone through: 0.2 of the 0.6 us in which a small product is planned)
    if (over == 0 || k / 2 < 96 || ring_estimate(m, n, k, t, over, 0) > 1.04 * best_us) continue;
    for (int pieces = 2; (t == 64 || over < tiles) && pieces <= 12 && k / pieces >= 96; ++pieces)
      consider(over, ring_pieces(over, k, t, pieces));
  }
  return best.tile > 0 || best.row_blocks > 0 ? best : best_direct;
}
}  // namespace

extern "C" int sarek_hip_gemm_f32_k_splits(int m, int n, int k) {
  if (m < 1 || n < 1 || k < 1) return 1;
  const Plan plan = plan_for(m, n, k, k >= 32 || k % 4 == 0, true);
  return plan.row_blocks > 0 || (plan.tile > 0 && plan.cut_tiles == tiles_of(m, n, plan.tile)) ? plan.splits : 1;
}

extern "C" int sarek_hip_gemm_f32(const float *a, const float *b, float *c, int m, int n, int k,
                                  sarek_hip_stream stream) {
  if (m <= 0 || n <= 0 || k <= 0)
    return fail(SAREK_HIP_E_INVALID_ARG, "gemm_f32: m, n, k must be positive (got %d %d %d)", m, n, k);
  if (!a || !b || !c) return fail(SAREK_HIP_E_INVALID_ARG, "gemm_f32: NULL matrix");
  hipStream_t st = as_stream(stream);
  // The direct-to-LDS kernels take any shape and alignment in their Ragged form, except a K below one slab that is
  // not a multiple of 4; the aligned form is the faster one where it applies.
  const bool aligned = (k % 4 == 0) && (reinterpret_cast<uintptr_t>(a) % 16 == 0) &&
                       (reinterpret_cast<uintptr_t>(b) % 16 == 0);
  const bool ab_ok = aligned || k >= 32;   // the ragged form needs no alignment once K fills a slab
  const int remap = (int)tunable("gemm.xcd_remap", 1);
  // DMA offsets are 32-bit: 256 rows of A and 32 rows of B must span less than 2 GiB
  const bool offsets_ok = static_cast<int64_t>(k) * 256 * 4 < 0x7FFFFFFF &&
                          static_cast<int64_t>(n) * 32 * 4 < 0x7FFFFFFF;
  const bool ring_ok = ab_ok && offsets_ok;
  const bool c_aligned = reinterpret_cast<uintptr_t>(c) % 16 == 0;
  const bool fallback = tunable("gemm_f32.force_simple", 0) != 0 || tunable("gemm_f32.force_staged", 0) != 0;
  Plan plan{0, 0, 0, 1, 0, 0};
  Workspace workspace;
  if (!fallback) {
    plan = plan_for(m, n, k, ring_ok, true);
    if (plan.splits > 1) workspace = splitk_workspace(st);
    if (plan.splits > 1 && !workspace.block) plan = plan_for(m, n, k, ring_ok, false);
  }
  float *const partials = workspace.block;
  if (plan.row_blocks > 0) return launch_gemm_f32_direct(a, b, c, m, n, k, plan.row_blocks, plan.waves, plan.splits, partials, st);
  if (plan.tile > 0) {
    const bool ragged = !aligned || n % 4 != 0 || k % 32 != 0 || !c_aligned;
    const int tile = plan.tile;
    const int64_t tiles = tiles_of(m, n, tile);
    const int splits = plan.splits, cut_tiles = plan.cut_tiles;
    // two workgroups to a CU where there is work for them and LDS (64 KiB for the two smaller tiles, 128 for the largest)
    const int64_t columns = compute_units(), cut_blocks = static_cast<int64_t>(cut_tiles) * splits;
    const int64_t turns = ceil_div(cut_blocks, columns) + ceil_div(tiles - cut_tiles, columns);
    const int64_t items = cut_blocks + tiles - cut_tiles;
    const int64_t workgroups = turns == 1 ? items : columns * (tile == 256 ? 1 : 2);
    const int k_chunk = cut_tiles > 0 ? splitk_chunk(k, slab_of(tile), splits) : k;
#define SAREK_LAUNCH_F32(T, TI, TJ, WMW, WNW, BKT, RAGGED, CHAINS)                                  \
  hipLaunchKernelGGL((gemm_f32_dma_kernel<TI, TJ, WMW, WNW, BKT, 4, RAGGED, CHAINS>),              \
                     dim3(static_cast<unsigned>(workgroups)),                                              \
                     dim3(64 * WMW * WNW), 0, st, a, b, c, m, n, k, (m + T - 1) / T, (n + T - 1) / T, remap, \
                     cut_tiles > 0 ? nullptr : clock_probe(workgroups), static_cast<int>(columns), cut_tiles, splits, k_chunk, partials, \
                     partials ? splitk_tickets(partials) : nullptr)
    if (ragged) {
      if (tile == 256) SAREK_LAUNCH_F32(256, 4, 2, 2, 4, 16, true, 1);
      else if (tile == 128) SAREK_LAUNCH_F32(128, 2, 2, 2, 2, 16, true, 2);
      else if (plan.chains == 8) SAREK_LAUNCH_F32(64, 1, 1, 2, 2, 32, true, 8);
      else SAREK_LAUNCH_F32(64, 1, 1, 2, 2, 32, true, 4);
    } else {
      if (tile == 256) SAREK_LAUNCH_F32(256, 4, 2, 2, 4, 16, false, 1);
      else if (tile == 128) SAREK_LAUNCH_F32(128, 2, 2, 2, 2, 16, false, 2);
      else if (plan.chains == 8) SAREK_LAUNCH_F32(64, 1, 1, 2, 2, 32, false, 8);
      else SAREK_LAUNCH_F32(64, 1, 1, 2, 2, 32, false, 4);
    }
#undef SAREK_LAUNCH_F32
    return check_launch("gemm_f32 kernel launch");
  }
  if (aligned && n % 4 == 0 && tunable("gemm_f32.force_simple", 0) == 0) {
    static bool attr_done = false;
    if (!attr_done) {
      SAREK_HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void *>(gemm_f32_staged_kernel),
                                        hipFuncAttributeMaxDynamicSharedMemorySize, LDS_BYTES));
      attr_done = true;
    }
    const int tiles_m = (m + BM - 1) / BM, tiles_n = (n + BN - 1) / BN;
    hipLaunchKernelGGL(gemm_f32_staged_kernel, dim3(tiles_m * tiles_n), dim3(THREADS), LDS_BYTES, st, a, b,
                       c, m, n, k, tiles_m, tiles_n, remap);
  } else {
    hipLaunchKernelGGL(gemm_f32_simple_kernel, dim3((n + 63) / 64, (m + 3) / 4), dim3(256), 0, st,
                       a, b, c, m, n, k);
  }
  return check_launch("gemm_f32 kernel launch");
}
