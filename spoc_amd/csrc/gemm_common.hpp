// Device helpers shared by the GEMM kernels: workgroup -> tile raster, the LDS ring of
// the direct-to-LDS pipelines, DMA and barrier primitives.
#pragma once
#include <mutex>

#include <hip/hip_runtime.h>

namespace sarek_hip {

// K-split products (gemm_splitk.hip): the per-stream block of device memory for the partial planes and the kernel that
// adds them into C in a fixed order.
constexpr size_t kSplitWorkspaceBytes = 64u << 20;
// A stream's block (nullptr: none), held by one call at a time until its launches are issued: those of another thread's call on
// the same stream would come between the launch that fills the planes and the one that adds them.
struct Workspace {
  float *block = nullptr;
  std::unique_lock<std::mutex> issuing;
};
Workspace splitk_workspace(hipStream_t st);
int launch_splitk_reduce(const float *partials, float *c, int m, int n, int splits, hipStream_t st);
int launch_splitk_reduce_fused(const float *partials, const float *bias, float *y, float *rowsum, int m, int n, int splits,
                               hipStream_t st);   // with the bias, the ReLU and the row sums
// Floats from one partial plane to the next: planes start at 16 bytes.
__host__ __device__ inline int64_t splitk_plane_floats(int m, int n) { return (static_cast<int64_t>(m) * n + 3) / 4 * 4; }
// K in at most `splits` pieces of whole stages of `stage`: their length (the last one takes what is left, at least a
// stage), and how many come out.
inline int splitk_chunk(int k, int stage, int64_t splits) {
  const int64_t stages = (k + stage - 1) / stage;
  return static_cast<int>((stages + splits - 1) / splits) * stage;
}
inline int splitk_pieces(int k, int stage, int64_t splits) {
  while (splits > 1 && k - splitk_chunk(k, stage, splits) * (splits - 1) < stage) --splits;
  return static_cast<int>(splits);
}
// Counters behind the planes of a block, zero between launches: one per tile for kernels whose last piece adds the planes, and
// one per row of tiles for those whose last tile adds the row sums.
constexpr int kSplitTickets = 4096, kFoldTickets = 4096;
inline unsigned *splitk_tickets(float *block) {
  return reinterpret_cast<unsigned *>(reinterpret_cast<char *>(block) + kSplitWorkspaceBytes);
}
inline unsigned *fold_tickets(float *block) { return splitk_tickets(block) + kSplitTickets; }

// Compute units of the current device (256 where it does not say).
int compute_units();

// float32 products straight from memory to registers (gemm_f32_direct.hip): variants (row_blocks, waves) = (1, 8), (1, 4),
// (2, 4)
bool gemm_f32_direct_serves(int m, int n, int k);
bool gemm_f32_direct_pays(int m, int n, int k, bool cuts);
int gemm_f32_direct_pieces(int m, int n, int k, int row_blocks, int splits);
double gemm_f32_direct_estimate(int m, int n, int k, int row_blocks, int waves, int splits);
int launch_gemm_f32_direct(const float *a, const float *b, float *c, int m, int n, int k, int row_blocks, int waves,
                           int splits, float *partials, hipStream_t st);   // partials: splitk_workspace's block where splits > 1

// 16-bit products in tiles of at most 64 rows, straight from memory to registers (gemm16_rows.hip)
bool gemm16_rows_serves(int m, int n, int k);
struct Gemm16Time { double us; int splits; };
using Gemm16Estimate = Gemm16Time (*)(int m, int n, int k, bool fused);   // on the 128 x 128 tile, in the pieces of K it would take
bool gemm16_rows_pays(int m, int n, int k, bool fused, Gemm16Estimate other);
// Whether a product that was to go to the tile in pieces goes here if it cannot be cut.
bool gemm16_rows_more_exact(int m, int n, int k, bool fused);
int gemm16_rows_k_splits(int m, int n, int k);
int launch_gemm16_rows(bool bf16, const uint16_t *a, const uint16_t *b, float *c, int m, int n, int k, hipStream_t st);
int launch_gemm16_rows_fused(const uint16_t *a, const uint16_t *b, const float *bias, float *c, float *rowsum, int m, int n,
                             int k, hipStream_t st);
// Row sums of the fused products, where the last workgroup of a row of tiles adds the planes (fold_rows): every plane of the
// product, M floats each, and the counters (nullptr: a launch of its own adds them).
struct RowFold {
  const float *planes;
  int count;
  unsigned *tickets;
};
// Row sums of the fused products (gemm16.hip): zeroes, and rowsum[r] = planes[r] + planes[m + r] + ... in plane order
int launch_zero_f32(float *p, int n, hipStream_t st);
int launch_rowsum_fold(const float *planes, int count, int m, float *rowsum, hipStream_t st);

namespace {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(8))) _Float16 f16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4_t;
typedef f32x4_t f32x4_u __attribute__((aligned(4)));   // at any element's address
typedef __attribute__((ext_vector_type(4))) unsigned int u32x4;
typedef __attribute__((ext_vector_type(2))) unsigned long long u64x2;

template <bool Bf16>
__device__ __forceinline__ f32x4_t mfma16(u32x4 a, u32x4 b, f32x4_t c) {
  if constexpr (Bf16)
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c,
                                                   0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0,
                                                  0, 0);
}

#define LDS_PTR __attribute__((address_space(3)))

constexpr int NUM_XCD = 8;   // XCDs of an MI355X; workgroup ids are dealt to them round-robin

// Workgroup -> tile.  The hardware deals consecutive workgroup ids round-robin to the
// 8 XCDs (each with its own L2), so ids are first regrouped to give every XCD one
// contiguous run of tiles, and the run is walked in bands of GROUP tile-rows, column by
// column: the ~32 tiles an XCD has in flight then form a compact GROUP x (32 / GROUP) patch that
// moves through K together and shares A row-panels and B column-panels in that L2.
// GROUP = 4 (xcd_remap = 1; a larger xcd_remap sets another height): with 32 x 32 tiles every XCD then owns one
// band of four tile-rows and all eight walk the same column panels of B at the same time, so what one of them
// brings past its L2 the others find in the memory-side cache.  Measured on bf16 products against bands of 8:
// 8192^3 0.729 against 0.740 ms, 8192 x 4096 x 8192 0.365 against 0.374, 16384 x 8192 x 2048 0.442 against 0.474,
// nothing lost on 3072^3, 4096^3, the fp16 epilogue shape and the f32 8192^3 product; bands of 2, 16 or 32 are slower.
// block: the workgroup's id, or what stands for it where not every tile has a workgroup of its own.
__device__ __forceinline__ void tile_of_block(int tiles_m, int tiles_n, int xcd_remap, int &tm,
                                              int &tn, int block) {
  const int GROUP = xcd_remap > 1 ? xcd_remap : 4;   // tile-rows per raster band
  const int nblocks = tiles_m * tiles_n;
  const int xcd = block % NUM_XCD, slot = block / NUM_XCD;
  int tile = xcd * (nblocks / NUM_XCD) + min(xcd, nblocks % NUM_XCD) + slot;
  if (xcd_remap == 0) tile = block;
  const int per_group = GROUP * tiles_n;
  const int g = tile / per_group;
  const int rows_in_group = min(GROUP, tiles_m - g * GROUP);
  const int in_g = tile - g * per_group;
  tm = g * GROUP + in_g % rows_in_group;
  tn = in_g / rows_in_group;
}

__device__ __forceinline__ void tile_of_block(int tiles_m, int tiles_n, int xcd_remap, int &tm, int &tn) {
  tile_of_block(tiles_m, tiles_n, xcd_remap, tm, tn, static_cast<int>(blockIdx.x));
}

// One static LDS array per ring stage and operand: distinct objects, so the compiler can
// tell that the DMA into one stage does not alias the ds_reads of another and need not
// wait for it.
template <int Id, int Bytes>
__shared__ __attribute__((aligned(1024))) char lds_ring[Bytes];

// Global -> LDS DMA: buffer_load_dwordx4 ... lds.  64 lanes x 16 bytes, lane l's piece lands
// at lds_dst + 16*l.  The buffer form (scalar resource + 32-bit lane offset + scalar offset)
// is used on purpose: measured on MI355X, four global_load_lds_dwordx4 per 32 MFMAs cut the
// MFMA issue rate by a third, the same number of buffer_load ... lds cost nothing.
// Offsets at or past `bytes` read as zero (raw buffer range check).
__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void *base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), 0, static_cast<int>(bytes),
                                           0x00020000);
}
// Cache-policy bits stay 0: sc0 / sc1 change nothing measurable for these loads, nt costs 8 % (the
// panels are shared through the L2 by the tiles of a patch, and nt lines leave it early).
__device__ __forceinline__ void dma16(__amdgpu_buffer_rsrc_t rsrc, uint32_t lane_off,
                                      uint32_t uniform_off, char *lds_dst) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (LDS_PTR void *)lds_dst, 16,
                                           static_cast<int>(lane_off),
                                           static_cast<int>(uniform_off), 0, 0);
}

// s_waitcnt immediate (gfx9 encoding) that waits for vmcnt <= n and lgkmcnt <= 0.
constexpr int waitcnt_vm_lgkm0(int n) { return (n & 15) | ((n >> 4) << 14) | (7 << 4) | (0 << 8); }
// Waits for this wave's LDS accesses, what it wrote before among them.
__device__ __forceinline__ void wait_lds() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

// Workgroup barrier without the fence __syncthreads() carries (which would drain every
// outstanding DMA): callers wait for exactly the DMA they need first.
__device__ __forceinline__ void barrier_no_fence() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// Cache policy of a buffer access that other XCDs take part in: past the L2s, which they do not share.
constexpr int kDeviceScope = 16;

// rowsum[r] = the planes' sums of row r for the `rows` rows (at most Pitch) from m0 on that exist, by the last of the `arrivals`
// workgroups that have put their shares of these rows into planes (with kDeviceScope; this workgroup's are on their way).  `rows` is
// the height of their tiles: the rows below belong to workgroups that this counter does not count.  In plane order, in double, one
// rounding, Threads / Pitch threads to a row: the same bits on every run.  Us, with a launch of its own for that and now: 128 x 128 x
// 256 10.0 -> 7.4 (one launch to issue), 419 x 285 x 3370 17.3 -> 16.3, 701 x 384 x 824 12.4 -> 11.9, 5760 x 2560 x 448 25.0 -> 24.1.
// What is left is a chain: C and the share stored, the counter's trip, the planes' loads.
// scratch: LDS that no wave reads or writes any more when all have called this.
template <int Threads, int Pitch>
__device__ __forceinline__ void fold_rows(const RowFold &fold, int M, int m0, int rows, float *__restrict__ rowsum, int tile_row,
                                          int arrivals, float *scratch) {
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
  barrier_no_fence();
  unsigned *const drawn = reinterpret_cast<unsigned *>(scratch);
  if (threadIdx.x == 0) *drawn = __hip_atomic_fetch_add(fold.tickets + tile_row, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  wait_lds();
  barrier_no_fence();
  if (__builtin_amdgcn_readfirstlane(*drawn) != static_cast<unsigned>(arrivals - 1)) return;
  constexpr int Parts = Threads / Pitch, InFlight = 16;
  double *const sums = reinterpret_cast<double *>(scratch + 16);
  const int row = threadIdx.x % Pitch, part = threadIdx.x / Pitch;
  const __amdgpu_buffer_rsrc_t rsrc = make_rsrc(fold.planes, 0x7FFFFFFFu);
  const int end = min(M, m0 + rows), at = min(m0 + row, end - 1) * 4;
  double acc = 0.0;
  for (int t = part; t < fold.count; t += Parts * InFlight) {
    float v[InFlight];
#pragma unroll
    for (int u = 0; u < InFlight; ++u)
      v[u] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rsrc, at + min(t + u * Parts, fold.count - 1) * M * 4, 0, kDeviceScope));
#pragma unroll
    for (int u = 0; u < InFlight; ++u) acc += t + u * Parts < fold.count ? static_cast<double>(v[u]) : 0.0;
  }
  sums[threadIdx.x] = acc;
  wait_lds();
  barrier_no_fence();
  if (part == 0 && m0 + row < end) {
#pragma unroll
    for (int q = 1; q < Parts; ++q) acc += sums[q * Pitch + row];
    rowsum[m0 + row] = static_cast<float>(acc);
  }
  if (threadIdx.x == 0) __hip_atomic_store(fold.tickets + tile_row, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

}  // namespace
}  // namespace sarek_hip
