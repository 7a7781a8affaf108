// gn_gemm_impl.h - what the GEMM translation units share: the kernel
// parameters, the workgroup -> tile order and the pipeline's barrier.
#pragma once

#include "gn_kernels.h"

namespace gn {

typedef float v4f __attribute__((ext_vector_type(4)));

struct GemmParams {
  const float* A;
  const float* B;
  float* C;
  const float* aux;  // EPI_ADD_SRC source / EPI_DRELU2 pre-activation
  float* aux_out;    // EPI_RELU2_SAVE pre-activation output
  int64_t lda, ldb, ldc, ldaux;
  int M, N, K;
  int k_per_split;
  int tiles_m, tiles_n, splits;
  int epi;
  float alpha;
  float* part;  // split-K: [splits][M][N] partial sums
  // Expert-grouped products (GEMM_GROUP_ROWS / GEMM_GROUP_K): goff[0..groups]
  // are row offsets on the device; gstride is the per-group element offset
  // of B (rows mode) or of C (K mode).
  const int* goff;
  int groups;
  int64_t gstride;
  int a_pad;  // rows mode: A is readable for at least 128 rows past its last row
  // batched products (grid y): product y reads A + y*bsa, B + y*bsb and
  // writes C + y*bsc, its split partials [splits][M][N] at part + y*splits*M*N
  int64_t bsa, bsb, bsc;
};

// Workgroup -> (tile row, tile column, split).  Workgroups are dealt to the
// 8 XCDs round-robin; renumbering gives each XCD a contiguous range of the
// logical order, so the tiles that share operand rows share one L2.  The
// logical order walks groups of 8 tile rows, column by column, so a group's
// A rows and the B columns in flight stay cache-resident.
__device__ __forceinline__ void tile_coords(const GemmParams& p, int& tm, int& tn, int& split) {
  const int total = p.tiles_m * p.tiles_n * p.splits;
  const int bid = blockIdx.x;
  const int x = bid % 8, q = total / 8, rem = total % 8;
  const int logical = x * q + min(x, rem) + bid / 8;
  const int T = p.tiles_m * p.tiles_n;
  split = logical / T;
  const int t = logical - split * T;
  constexpr int GM = 8;
  const int per_group = GM * p.tiles_n;
  const int first = (t / per_group) * GM;
  const int gsz = min(p.tiles_m - first, GM);
  const int r = t % per_group;
  tm = first + r % gsz;
  tn = r / gsz;
}

// Workgroup barrier for the tile pipeline.  No release fence: a fence would
// make the compiler wait for every outstanding LDS-DMA load (vmcnt(0)) and
// defeat the prefetch; the explicit wait before it covers this wave's own
// accesses.  The acquire fence keeps LDS reads below the barrier.
__device__ __forceinline__ void tile_barrier() {
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Sums the [splits][M][N] partials of each of `batch` products (in split order
// in float64) and applies the epilogue.
void launch_gemm_reduce(const GemmParams& p, int batch, hipStream_t st);
// The wide-tile engine (gn_gemm_wide.hip); false: not a product for it.
bool gemm_wide(const GemmDesc& d, GemmParams p, bool vec, hipStream_t st, DeviceArena* ws);
// The few-row engine (gn_gemm_skinny.hip); false: not a product for it.
bool gemm_skinny(const GemmDesc& d, GemmParams p, bool vec, hipStream_t st, DeviceArena* ws);

inline bool aligned16(const void* ptr) { return ((uintptr_t)ptr & 15) == 0; }

}  // namespace gn
