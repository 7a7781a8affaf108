// gn_gemm_skinny.hip - x.W^T with few rows (M <= 32): the projections and the
// lm_head of small decode batches, scoring of short prompts.
//
// Such a product reads every weight once for a few rows, so it is bound by
// the latency of its first loads and by how much of the weight matrix is in
// flight.  One workgroup of NW waves (16 where the K range and the registers
// allow, 4 for many output tiles, whose workgroups walk several) owns 16
// outputs; each wave takes an equal part of the (split's) K range and requests
// its whole 16-row slice of the weights at once (16 KV k per chunk, KV 16-byte
// loads per lane) beside the same k of x, which stay in registers while the
// workgroup walks its output tiles (the next tile's weights are requested
// before the current one's sums meet).  The waves' partial sums meet in LDS,
// in wave order, in float64.
//
// Why: at these sizes gemm_kernel's 64 x 64 tiles ran 16-fold padding through
// a four-stage LDS pipeline, 13.4 us per d12 projection of one decode row.
// Here the projections of one to 16 rows take 3.9 us (qkv, attention output),
// 5.5 us (the MLP pair: 9.4 MB of weights, 1.9 us at the copy rate) and the
// lm_head (201 MB) about 50 us; a decode step of one row 1000 -> 495 us.
//
// v_mfma_f32_16x16x4_f32 with the weights as the row operand: lane (i, q) =
// (lane & 15, lane >> 4) holds k 16 t + 4 q + c of weight row i and of x row
// i for step (t, c), and receives four consecutive outputs of one x row.
#include <algorithm>
#include <cstdlib>

#include "gn_gemm_impl.h"

namespace gn {
namespace skinny {

// NORM: y = rmsnorm(x).W^T = x.W^T times 1 / rms(x), a factor per row that the
// waves find from the x in their registers (one chunk: their whole k range).
template <int MB, int KV, int NW, bool NORM>
__global__ __launch_bounds__(64 * NW, NW == 4 ? 2 : 1) void gemm_skinny_kernel(GemmParams p,
                                                                             int chunks,
                                                                             float eps) {
  __shared__ v4f red[2][NW][MB][64];
  __shared__ float ssq[NW][MB][16];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int i = lane & 15, q = lane >> 4;
  const int k0 = ((int)blockIdx.y * NW + w) * chunks * 16 * KV + 4 * q;
  const int tiles = (p.N + 15) / 16;
  const float* xr[MB];
  bool live[MB];
#pragma unroll
  for (int b = 0; b < MB; b++) {
    live[b] = 16 * b + i < p.M;
    xr[b] = p.A + (int64_t)(live[b] ? 16 * b + i : 0) * p.lda + k0;
  }
  auto load_x = [&](int ch, v4f (&x)[MB][KV]) {
#pragma unroll
    for (int b = 0; b < MB; b++)
#pragma unroll
      for (int t = 0; t < KV; t++) {
        x[b][t] = *reinterpret_cast<const v4f*>(xr[b] + (ch * KV + t) * 16);
        if (!live[b]) x[b][t] = (v4f){0.f, 0.f, 0.f, 0.f};
      }
  };
  auto load_w = [&](int tile, int ch, v4f (&wv)[KV]) {
    const float* r = p.B + (int64_t)min(16 * tile + i, p.N - 1) * p.ldb + k0;
#pragma unroll
    for (int t = 0; t < KV; t++) wv[t] = *reinterpret_cast<const v4f*>(r + (ch * KV + t) * 16);
  };
  v4f wv[KV], x[MB][KV];
  int par = 0;
  load_w(blockIdx.x, 0, wv);
  load_x(0, x);
  if constexpr (NORM) {
#pragma unroll
    for (int b = 0; b < MB; b++) {
      float s = 0.f;
#pragma unroll
      for (int t = 0; t < KV; t++)
#pragma unroll
        for (int r = 0; r < 4; r++) s += x[b][t][r] * x[b][t][r];
      s += __shfl_xor(s, 16, 64);
      s += __shfl_xor(s, 32, 64);
      if (q == 0) ssq[w][b][i] = s;  // read after the first tile's barrier
    }
  }
  for (int tile = blockIdx.x; tile < tiles; tile += gridDim.x, par ^= 1) {
    // four independent chains per block: a dependent MFMA would wait for the
    // one before, and each chain rounds K / 64 times instead of K / 16
    v4f acc[MB][4];
#pragma unroll
    for (int b = 0; b < MB; b++)
#pragma unroll
      for (int c = 0; c < 4; c++) acc[b][c] = (v4f){0.f, 0.f, 0.f, 0.f};
    for (int ch = 0; ch < chunks; ch++) {
#pragma unroll
      for (int t = 0; t < KV; t++)
#pragma unroll
        for (int c = 0; c < 4; c++)
#pragma unroll
          for (int b = 0; b < MB; b++)
            acc[b][c] =
                __builtin_amdgcn_mfma_f32_16x16x4f32(wv[t][c], x[b][t][c], acc[b][c], 0, 0, 0);
      const bool last = ch + 1 == chunks;
      const int nt = last ? tile + gridDim.x : tile, nc = last ? 0 : ch + 1;
      if (nt < tiles) {
        load_w(nt, nc, wv);
        if (chunks > 1) load_x(nc, x);
      }
    }
#pragma unroll
    for (int b = 0; b < MB; b++) red[par][w][b][lane] = (acc[b][0] + acc[b][1]) + (acc[b][2] + acc[b][3]);
    // the next tile writes the other half, so one barrier per tile
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    tile_barrier();
    const int b = w, m = 16 * b + i, n = 16 * tile + 4 * q;
    if (b < MB && m < p.M && n < p.N) {
      float inv = 1.f;
      if constexpr (NORM) {
        float ss = 0.f;
#pragma unroll
        for (int u = 0; u < NW; u++) ss += ssq[u][b][i];
        inv = 1.f / sqrtf(ss / (float)p.K + eps);
      }
      double s[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll 4
      for (int u = 0; u < NW; u++) {
        const v4f e = red[par][u][b][lane];
#pragma unroll
        for (int r = 0; r < 4; r++) s[r] += (double)e[r];
      }
      v4f v;
#pragma unroll
      for (int r = 0; r < 4; r++) {
        v[r] = (float)s[r] * inv;
      }
      if (p.part) {
        *reinterpret_cast<v4f*>(&p.part[((int64_t)blockIdx.y * p.M + m) * p.N + n]) = v;
      } else {
        float* c = &p.C[(int64_t)m * p.ldc + n];
        if (p.epi == EPI_ADD_SRC) {
          v += *reinterpret_cast<const v4f*>(&p.aux[(int64_t)m * p.ldaux + n]);
        } else if (p.epi == EPI_RELU2_SAVE) {
          if (p.aux_out) *reinterpret_cast<v4f*>(&p.aux_out[(int64_t)m * p.ldaux + n]) = v;
#pragma unroll
          for (int r = 0; r < 4; r++) {
            const float u = v[r] < 0.f ? 0.f : v[r];
            v[r] = u * u;
          }
        } else if (p.epi == EPI_SOFTCAP) {
#pragma unroll
          for (int r = 0; r < 4; r++) v[r] = softcap15(v[r]);
        } else {
          v *= p.alpha;
        }
        *reinterpret_cast<v4f*>(c) = v;
      }
    }
  }
}

}  // namespace skinny

typedef void (*SkinnyKernel)(GemmParams, int, float);
// Widest chunk whose x and weights fit the registers of a workgroup of NW
// waves beside the accumulators.
constexpr int max_kv(int mb, int nw) { return nw == 4 ? 12 : mb == 1 ? 6 : 3; }
template <int MB, int NW, bool NORM>
static SkinnyKernel skinny_kernel_n(int kv) {
  using namespace skinny;
  constexpr int MX = max_kv(MB, NW);
  switch (kv) {
    case 3: return gemm_skinny_kernel<MB, 3, NW, NORM>;
    case 2: return gemm_skinny_kernel<MB, 2, NW, NORM>;
    case 1: return gemm_skinny_kernel<MB, 1, NW, NORM>;
  }
  if constexpr (MX >= 6) {
    if (kv == 6) return gemm_skinny_kernel<MB, 6, NW, NORM>;
    if (kv == 5) return gemm_skinny_kernel<MB, 5, NW, NORM>;
    if (kv == 4) return gemm_skinny_kernel<MB, 4, NW, NORM>;
  }
  if constexpr (MX >= 12) {
    if (kv == 12) return gemm_skinny_kernel<MB, 12, NW, NORM>;
    if (kv == 10) return gemm_skinny_kernel<MB, 10, NW, NORM>;
    if (kv == 8) return gemm_skinny_kernel<MB, 8, NW, NORM>;
  }
  return nullptr;
}

// Waves per workgroup: 16 when the K range and the register budget of a
// 1024-thread workgroup allow (x and the weights of one chunk, 16 KV bytes
// each per lane), so that the whole slice is in flight in fewer registers and
// each wave's chain of MFMAs is short; 4 for many output tiles (the lm_head),
// whose workgroups walk several.
static int largest_kv(int units, int mx) {
  for (int v : {12, 10, 8, 6, 5, 4, 3, 2, 1})
    if (v <= mx && units % v == 0) return v;
  return 1;
}

bool skinny_norm_supported(int rows, int C) {
  return rows <= 32 && C % 256 == 0 && C / 256 <= max_kv(rows <= 16 ? 1 : 2, 16);
}

// y = rmsnorm(x).W^T through EPI_STORE or EPI_RELU2_SAVE for at most 32 rows.
void launch_skinny_norm(const float* x, const float* W, float* y, int rows, int C, int N, int epi,
                        float eps, hipStream_t st) {
  GN_CHECK(skinny_norm_supported(rows, C) && N % 4 == 0 && aligned16(x) && aligned16(W) &&
               aligned16(y) && (epi == EPI_STORE || epi == EPI_RELU2_SAVE),
           "skinny norm product: shape");
  GemmParams p{};
  p.A = x; p.lda = C; p.B = W; p.ldb = C; p.C = y; p.ldc = N;
  p.M = rows; p.N = N; p.K = C;
  p.epi = epi;
  p.alpha = 1.f;
  const int kv = C / 256;  // 16 waves
  const SkinnyKernel k =
      rows <= 16 ? skinny_kernel_n<1, 16, true>(kv) : skinny_kernel_n<2, 16, true>(kv);
  GN_CHECK(k != nullptr, "skinny norm product: width");
  hipLaunchKernelGGL(k, dim3((unsigned)ceil_div(N, 16)), dim3(1024), 0, st, p, 1, eps);
  GN_HIP(hipGetLastError());
}

// Runs d on the skinny engine: x.W^T with at most 32 rows (two 16-row blocks'
// x and weights fit the registers; 64 rows take the other engines), K a
// multiple of 64, N a multiple of 4.  K is split over up to 4 workgroups
// when the consumer can sum the partials (deferred sums) and the output
// tiles alone leave CUs idle.
bool gemm_skinny(const GemmDesc& d, GemmParams p, bool vec, hipStream_t st, DeviceArena* ws) {
  if (d.group != GEMM_GROUP_NONE || d.batch > 1 || d.force_splits > 0 || !vec) return false;
  if (!d.a_kcontig || !d.b_kcontig || d.M > 32 || d.K % 64 || d.K == 0 || d.N % 4) return false;
  if (d.epi != EPI_STORE && d.epi != EPI_ADD_SRC && d.epi != EPI_RELU2_SAVE &&
      d.epi != EPI_SOFTCAP)
    return false;
  if (d.ldc % 4 || !aligned16(d.C)) return false;
  if (d.epi == EPI_ADD_SRC && (!aligned16(d.aux) || d.ldaux % 4)) return false;
  if (d.epi == EPI_RELU2_SAVE && d.aux_out && (!aligned16(d.aux_out) || d.ldaux % 4)) return false;
  // GN_GEMM_SKINNY=0 leaves these products to the other engines (tests)
  if (const char* e = std::getenv("GN_GEMM_SKINNY"); e && std::atoi(e) == 0) return false;
  const bool can_defer = d.defer && ws && ((d.epi == EPI_STORE && d.alpha == 1.f) ||
                                           d.epi == EPI_ADD_SRC);
  if (d.defer) {
    GN_CHECK(d.ldc == d.N && ((d.epi == EPI_STORE && d.alpha == 1.f) ||
                              (d.epi == EPI_ADD_SRC && d.aux == d.C && d.ldaux == d.N)),
             "gemm: a deferred split-K sum needs a plain or in-place residual product");
    *d.defer = PendingSum{};
  }
  const int tiles = (int)ceil_div(d.N, 16);
  // a consumer that sums split-K partials: 4 waves and up to 4 splits
  int splits = 1;
  if (can_defer)
    for (int s = 2; s <= 4; s++)
      if ((d.K / 64) % s == 0 && tiles * s <= 256) splits = s;
  // long K behind few tiles: splits and a reduction launch (16 rows, N 768, K
  // 3072: 15.5 us unsplit, a workgroup's 196 KB being all one CU can have in
  // flight; 10 us split)
  const bool reduce = splits == 1 && ws && d.K >= 2048 && d.K % 256 == 0 && tiles <= 64;
  if (reduce) splits = 4;
  const bool wide = splits == 1 && tiles < 512 && d.K % 256 == 0;
  const int units = d.K / (wide ? 256 : 64) / splits;
  const int kv = largest_kv(units, max_kv(d.M <= 16 ? 1 : 2, wide ? 16 : 4));
  const int chunks = units / kv;
  p.part = nullptr;
  if (splits > 1)
    p.part = ws->get<float>(reduce ? std::string("gemm_splitk")
                                   : "gemm_splitk_defer" + std::to_string(d.defer_slot),
                            (size_t)splits * d.M * d.N);
  using namespace skinny;
  const SkinnyKernel k =
      wide ? (d.M <= 16 ? skinny_kernel_n<1, 16, false>(kv) : skinny_kernel_n<2, 16, false>(kv))
           : (d.M <= 16 ? skinny_kernel_n<1, 4, false>(kv) : skinny_kernel_n<2, 4, false>(kv));
  hipLaunchKernelGGL(k, dim3((unsigned)std::min(tiles, 512), (unsigned)splits),
                     dim3(wide ? 1024 : 256), 0, st, p, chunks, 0.f);
  GN_HIP(hipGetLastError());
  if (reduce) {
    p.splits = splits;
    launch_gemm_reduce(p, 1, st);
  } else if (splits > 1) {
    d.defer->part = p.part;
    d.defer->splits = splits;
    d.defer->stride = (int64_t)d.M * d.N;
  }
  return true;
}

}  // namespace gn
