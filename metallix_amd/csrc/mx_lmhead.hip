// mx_lmhead.hip -- a bf16 lm_head GEMM for gfx950 (mxs_lmhead_bf16): the
// logits producer whose epilogue writes the tile statistics of
// mxs_epilogue.h for mxs_finish_tiles.
//
// logits[n][v] = sum_k hidden[n][k] weight[v][k] (bf16 in, f32 accumulate),
// the lm_head of a Qwen3-shaped forward (the reference computes it in MLX
// before its picks, crates/models/qwen/src/forward.rs:1745-1761).  One
// 512-thread workgroup per 256-row vocabulary tile; wave w owns the tile's
// vocabulary rows 32 w .. 32 w + 31 against every batch row (at most 64), as
// 2 x 4 blocks of v_mfma_f32_16x16x32_bf16 (A: 16 vocabulary rows x 32 k, B:
// 32 k x 16 batch rows; lane l holds row l % 16 and k (l / 16) 8 .. + 7 of
// each, 16 contiguous bytes; D: lane l holds vocabulary rows (l / 16) 4 + j
// of batch row l % 16).  The weights stream from HBM once (the roofline:
// V K 2 bytes); the hidden states pass through LDS once per workgroup.
//
// The weight stream bounds it, and how a line of it is fetched matters: one
// load instruction takes 64 bytes of 16 rows, half of each 128-byte line.
// With four waves of 64 rows and loads per 32-k step, the line's second half
// was asked for a step later, after the other waves' loads had passed through
// the vector cache.  Eight waves of 32 rows hold 64 k of each row in the same
// registers, and both halves are loaded back to back: 64 x 1024 x 151936
// 89.8 -> 84.0 us (350 MB at 3.9 -> 4.2 TB/s), 64 x 4096 x 37984 104.6 ->
// 95.0 us, 7 x 512 x 200000 49.6 -> 44.9 us.  Also measured there, in the
// first shape: nontemporal weight loads 93.2 us (106.7 with four waves);
// three workgroups on a CU, which spills, 152.9 us.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/mx_sampler.h"
#include "mxs_ctx.h"
#include "mxs_device.h"
#include "mxs_epilogue.h"

namespace mxs {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

static_assert(sizeof(EpiTileStat) == MXS_TILE_STAT_BYTES && EPI_TILE == MXS_TILE_TOKENS, "the header's tile layout");

constexpr uint32_t LM_ROWS = 64;   // batch rows per launch (four 16-row MFMA blocks)
constexpr uint32_t LM_KC = 128;    // hidden-state k staged in LDS per chunk
constexpr int LM_NT = 512;         // threads per workgroup
constexpr int LM_WPS = 4;          // waves per SIMD: two workgroups on a CU
constexpr int LM_MB = (int)EPI_TILE / 16 / (LM_NT / 64);   // 16-row vocabulary blocks per wave
constexpr uint32_t LM_ST = LM_NT / LM_ROWS;                // threads that stage a batch row's chunk
constexpr uint32_t LM_SQ = LM_KC / LM_ST / 8u;             // their 16-byte pieces
constexpr uint32_t LM_BST = LM_KC + 8u;   // LDS row stride (bf16): rows 16 B apart in the banks

template <bool STATS>
__global__ __launch_bounds__(LM_NT, LM_WPS) void lmhead_kernel(const __bf16* __restrict__ H,
                                                               const __bf16* __restrict__ W, uint32_t rows,
                                                               uint32_t K, uint32_t V, float* __restrict__ logits,
                                                               uint64_t ld, EpiTileStat* __restrict__ stats,
                                                               uint32_t ntiles) {
  __shared__ EpiPartial part[LM_NT / 64][LM_ROWS];
  __shared__ __align__(16) __bf16 Bs[2][LM_ROWS * LM_BST];   // staged hidden-state chunks
  const uint32_t tile = blockIdx.x, w = threadIdx.x >> 6, l = threadIdx.x & 63u;
  const uint32_t lr = l & 15u, lg = l >> 4;
  const uint32_t vw = tile * EPI_TILE + w * (LM_MB * 16u);   // this wave's first vocabulary row
  // weight rows, clamped in range (the clamped rows' results are dropped)
  const __bf16* ap[LM_MB];
#pragma unroll
  for (int mb = 0; mb < LM_MB; ++mb) {
    const uint32_t v = min(vw + (uint32_t)mb * 16u + lr, V - 1u);
    ap[mb] = W + (uint64_t)v * K + lg * 8u;
  }
  f32x4 acc[LM_MB][4];
#pragma unroll
  for (int mb = 0; mb < LM_MB; ++mb)
#pragma unroll
    for (int nb = 0; nb < 4; ++nb) acc[mb][nb] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  // The hidden states pass through LDS in chunks of LM_KC k, double
  // buffered: thread t stages 16 k of row t / 8 (rows clamped; the clamped
  // rows' results are dropped), once per workgroup instead of once per wave.
  const uint32_t sn = min(threadIdx.x / LM_ST, rows - 1u), sk = (threadIdx.x % LM_ST) * (LM_KC / LM_ST);
  const __bf16* hsrc = H + (uint64_t)sn * K + sk;
  bf16x8 st[LM_SQ];
  auto stage_load = [&](uint32_t c) {
#pragma unroll
    for (int j = 0; j < (int)LM_SQ; ++j) st[j] = *reinterpret_cast<const bf16x8*>(hsrc + c * LM_KC + 8u * (uint32_t)j);
  };
  auto stage_store = [&](uint32_t buf) {
    __bf16* dst = &Bs[buf][(threadIdx.x / LM_ST) * LM_BST + sk];
#pragma unroll
    for (int j = 0; j < (int)LM_SQ; ++j) *reinterpret_cast<bf16x8*>(dst + 8u * (uint32_t)j) = st[j];
  };
  // The weights stream from HBM into registers two 64-k steps ahead: step
  // s + 2's rows load while step s's products issue.  The loads are
  // unconditional (past the last step they repeat it, in bounds, unused) so
  // the memory counter waits stay exact.
  const uint32_t pairs = K / 64u, nch = K / LM_KC;
  bf16x8 a[2][LM_MB][2];
  auto load_a = [&](bf16x8 (&d)[LM_MB][2], uint32_t s) {
    const uint32_t k0 = min(s, pairs - 1u) * 64u;
#pragma unroll
    for (int mb = 0; mb < LM_MB; ++mb)
#pragma unroll
      for (int h = 0; h < 2; ++h) d[mb][h] = *reinterpret_cast<const bf16x8*>(ap[mb] + k0 + 32u * (uint32_t)h);
  };
  stage_load(0u);
  load_a(a[0], 0u);
  load_a(a[1], 1u);
  stage_store(0u);
  __syncthreads();
  for (uint32_t c = 0; c < nch; ++c) {
    if (c + 1u < nch) stage_load(c + 1u);
    const __bf16* bs = &Bs[c & 1u][0];
#pragma unroll
    for (uint32_t p = 0; p < LM_KC / 64u; ++p) {
#pragma unroll
      for (uint32_t h = 0; h < 2u; ++h) {
        bf16x8 b[4];
#pragma unroll
        for (int nb = 0; nb < 4; ++nb)
          b[nb] = *reinterpret_cast<const bf16x8*>(bs + ((uint32_t)nb * 16u + lr) * LM_BST + p * 64u + h * 32u + lg * 8u);
#pragma unroll
        for (int mb = 0; mb < LM_MB; ++mb)
#pragma unroll
          for (int nb = 0; nb < 4; ++nb)
            acc[mb][nb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[p][mb][h], b[nb], acc[mb][nb], 0, 0, 0);
      }
      load_a(a[p], c * (LM_KC / 64u) + p + 2u);
    }
    if (c + 1u < nch) stage_store((c + 1u) & 1u);
    __syncthreads();
  }
  // acc[mb][nb][j]: token vw + 16 mb + 4 lg + j of batch row 16 nb + lr
#pragma unroll
  for (int nb = 0; nb < 4; ++nb) {
    const uint32_t n = (uint32_t)nb * 16u + lr;
    EpiPartial p = epi_empty();
#pragma unroll
    for (int mb = 0; mb < LM_MB; ++mb) {
      const uint32_t v0 = vw + (uint32_t)mb * 16u + lg * 4u;
      if (v0 < V) {   // V % 4 == 0: the quad is in range
        if (n < rows) *reinterpret_cast<f32x4*>(logits + (uint64_t)n * ld + v0) = acc[mb][nb];
        if (STATS) {
#pragma unroll
          for (int j = 0; j < 4; ++j) epi_add(p, acc[mb][nb][j]);
        }
      }
    }
    if (STATS) {
      epi_xor(p, 16);
      epi_xor(p, 32);
      if (lg == 0u) part[w][n] = p;
    }
  }
  if (STATS) {
    __syncthreads();
    if (threadIdx.x < rows) {
      const uint32_t n = threadIdx.x;
      EpiPartial p = part[0][n];
#pragma unroll
      for (int q = 1; q < LM_NT / 64; ++q) epi_merge(p, part[q][n]);
      epi_store(&stats[(uint64_t)n * ntiles + tile], p);
    }
  }
}

}  // namespace mxs

extern "C" int mxs_lmhead_bf16(mxs_ctx* ctx, const void* hidden, const void* weight, uint32_t rows,
                               uint32_t hidden_dim, uint32_t vocab, float* logits, uint64_t logits_stride,
                               void* tile_stats) {
  using namespace mxs;
  if (!ctx) return MXS_EINVAL;
  if (rows == 0) return MXS_OK;
  if (!hidden || !weight || !logits) return fail(ctx, MXS_EINVAL, "hidden, weight and logits are required");
  if (rows > LM_ROWS) return fail(ctx, MXS_EINVAL, "rows must be at most 64");
  if (hidden_dim == 0 || hidden_dim % LM_KC) return fail(ctx, MXS_EINVAL, "hidden_dim must be a positive multiple of 128");
  if (vocab == 0 || vocab % 4u) return fail(ctx, MXS_EINVAL, "vocab must be a positive multiple of 4");
  if (logits_stride < vocab || logits_stride % 4u) return fail(ctx, MXS_EINVAL, "logits_stride must be >= vocab and a multiple of 4");
  if (((uintptr_t)hidden | (uintptr_t)weight | (uintptr_t)logits) % 16u)
    return fail(ctx, MXS_EINVAL, "hidden, weight and logits must be 16-byte aligned");
  const uint32_t ntiles = (vocab + EPI_TILE - 1u) / EPI_TILE;
  int prev = 0;
  (void)hipGetDevice(&prev);
  if (prev != ctx->device) (void)hipSetDevice(ctx->device);
  const __bf16* H = reinterpret_cast<const __bf16*>(hidden);
  const __bf16* W = reinterpret_cast<const __bf16*>(weight);
  EpiTileStat* S = reinterpret_cast<EpiTileStat*>(tile_stats);
  if (S)
    hipLaunchKernelGGL(lmhead_kernel<true>, dim3(ntiles), dim3(LM_NT), 0, ctx->stream, H, W, rows, hidden_dim, vocab,
                       logits, logits_stride, S, ntiles);
  else
    hipLaunchKernelGGL(lmhead_kernel<false>, dim3(ntiles), dim3(LM_NT), 0, ctx->stream, H, W, rows, hidden_dim, vocab,
                       logits, logits_stride, S, ntiles);
  hipError_t e = hipGetLastError();
  if (prev != ctx->device) (void)hipSetDevice(prev);
  if (e != hipSuccess) return hip_fail(ctx, e, "lmhead_kernel launch");
  return MXS_OK;
}
