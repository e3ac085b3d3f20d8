// GEMMs for gfx950.
//
// zk_gemm_f16 / zk_gemm_i8 share one MFMA kernel. Both operands are K-major
// in memory (A[M,K], W[N,K]) and the kernel is byte-generic: an fp16 MFMA
// step (32x32x16 or 16x16x32) and an int8 step (32x32x32 or 16x16x64) read
// the same 16 bytes per lane and operand, so one LDS layout serves both.
//
// Workgroup: 4 wavefronts in a 2 x 2 grid or 8 in a 2 x 4 / 4 x 2 grid,
// each owning a (BM/WM) x (BN/WN) wave tile made of MS x MS MFMA blocks
// (MS = 32 or 16). The macro tile is chosen per shape from measurements
// (pick_cfg): 8-wave 256-row tiles (two waves of one workgroup per SIMD)
// where the grid still fills the chip, small tiles with several workgroups
// per CU for the narrow projections.
//
// K is walked in slices of BKB bytes per row. A slice of A and W goes from
// global memory straight into LDS with buffer_load ... lds (16 bytes per
// lane, 1 KB per wavefront instruction, no VGPR staging), into a ring of
// ST stages; slices are issued ST-1 ahead, and each iteration has exactly
// one barrier, preceded by an explicit vmcnt wait that leaves the younger
// slices in flight. Rows are addressed through raw buffer descriptors that
// end at the last valid row, so loads past M / N return zeros; chunks past
// K are redirected out of range.
//
// LDS rows hold BKB bytes as 16-byte chunks; chunk c of row r sits at slot
// c ^ f(r), with f spreading the 16 rows one fragment read touches over
// 16 distinct 16-byte bank groups (a 256-byte bank period holds 2 rows of
// 128 bytes or 4 rows of 64 bytes).
//
// Epilogue: each wavefront stages one MS-row stripe of its wave tile in
// LDS as fp32 (after scale / bias / activation), then streams it out as
// 8-column vectors, adding the residual on the way; no workgroup barrier is
// needed between stripes.
//
// The B[K,N] (n-contiguous) layout of wmma_matmul: zk_gemm_f16_nn
// (zk_gemm_nn.hip) reads it with the transposing LDS read where its rows
// start on 16 bytes; otherwise the Python layer transposes it once
// (zk_transpose_f16).
//
// zk_gemm_f32 (the reference's fp32 `matmul`): small W[N,K] products run the
// same kernel on fp32 matrix instructions, larger ones and B[K,N] the
// bf16-split kernel of zk_gemm_f32s.hip, whose error against 64 bits is no
// larger than theirs, the rest an fp32 SIMT kernel (64x64 tiles, 4x4 outputs
// per thread).
#include <type_traits>

#include "zk_gemm_kernel.hpp"

namespace zk {

// ------------------------------------------------------------ dispatch ----
// Tile configurations (BM, BN, MS, BKB, ST, wave grid); the choice rule is
// in pick_cfg.
//   0: 256x256, 32x32 MFMA, 128-byte slices, 2-stage ring, 8 waves (2 x 4)
//   1: 128x128, 32x32, 128-byte slices, 2-stage ring (2 WG/CU)
//   2: 128x96,  16x16, 128-byte slices, 2-stage ring (2 WG/CU)
//   3: 64x64,   16x16, 128-byte slices, 2-stage ring (up to 5 WG/CU), or a
//      4-stage one (2 WG/CU) for at most 512 workgroups (see launch_64)
//   4: 128x96,  32x32, 128-byte slices, 3-stage ring, 4 waves (4 x 1)
//   5: 256x192, 32x32, 128-byte slices, 2-stage ring, 8 waves (4 x 2)
//   6: 128x96,  32x32, 128-byte slices, 2-stage ring, 4 waves (4 x 1; 2 WG/CU)
//   7: 64x96,   16x16, 128-byte slices, 3-stage ring (fp16; 2 WG/CU)
//   8: 64x128,  32x32, 128-byte slices, 3-stage ring (fp16; 2 WG/CU)
// The 8-wave tiles put two wavefronts of one workgroup on every SIMD, so
// one wave's barrier or memory wait is covered by the other's MFMAs.

// Returns false when no kernel of this configuration implements `epi` for
// these operand types (nothing is launched then): callers turn that into
// ZK_ERR_UNSUPPORTED instead of leaving the output unwritten.
template <class OP, int BM, int BN, int MS, int BKB, int ST, typename OutT, bool DEQ, int WM = 2,
          int WN = 2>
static bool launch_epi(GemmParams p, int epi, hipStream_t s) {
  const int grid = tile_grid(p, BM, BN);
#define ZK_L(E) \
  (gemm_mfma_kernel<OP, BM, BN, MS, BKB, ST, WM, WN, E, OutT, DEQ><<<grid, 64 * WM * WN, 0, s>>>(p), \
   true)
  switch (epi) {
    case ZK_EPI_NONE: return ZK_L(ZK_EPI_NONE);
    case ZK_EPI_BIAS: return ZK_L(ZK_EPI_BIAS);
    case ZK_EPI_BIAS_GELU_ERF: return ZK_L(ZK_EPI_BIAS_GELU_ERF);
    case ZK_EPI_BIAS_GELU_TANH: return ZK_L(ZK_EPI_BIAS_GELU_TANH);
    case ZK_EPI_BIAS_RESIDUAL:
      if constexpr (!std::is_same<OutT, int8_t>::value) return ZK_L(ZK_EPI_BIAS_RESIDUAL);
      return false;
    case ZK_EPI_BIAS_RELU: return ZK_L(ZK_EPI_BIAS_RELU);
    default:
      // the folded-LayerNorm epilogues: fp16 in and out; statistics need
      // wave tiles of whole kLnSeg-column segments
      if constexpr (std::is_same<OP, F16Op>::value && std::is_same<OutT, f16>::value && !DEQ) {
        if (epi == kEpiLnIn) return ZK_L(kEpiLnIn);
        if (epi == kEpiLnInGelu) return ZK_L(kEpiLnInGelu);
        if constexpr ((BN / WN) % kLnSeg == 0)
          if (epi == kEpiResStats) return ZK_L(kEpiResStats);
      }
      // the residual + statistics epilogue on the dequantised int8 product
      if constexpr (std::is_same<OP, I8Op>::value && std::is_same<OutT, f16>::value && DEQ &&
                    (BN / WN) % kLnSeg == 0)
        if (epi == kEpiResStats) return ZK_L(kEpiResStats);
      return false;
  }
#undef ZK_L
}

// The 128x96 tile of the residual + statistics epilogues: one workgroup per
// CU with a 3-stage ring (configuration 4) while every CU has at most one
// tile; beyond, a 2-stage ring (6) lets a CU hold two, whose second costs
// little (4608 x 768 x 3072, 288 tiles: 50.9 -> 35.8 us; 4096 rows, 256 tiles:
// 28.8 and 32.7).
static int cfg_128x96(int M, int N) {
  return (int64_t)((M + 127) / 128) * ((N + 95) / 96) <= 256 ? 4 : 6;
}

// The residual + statistics epilogue on fragment-ordered A (p.a_pk): the
// 128x96 tile of 4 x 1 waves that FFN-down runs on with row-major A.
template <class OP, bool DEQ, int EPI = kEpiResStats>
static void launch_frag_res_stats(GemmParams p, hipStream_t s) {
  const int grid = tile_grid(p, 128, 96);
  if (cfg_128x96(p.M, p.N) == 4)
    gemm_mfma_kernel<OP, 128, 96, 32, 128, 3, 4, 1, EPI, f16, DEQ, true><<<grid, 256, 0, s>>>(p);
  else
    gemm_mfma_kernel<OP, 128, 96, 32, 128, 2, 4, 1, EPI, f16, DEQ, true><<<grid, 256, 0, s>>>(p);
}

// Shape -> configuration, from measurements (us, bias epilogue, one box,
// graph replays). What decides is how many rounds of workgroups a tile needs:
// 256 CUs hold one workgroup of 0, 4 and 5 each, two of 1, 2, 6, 7 and 8 (the
// second at little cost), up to five of 3.
//   M < 1024: 64x64 unless the 128x96 tiles fill the CUs (few rows are split
//     along K by the callers with a workspace);
//   N > 1024, fewer than 256 tiles of 256x256: the smallest of 128x96 and
//     128x128 that fits in one round of two per CU, else 256x192, else
//     256x256 that fits in one of one per CU (M x 3072 x 768, erf-GELU;
//     128x96 / 128x128 / 256x192 / 256x256: M 1577 15.8 / 17.6 / 22.1 / 26.1,
//     2560 24.3 / 19.7 / 23.0 / 26.9, 3500 28.9 / 28.2 / 24.5 / 28.2, 4608
//     37.4 / 34.1 / 43.6 / 30.1; int8, re-quantising, the same order: 16.6 / 17.2 /
//     23.4 / 28.8, 25.2 / 18.5 / 24.6 / 29.8, 30.1 / 27.2 / 25.8 / 30.9, 37.6 / 32.5 /
//     46.3 / 31.6);
//   from 256 tiles of 256x256: that tile, unless 256x192 takes fewer whole
//     rounds times area (QKV at s512, 16384 x 2304: 576 tiles of 256x256, three
//     rounds with the last a quarter full, or 768 of 256x192);
//   N <= 1024: 256x192 once it fills the CUs (s512: FFN-down 96.5 -> 73.6 us).
//     Deep K (FFN-down, K >= 2048): the smallest tile with one round of one
//     per CU, then of two (M x 768 x 3072; 64x96 / 64x128 / 128x96 with three
//     stages / with two: M 1577 20.8 / 22.1 / 26.2 / 31.0, 2560 26.1 / 22.8 /
//     26.2 / 32.8, 4096 28.8 / 31.2 / 28.8 / 32.7, 4608 43.6 / 33.1 / 50.9 /
//     35.8, 6144 45 / 52 / 51.6 / 38.0; int8 keeps the 128x96 tiles, measured
//     in the encoder). Short K: 64x64 up to three tiles per CU, then 128x128
//     or 128x96 in one round (M x 768 x 768; 64x64 / 128x128 / 128x96: 4608 11.9 /
//     10.8 / 12.1, 6144 15.4 / 14.8 / 12.7, 8192 17.9 / 15.4 / 14.1; where 96 and
//     192 do not divide N, 64x64 / 128x128 / 256x192: 12288 x 512 x 512 13.4 / 12.5 /
//     15.3, 6144 x 1024 x 1024 22.9 / 20.3 / 24.7, 7000 x 1024 x 512 16.3 / 14.5 /
//     18.5).
static int pick_cfg(int M, int N, int K, bool f16) {
  if (forced_cfg() >= 0) return forced_cfg();
  auto tiles = [&](int bm, int bn) {
    return (int64_t)((M + bm - 1) / bm) * ((N + bn - 1) / bn);
  };
  const int64_t t256 = tiles(256, 256), t192 = tiles(256, 192), t128 = tiles(128, 128),
                t96 = tiles(128, 96);
  if (M < 1024) return t96 < 256 ? 3 : t128 >= 640 ? 1 : 2;
  if (N > 1024) {
    if (t256 >= 256) return (t192 + 255) / 256 * 3 < (t256 + 255) / 256 * 4 ? 5 : 0;
    return t96 <= 512 ? 2 : t128 <= 512 ? 1 : t192 <= 256 ? 5 : 0;
  }
  if (t192 >= 256) return 5;
  if (K >= 2048) {
    const int64_t t64 = tiles(64, 128);
    if (f16 && tiles(64, 96) <= 256) return 7;
    if (f16 && t64 <= 256) return 8;
    if (t96 <= 256) return 4;
    if (f16 && t64 <= 512) return 8;
    return t96 <= 512 ? 6 : 5;
  }
  if (!f16 || tiles(64, 64) <= 768) return 3;
  return t128 <= 256 ? 1 : t96 <= 512 ? 6 : t128 <= 512 ? 1 : 5;
}

// Every 32x32-MFMA tile has the fragment-ordered store; the 16x16 ones give
// way to 128x128 (2, whose one round it fits in as well) or 128x96.
static int frag_cfg(int cfg) { return cfg == 2 ? 1 : cfg == 3 || cfg == 7 ? 4 : cfg; }

// The 64x64 tile. Up to 512 workgroups (two per CU) nothing but its own ring
// hides a workgroup's memory latency, and in a model the weights come from
// HBM: four stages, all requested at the start. BERT encoder, s128, 12 layers,
// ring of 2 / 3 / 4 / 6 stages: b1 502 / 463 / 461 / 470 us, b2 554 / 471 /
// 459 / 473, b4 604 / 525 / 527 / 654 (6 stages leave one workgroup per CU).
// (b8 s128 with it for the split products alone 818, for all 796.) More
// workgroups hide each other's: 4096x768x768 (768 tiles) 10.0 / 10.8 / 12.0 us.
// Called over and over on the same weights it costs 0.2 to 0.4 us (2048x768x768,
// ring of 2 / 4: 7.4 / 7.7). The sums and their order are the same.
template <class OP, typename OutT, bool DEQ>
[[nodiscard]] static bool launch_64(GemmParams p, int epi, hipStream_t s) {
  const int64_t wgs = (int64_t)((p.M + 63) / 64) * ((p.N + 63) / 64) * (p.splits > 1 ? p.splits : 1);
  if (wgs <= 512) return launch_epi<OP, 64, 64, 16, 128, 4, OutT, DEQ>(p, epi, s);
  return launch_epi<OP, 64, 64, 16, 128, 2, OutT, DEQ>(p, epi, s);
}

// Returns whether a kernel was launched (see launch_epi).
template <class OP, typename OutT, bool DEQ>
[[nodiscard]] static bool launch_mfma(GemmParams p, int epi, hipStream_t s, int cfg = -1) {
  // fp32 products that reach this kernel have at most 256 tiles of 64x64
  // (plan_f32s takes the others)
  if constexpr (std::is_same<OP, F32Op>::value)
    return launch_64<OP, OutT, DEQ>(p, epi, s);
  else
  switch (cfg >= 0 ? cfg : pick_cfg(p.M, p.N, p.K, std::is_same<OP, F16Op>::value)) {
    case 0: return launch_epi<OP, 256, 256, 32, 128, 2, OutT, DEQ, 2, 4>(p, epi, s);
    case 1: return launch_epi<OP, 128, 128, 32, 128, 2, OutT, DEQ>(p, epi, s);
    case 2: return launch_epi<OP, 128, 96, 16, 128, 2, OutT, DEQ>(p, epi, s);
    case 4: return launch_epi<OP, 128, 96, 32, 128, 3, OutT, DEQ, 4, 1>(p, epi, s);
    case 5: return launch_epi<OP, 256, 192, 32, 128, 2, OutT, DEQ, 4, 2>(p, epi, s);
    case 6: return launch_epi<OP, 128, 96, 32, 128, 2, OutT, DEQ, 4, 1>(p, epi, s);
    case 7:
      if constexpr (std::is_same<OP, F16Op>::value)
        return launch_epi<OP, 64, 96, 16, 128, 3, OutT, DEQ>(p, epi, s);
      return false;
    case 8:
      if constexpr (std::is_same<OP, F16Op>::value)
        return launch_epi<OP, 64, 128, 32, 128, 3, OutT, DEQ>(p, epi, s);
      return false;
    default: return launch_64<OP, OutT, DEQ>(p, epi, s);
  }
}

// The status of a GEMM entry point after launch_mfma: unsupported when no
// kernel implements the epilogue for the chosen tile, else the launch check.
static int launched(bool ok, const char *who, int epi) {
  if (!ok) return fail(ZK_ERR_UNSUPPORTED, "%s: epilogue %d has no kernel for this shape", who, epi);
  return check_launch(who);
}

// --------------------------------------------------------------- split-K --
// p describes the final product (C, ldc, bias, residual); the partials go to
// ws (at least split_ws_bytes). OP is F16Op or F32Op.
// Returns whether both kernels were launched (false for an epilogue the
// reduction does not implement; nothing is launched then).
template <class OP, typename OutT>
[[nodiscard]] static bool launch_split(GemmParams p, int epi, const SplitPlan &sp, float *ws,
                                       hipStream_t s) {
  switch (epi) {
    case ZK_EPI_NONE: case ZK_EPI_BIAS: case ZK_EPI_BIAS_GELU_ERF: case ZK_EPI_BIAS_GELU_TANH:
    case ZK_EPI_BIAS_RESIDUAL: case ZK_EPI_BIAS_RELU: break;
    default: return false;
  }
  GemmParams q = p;
  q.C = ws;
  q.ldc = p.N;
  q.bias = nullptr;
  q.res = nullptr;
  q.splits = sp.splits;
  q.nk_per = sp.nk_per;
  q.split_stride = (int64_t)p.M * p.N;
  if (!launch_mfma<OP, float, false>(q, ZK_EPI_NONE, s, 3)) return false;
  launch_reduce<OutT>(ws, sp.splits, q.split_stride, p.M, p.N, (const OutT *)p.bias,
                      (const OutT *)p.res, p.ldr, (OutT *)p.C, p.ldc, epi, s);
  return true;
}

// ------------------------------------------------------------- fp32 SIMT --
template <bool TRANS_B>
__global__ __launch_bounds__(256) void gemm_f32_kernel(
    const float *__restrict__ A, const float *__restrict__ B,
    float *__restrict__ C, int M, int N, int K, int64_t lda, int64_t ldb,
    int64_t ldc) {
  __shared__ float As[16][64 + 4];
  __shared__ float Bs[16][64 + 4];
  const int tid = threadIdx.x, tx = tid & 15, ty = tid >> 4;
  const int m0 = blockIdx.y * 64, n0 = blockIdx.x * 64;
  float acc[4][4] = {};
  for (int k0 = 0; k0 < K; k0 += 16) {
    // A tile: 64 rows x 16 k, k fastest across lanes
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int idx = tid + v * 256, r = idx >> 4, k = idx & 15;
      const int gr = m0 + r, gk = k0 + k;
      As[k][r] = (gr < M && gk < K) ? A[(int64_t)gr * lda + gk] : 0.f;
    }
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int idx = tid + v * 256;
      if (TRANS_B) {  // W[N,K]: k fastest
        const int c = idx >> 4, k = idx & 15, gc = n0 + c, gk = k0 + k;
        Bs[k][c] = (gc < N && gk < K) ? B[(int64_t)gc * ldb + gk] : 0.f;
      } else {  // B[K,N]: n fastest
        const int k = idx >> 6, c = idx & 63, gc = n0 + c, gk = k0 + k;
        Bs[k][c] = (gc < N && gk < K) ? B[(int64_t)gk * ldb + gc] : 0.f;
      }
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      float a[4], b[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) a[i] = As[k][ty * 4 + i];
#pragma unroll
      for (int j = 0; j < 4; ++j) b[j] = Bs[k][tx * 4 + j];
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = fmaf(a[i], b[j], acc[i][j]);
    }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = m0 + ty * 4 + i;
    if (r >= M) continue;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int c = n0 + tx * 4 + j;
      if (c < N) C[(int64_t)r * ldc + c] = acc[i][j];
    }
  }
}

static int check_dims(const char *who, int64_t M, int64_t N, int64_t K) {
  if (M < 0 || N < 0 || K < 0) return fail(ZK_ERR_INVALID, "%s: negative size", who);
  if (M > 0x7fffffff || N > 0x7fffffff || K > 0x7fffffff)
    return fail(ZK_ERR_UNSUPPORTED, "%s: dimension exceeds int32", who);
  return ZK_OK;
}

// The MFMA kernel addresses a tile's rows through a buffer descriptor of
// (rows - 1) * ld + K bytes (rows <= 256) with 32-bit offsets, and pushes
// K-tail chunks out of range with the offset 0x7ffffff0; both operands'
// spans must stay below it.
static int check_span(const char *who, int64_t lda, int64_t ldb, int64_t K, int elem) {
  const int64_t lim = 0x7ffffff0LL;
  if (255 * lda * elem + K * elem >= lim || 255 * ldb * elem + K * elem >= lim)
    return fail(ZK_ERR_UNSUPPORTED,
                "%s: leading dimension / K too large for 32-bit tile addressing", who);
  return ZK_OK;
}

}  // namespace zk

using namespace zk;

int zk::gemm_f16_impl(const void *A, const void *B, void *C, int64_t M, int64_t N, int64_t K,
                      int64_t lda, int64_t ldb, int64_t ldc, int trans_b, int out_dtype,
                      const void *bias, const void *residual, int64_t ldr, int epilogue,
                      void *ws, int64_t ws_bytes, void *stream) {
  int st = check_dims("zk_gemm_f16", M, N, K);
  if (st) return st;
  if (M == 0 || N == 0) return ZK_OK;
  if (!A || !B || !C) return fail(ZK_ERR_INVALID, "zk_gemm_f16: null pointer");
  if (epilogue < ZK_EPI_NONE || epilogue > ZK_EPI_BIAS_RELU)
    return fail(ZK_ERR_INVALID, "zk_gemm_f16: bad epilogue %d", epilogue);
  if (epilogue != ZK_EPI_NONE && !bias)
    return fail(ZK_ERR_INVALID, "zk_gemm_f16: epilogue needs a bias");
  if (epilogue == ZK_EPI_BIAS_RESIDUAL && (!residual || ldr < N))
    return fail(ZK_ERR_INVALID, "zk_gemm_f16: residual epilogue needs residual and ldr >= N");
  if (!trans_b)
    return fail(ZK_ERR_UNSUPPORTED,
                "zk_gemm_f16: B[K,N] operand must be transposed to W[N,K] first "
                "(zk_transpose_f16)");
  if (lda < K || ldb < K || ldc < N)
    return fail(ZK_ERR_INVALID, "zk_gemm_f16: leading dimension too small");
  if (K % 8 || lda % 8 || ldb % 8 || !aligned16(A) || !aligned16(B))
    return fail(ZK_ERR_UNSUPPORTED,
                "zk_gemm_f16: K, lda, ldb must be multiples of 8 and A, B 16-byte aligned");
  if (out_dtype != ZK_F16 && out_dtype != ZK_F32)
    return fail(ZK_ERR_UNSUPPORTED, "zk_gemm_f16: out_dtype %d not supported", out_dtype);
  if (K == 0) return fail(ZK_ERR_UNSUPPORTED, "zk_gemm_f16: K == 0");
  if ((st = check_span("zk_gemm_f16", lda, ldb, K, 2))) return st;
  GemmParams p{A, B, C, (int)M, (int)N, (int)K, lda, ldb, ldc, bias, residual, ldr, 1.f, nullptr, 0};
  hipStream_t s = as_stream(stream);
  const SplitPlan sp = plan_split(M, N, K, 2);
  bool ok;
  if (ws && sp.splits > 1 && ws_bytes >= split_ws_bytes(M, N, sp) && aligned16(ws)) {
    if (out_dtype == ZK_F16) ok = launch_split<F16Op, f16>(p, epilogue, sp, (float *)ws, s);
    else ok = launch_split<F16Op, float>(p, epilogue, sp, (float *)ws, s);
  } else if (out_dtype == ZK_F16) {
    ok = launch_mfma<F16Op, f16, false>(p, epilogue, s);
  } else {
    ok = launch_mfma<F16Op, float, false>(p, epilogue, s);
  }
  return launched(ok, "zk_gemm_f16", epilogue);
}

extern "C" int zk_gemm_f16(const void *A, const void *B, void *C, int64_t M,
                           int64_t N, int64_t K, int64_t lda, int64_t ldb,
                           int64_t ldc, int trans_b, int out_dtype,
                           const void *bias, const void *residual, int64_t ldr,
                           int epilogue, void *stream) {
  return gemm_f16_impl(A, B, C, M, N, K, lda, ldb, ldc, trans_b, out_dtype, bias, residual, ldr,
                       epilogue, nullptr, 0, stream);
}

extern "C" int zk_gemm_f16_ws(const void *A, const void *B, void *C, int64_t M, int64_t N,
                              int64_t K, int64_t lda, int64_t ldb, int64_t ldc, int trans_b,
                              int out_dtype, const void *bias, const void *residual,
                              int64_t ldr, int epilogue, void *workspace, int64_t ws_bytes,
                              void *stream) {
  if (ws_bytes < 0) return fail(ZK_ERR_INVALID, "zk_gemm_f16_ws: negative workspace size");
  return gemm_f16_impl(A, B, C, M, N, K, lda, ldb, ldc, trans_b, out_dtype, bias, residual, ldr,
                       epilogue, workspace, ws_bytes, stream);
}

// Linear + residual + LayerNorm. A product that splits along K (and whose
// rows the wave LayerNorm can hold) runs as its split partials plus one
// LayerNorm launch that forms the rows from the partials; anything else as
// zk_gemm_f16_ws into T followed by zk_layernorm. Both give the pair's
// result bit for bit. Below 2048 rows of at most 1024 values each row gets a
// workgroup of four wavefronts to form it (BERT encoder per step, s128,
// pair -> partials: b1 0.602 -> 0.555 ms, b2 0.635 -> 0.581, b4 0.679 ->
// 0.626); otherwise one wavefront per row reads every split of its row,
// which needs at least 32 rows per split to pay (with it b1, 6 and 10
// splits of 128 rows, measured 0.604 -> 0.621 ms, b2 0.617, b4 0.646).
extern "C" int zk_gemm_f16_add_ln(const void *A, const void *W, const void *bias, const void *R,
                                  const void *gamma, const void *beta, void *T, void *Y,
                                  int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldw,
                                  float eps, void *workspace, int64_t ws_bytes, void *stream) {
  const char *who = "zk_gemm_f16_add_ln";
  int st = check_dims(who, M, N, K);
  if (st) return st;
  if (M == 0 || N == 0) return ZK_OK;
  if (!A || !W || !bias || !R || !gamma || !beta || !T || !Y)
    return fail(ZK_ERR_INVALID, "%s: null pointer", who);
  if (!(eps >= 0.0f)) return fail(ZK_ERR_INVALID, "%s: eps must be >= 0", who);
  if (ws_bytes < 0) return fail(ZK_ERR_INVALID, "%s: negative workspace size", who);
  if (lda < K || ldw < K) return fail(ZK_ERR_INVALID, "%s: leading dimension too small", who);
  if (K == 0) return fail(ZK_ERR_UNSUPPORTED, "%s: K == 0", who);
  if (K % 8 || lda % 8 || ldw % 8 || !aligned16(A) || !aligned16(W))
    return fail(ZK_ERR_UNSUPPORTED,
                "%s: K, lda, ldw must be multiples of 8 and A, W 16-byte aligned", who);
  if ((st = check_span(who, lda, ldw, K, 2))) return st;
  hipStream_t s = as_stream(stream);
  const SplitPlan sp = plan_split(M, N, K, 2);
  const float *ws = (const float *)workspace;
  const bool wide = ln_partials_wide_ok(M, N), narrow = !wide && sp.splits * 32 <= M;
  if (ws && sp.splits > 1 && ws_bytes >= split_ws_bytes(M, N, sp) && (narrow || wide) &&
      ln_partials_ok(ws, M * N, bias, R, gamma, beta, Y, M, N)) {
    GemmParams q{A, W, workspace, (int)M, (int)N, (int)K, lda, ldw, N, nullptr, nullptr, 0, 1.f,
                 nullptr, 0};
    q.splits = sp.splits;
    q.nk_per = sp.nk_per;
    q.split_stride = M * N;
    if (!launch_mfma<F16Op, float, false>(q, ZK_EPI_NONE, s, 3))
      return fail(ZK_ERR_UNSUPPORTED, "%s: no partial-product kernel for this shape", who);
    if ((st = check_launch(who))) return st;
    return ln_add_partials_f16(ws, sp.splits, M * N, bias, R, gamma, beta, Y, M, N, eps, wide, s);
  }
  st = gemm_f16_impl(A, W, T, M, N, K, lda, ldw, N, 1, ZK_F16, bias, nullptr, 0, ZK_EPI_BIAS,
                     workspace, ws_bytes, stream);
  if (st) return st;
  return zk_layernorm(T, R, gamma, beta, Y, M, N, eps, ZK_F16, stream);
}

// Fused QKV projection + attention (sequences of 64 or 128 tokens, head dim
// 64): one 256 x 192 tile per workgroup, the q, k and v columns of one head
// for 256 rows, with the attention of the tile's sequences in its epilogue.
static void launch_qkv_attn(GemmParams p, hipStream_t s) {
  p.tiles_n = p.N / 192;
  p.tiles_m = (p.M + 255) / 256;
  const int grid = p.tiles_m * p.tiles_n;
  int gm = 1;
  const int per_xcd = (grid + 7) / 8;
  while (gm * 2 <= p.tiles_m && gm * gm * 4 <= per_xcd) gm *= 2;
  p.group_m = gm;
  gemm_mfma_kernel<F16Op, 256, 192, 32, 128, 2, 4, 2, kEpiQkvAttn, f16, false>
      <<<grid, 512, 0, s>>>(p);
}

static int qkv_attn_impl(const char *who, const void *X, const void *Wqkv, const void *bqkv,
                         const float *ln_part, float ln_eps, const float *ln_s,
                         const float *ln_c, float *ln_out, void *ctx, int64_t batch,
                         int64_t seq, int64_t hidden, int64_t heads, const int32_t *valid_lens,
                         float scale, void *stream, bool frag = false) {
  if (batch < 0 || seq <= 0 || hidden <= 0 || heads <= 0)
    return fail(ZK_ERR_INVALID, "%s: bad size", who);
  if (batch == 0) return ZK_OK;
  if (!X || !Wqkv || !ctx) return fail(ZK_ERR_INVALID, "%s: null pointer", who);
  if (!ln_part && !bqkv) return fail(ZK_ERR_INVALID, "%s: null bias", who);
  if (ln_part && (!ln_s || !ln_c || !(ln_eps >= 0.f)))
    return fail(ZK_ERR_INVALID, "%s: LayerNorm needs column sums, offsets and eps >= 0", who);
  if (!aligned8(ln_part) || !aligned8(ln_out))
    return fail(ZK_ERR_UNSUPPORTED, "%s: statistics arrays must be 8-byte aligned", who);
  if (ln_part && (hidden % kLnSeg || hidden / kLnSeg > kLnMaxParts))
    return fail(ZK_ERR_UNSUPPORTED, "%s: hidden must be a multiple of %d, at most %d", who,
                kLnSeg, kLnSeg * kLnMaxParts);
  if (hidden != heads * 64)
    return fail(ZK_ERR_UNSUPPORTED, "%s: head dim must be 64 (hidden %lld, heads %lld)", who,
                (long long)hidden, (long long)heads);
  if (seq != 64 && seq != 128)
    return fail(ZK_ERR_UNSUPPORTED, "%s: seq must be 64 or 128 (got %lld)", who, (long long)seq);
  if (!(scale > 0.0f) || scale == __builtin_inff())
    return fail(ZK_ERR_INVALID, "%s: scale must be finite and > 0", who);
  if (batch > 0x7fffffff / seq) return fail(ZK_ERR_UNSUPPORTED, "%s: batch * seq exceeds int32", who);
  const int64_t M = batch * seq, N = 3 * hidden, K = hidden;
  int st = check_dims(who, M, N, K);
  if (st) return st;
  if (!aligned16(X) || !aligned16(Wqkv) || !aligned8(ctx))
    return fail(ZK_ERR_UNSUPPORTED, "%s: X and Wqkv must be 16-byte, ctx 8-byte aligned", who);
  if (frag && !aligned16(ctx))
    return fail(ZK_ERR_UNSUPPORTED, "%s: ctx in fragment order must be 16-byte aligned", who);
  if ((st = check_span(who, K, K, K, 2))) return st;
  GemmParams p{X, Wqkv, ctx, (int)M, (int)N, (int)K, K, K, hidden, bqkv, nullptr, 0, 1.f, nullptr, 0};
  p.seq = (int)seq;
  p.batch = (int)batch;
  p.valid_lens = valid_lens;
  p.scale_log2 = scale * 1.4426950408889634f;
  p.ln_part = ln_part;
  p.ln_nparts = (int)(K / kLnSeg);
  p.ln_eps = ln_eps;
  p.ln_s = ln_s;
  p.ln_c = ln_c;
  p.ln_out = ln_out;
  p.c_pk = frag;
  launch_qkv_attn(p, as_stream(stream));
  return check_launch(who);
}

extern "C" int zk_qkv_attn_f16(const void *X, const void *Wqkv, const void *bqkv, void *ctx,
                               int64_t batch, int64_t seq, int64_t hidden, int64_t heads,
                               const int32_t *valid_lens, float scale, void *stream) {
  return qkv_attn_impl("zk_qkv_attn_f16", X, Wqkv, bqkv, nullptr, 0.f, nullptr, nullptr, nullptr,
                       ctx, batch, seq, hidden, heads, valid_lens, scale, stream);
}

extern "C" int zk_qkv_attn_f16_ln(const void *X, const void *Wqkv, const float *ln_part,
                                  float ln_eps, const float *ln_s, const float *ln_c,
                                  float *ln_out, void *ctx, int64_t batch, int64_t seq,
                                  int64_t hidden, int64_t heads, const int32_t *valid_lens,
                                  float scale, void *stream) {
  if (!ln_part) return fail(ZK_ERR_INVALID, "zk_qkv_attn_f16_ln: null statistics");
  return qkv_attn_impl("zk_qkv_attn_f16_ln", X, Wqkv, nullptr, ln_part, ln_eps, ln_s, ln_c,
                       ln_out, ctx, batch, seq, hidden, heads, valid_lens, scale, stream);
}

extern "C" int zk_qkv_attn_f16_frag(const void *X, const void *Wqkv, const void *bqkv,
                                    const float *ln_part, float ln_eps, const float *ln_s,
                                    const float *ln_c, float *ln_out, void *ctx, int64_t batch,
                                    int64_t seq, int64_t hidden, int64_t heads,
                                    const int32_t *valid_lens, float scale, void *stream) {
  return qkv_attn_impl("zk_qkv_attn_f16_frag", X, Wqkv, ln_part ? nullptr : bqkv, ln_part,
                       ln_eps, ln_s, ln_c, ln_out, ctx, batch, seq, hidden, heads, valid_lens,
                       scale, stream, true);
}

// Operand checks of the folded-LayerNorm GEMMs: fp16, W[N,K], dense-enough
// rows in multiples of 8, 16-byte aligned.
static int check_ln_gemm(const char *who, const void *A, const void *W, const void *C, int64_t M,
                         int64_t N, int64_t K, int64_t lda, int64_t ldw, int64_t ldc) {
  int st = check_dims(who, M, N, K);
  if (st) return st;
  if (!A || !W || !C) return fail(ZK_ERR_INVALID, "%s: null pointer", who);
  if (lda < K || ldw < K || ldc < N) return fail(ZK_ERR_INVALID, "%s: leading dimension too small", who);
  if (K == 0 || K % 8 || lda % 8 || ldw % 8 || ldc % 8 || !aligned16(A) || !aligned16(W) ||
      !aligned16(C))
    return fail(ZK_ERR_UNSUPPORTED,
                "%s: K and the leading dimensions must be multiples of 8, operands 16-byte "
                "aligned", who);
  return check_span(who, lda, ldw, K, 2);
}

static int check_i8(const char *who, const int8_t *A, const int8_t *W, const void *C, int64_t M,
                    int64_t N, int64_t K, int64_t lda, int64_t ldw, int64_t ldc, int epilogue);

// The residual / statistics operands of zk_gemm_f16_res_stats and
// zk_gemm_i8_res_stats, checked, then the launch on the configurations whose
// wave tiles are one statistics segment wide: 256x192 (8 waves) once it
// fills the CUs, else 128x96 (4 waves).
template <class OP, bool DEQ>
static int res_stats_run(const char *who, GemmParams p, const float *res_ln, const void *res_gamma,
                         const void *res_beta, float *part_out, void *stream) {
  const int64_t M = p.M, N = p.N;
  if (!p.bias || !p.res || !part_out)
    return fail(ZK_ERR_INVALID, "%s: null bias, residual or statistics", who);
  if (N % kLnSeg) return fail(ZK_ERR_UNSUPPORTED, "%s: N must be a multiple of %d", who, kLnSeg);
  if (res_ln && (!res_gamma || !res_beta))
    return fail(ZK_ERR_INVALID, "%s: residual LayerNorm needs gamma and beta", who);
  if (p.ldr < N) return fail(ZK_ERR_INVALID, "%s: ldr < N", who);
  if (p.ldr % 8 || !aligned16(p.res))
    return fail(ZK_ERR_UNSUPPORTED, "%s: residual rows must be 16-byte aligned", who);
  if (!aligned8(res_ln) || !aligned8(part_out) || !aligned16(res_gamma) || !aligned16(res_beta))
    return fail(ZK_ERR_UNSUPPORTED,
                "%s: statistics 8-byte, gamma and beta 16-byte aligned", who);
  p.res_ln = res_ln;
  p.res_gamma = res_gamma;
  p.res_beta = res_beta;
  p.part_out = part_out;
  if (p.a_pk) {
    launch_frag_res_stats<OP, DEQ>(p, as_stream(stream));
    return launched(true, who, kEpiResStats);
  }
  const int64_t t192 = (M + 255) / 256 * (N / 192);
  const bool ok = launch_mfma<OP, f16, DEQ>(
      p, kEpiResStats, as_stream(stream),
      M >= 1024 && N % 192 == 0 && t192 >= 160 ? 5 : cfg_128x96(p.M, p.N));
  return launched(ok, who, kEpiResStats);
}

extern "C" int zk_gemm_f16_res_stats(const void *A, const void *W, void *C, int64_t M, int64_t N,
                                     int64_t K, int64_t lda, int64_t ldw, int64_t ldc,
                                     const void *bias, const void *res, int64_t ldr,
                                     const float *res_ln, const void *res_gamma,
                                     const void *res_beta, float *part_out, void *stream) {
  const char *who = "zk_gemm_f16_res_stats";
  int st = check_ln_gemm(who, A, W, C, M, N, K, lda, ldw, ldc);
  if (st) return st;
  if (M == 0 || N == 0) return ZK_OK;
  GemmParams p{A, W, C, (int)M, (int)N, (int)K, lda, ldw, ldc, bias, res, ldr, 1.f, nullptr, 0};
  return res_stats_run<F16Op, false>(who, p, res_ln, res_gamma, res_beta, part_out, stream);
}

extern "C" int zk_gemm_f16_frag(const void *A, const void *W, void *C, int64_t M, int64_t N,
                                int64_t K, int64_t ldw, int64_t ldc, const void *bias,
                                void *stream) {
  const char *who = "zk_gemm_f16_frag";
  int st = check_ln_gemm(who, A, W, C, M, N, K, K, ldw, ldc);
  if (st) return st;
  if (M == 0 || N == 0) return ZK_OK;
  if (K % 64) return fail(ZK_ERR_UNSUPPORTED, "%s: K must be a multiple of 64", who);
  if (!bias) return fail(ZK_ERR_INVALID, "%s: null bias", who);
  GemmParams p{A, W, C, (int)M, (int)N, (int)K, K, ldw, ldc, bias, nullptr, 0, 1.f, nullptr, 0};
  p.a_pk = A;
  launch_frag_res_stats<F16Op, false, ZK_EPI_BIAS>(p, as_stream(stream));
  return check_launch(who);
}

extern "C" int zk_gemm_f16_res_stats_frag(const void *A, const void *W, void *C, int64_t M,
                                          int64_t N, int64_t K, int64_t ldw, int64_t ldc,
                                          const void *bias, const void *res, int64_t ldr,
                                          const float *res_ln, const void *res_gamma,
                                          const void *res_beta, float *part_out, void *stream) {
  const char *who = "zk_gemm_f16_res_stats_frag";
  int st = check_ln_gemm(who, A, W, C, M, N, K, K, ldw, ldc);
  if (st) return st;
  if (M == 0 || N == 0) return ZK_OK;
  if (K % 64) return fail(ZK_ERR_UNSUPPORTED, "%s: K must be a multiple of 64", who);
  GemmParams p{A, W, C, (int)M, (int)N, (int)K, K, ldw, ldc, bias, res, ldr, 1.f, nullptr, 0};
  p.a_pk = A;
  return res_stats_run<F16Op, false>(who, p, res_ln, res_gamma, res_beta, part_out, stream);
}

extern "C" int zk_gemm_i8_res_stats(const int8_t *A, const int8_t *W, void *C, int64_t M,
                                    int64_t N, int64_t K, int64_t lda, int64_t ldw, int64_t ldc,
                                    float s_x, const float *s_w, const void *bias,
                                    const void *res, int64_t ldr, const float *res_ln,
                                    const void *res_gamma, const void *res_beta, float *part_out,
                                    void *stream) {
  const char *who = "zk_gemm_i8_res_stats";
  int st = check_i8(who, A, W, C, M, N, K, lda, ldw, ldc, ZK_EPI_BIAS);
  if (st || M == 0 || N == 0) return st;
  if (!s_w || !(s_x > 0.f)) return fail(ZK_ERR_INVALID, "%s: s_w and s_x > 0 are required", who);
  if (ldc % 8 || !aligned16(C))
    return fail(ZK_ERR_UNSUPPORTED, "%s: ldc must be a multiple of 8 and C 16-byte aligned", who);
  GemmParams p{A, W, C, (int)M, (int)N, (int)K, lda, ldw, ldc, bias, res, ldr, s_x, s_w, 0};
  return res_stats_run<I8Op, true>(who, p, res_ln, res_gamma, res_beta, part_out, stream);
}

static int gemm_f16_ln(const char *who, const void *A, const void *W, void *C, int64_t M,
                       int64_t N, int64_t K, int64_t lda, int64_t ldw, int64_t ldc,
                       const float *ln_part, float ln_eps, const float *ln_s, const float *ln_c,
                       float *ln_out, int epilogue, bool frag, void *stream) {
  int st = check_ln_gemm(who, A, W, C, M, N, K, lda, ldw, ldc);
  if (st) return st;
  if (M == 0 || N == 0) return ZK_OK;
  if (!ln_part || !ln_s || !ln_c || !(ln_eps >= 0.f))
    return fail(ZK_ERR_INVALID, "%s: null statistics, column sums or offsets, or eps < 0", who);
  if (epilogue != ZK_EPI_BIAS && epilogue != ZK_EPI_BIAS_GELU_ERF)
    return fail(ZK_ERR_UNSUPPORTED, "%s: epilogue must be ZK_EPI_BIAS or ZK_EPI_BIAS_GELU_ERF", who);
  if (K % kLnSeg || K / kLnSeg > kLnMaxParts)
    return fail(ZK_ERR_UNSUPPORTED, "%s: K must be a multiple of %d, at most %d", who, kLnSeg,
                kLnSeg * kLnMaxParts);
  if (!aligned8(ln_part) || !aligned8(ln_out) || !aligned16(ln_s) || !aligned16(ln_c))
    return fail(ZK_ERR_UNSUPPORTED,
                "%s: statistics 8-byte, column sums and offsets 16-byte aligned", who);
  GemmParams p{A, W, C, (int)M, (int)N, (int)K, lda, ldw, ldc, nullptr, nullptr, 0, 1.f, nullptr, 0};
  p.ln_part = ln_part;
  p.ln_nparts = (int)(K / kLnSeg);
  p.ln_eps = ln_eps;
  p.ln_s = ln_s;
  p.ln_c = ln_c;
  p.ln_out = ln_out;
  const int epi = epilogue == ZK_EPI_BIAS ? kEpiLnIn : kEpiLnInGelu;
  int cfg = pick_cfg(p.M, p.N, p.K, true);
  if (frag) {
    p.c_pk = 1;
    cfg = frag_cfg(cfg);
  }
  return launched(launch_mfma<F16Op, f16, false>(p, epi, as_stream(stream), cfg), who, epi);
}

extern "C" int zk_gemm_f16_ln(const void *A, const void *W, void *C, int64_t M, int64_t N,
                              int64_t K, int64_t lda, int64_t ldw, int64_t ldc,
                              const float *ln_part, float ln_eps, const float *ln_s,
                              const float *ln_c, float *ln_out, int epilogue, void *stream) {
  return gemm_f16_ln("zk_gemm_f16_ln", A, W, C, M, N, K, lda, ldw, ldc, ln_part, ln_eps, ln_s,
                     ln_c, ln_out, epilogue, false, stream);
}

extern "C" int zk_gemm_f16_ln_frag(const void *A, const void *W, void *C, int64_t M, int64_t N,
                                   int64_t K, int64_t lda, int64_t ldw, const float *ln_part,
                                   float ln_eps, const float *ln_s, const float *ln_c,
                                   float *ln_out, void *stream) {
  const char *who = "zk_gemm_f16_ln_frag";
  if (N % 64) return fail(ZK_ERR_UNSUPPORTED, "%s: N must be a multiple of 64", who);
  return gemm_f16_ln(who, A, W, C, M, N, K, lda, ldw, N, ln_part, ln_eps, ln_s, ln_c, ln_out,
                     ZK_EPI_BIAS_GELU_ERF, true, stream);
}

// Shape / operand checks shared by the int8 entry points.
static int check_i8(const char *who, const int8_t *A, const int8_t *W, const void *C, int64_t M,
                    int64_t N, int64_t K, int64_t lda, int64_t ldw, int64_t ldc, int epilogue) {
  int st = check_dims(who, M, N, K);
  if (st) return st;
  if (M == 0 || N == 0) return ZK_OK;
  if (!A || !W || !C) return fail(ZK_ERR_INVALID, "%s: null pointer", who);
  if (epilogue < ZK_EPI_NONE || epilogue > ZK_EPI_BIAS_RELU)
    return fail(ZK_ERR_INVALID, "%s: bad epilogue %d", who, epilogue);
  if (lda < K || ldw < K || ldc < N)
    return fail(ZK_ERR_INVALID, "%s: leading dimension too small", who);
  if (K % 16 || lda % 16 || ldw % 16 || !aligned16(A) || !aligned16(W))
    return fail(ZK_ERR_UNSUPPORTED,
                "%s: K, lda, ldw must be multiples of 16 and A, W 16-byte aligned", who);
  if (K == 0) return fail(ZK_ERR_UNSUPPORTED, "%s: K == 0", who);
  // |acc| <= 128 * 128 * K, which reaches 2^31 (int32 overflow) at K = 131072
  if (K >= 131072)
    return fail(ZK_ERR_UNSUPPORTED, "%s: K >= 131072 could overflow int32 accumulators", who);
  return check_span(who, lda, ldw, K, 1);
}

extern "C" int zk_gemm_i8(const int8_t *A, const int8_t *W, void *C, int64_t M,
                          int64_t N, int64_t K, int64_t lda, int64_t ldw,
                          int64_t ldc, float s_x, const float *s_w,
                          const void *bias, const void *residual, int64_t ldr,
                          int epilogue, int out_dtype, void *stream) {
  int st = check_i8("zk_gemm_i8", A, W, C, M, N, K, lda, ldw, ldc, epilogue);
  if (st || M == 0 || N == 0) return st;
  hipStream_t s = as_stream(stream);
  GemmParams p{A, W, C, (int)M, (int)N, (int)K, lda, ldw, ldc, bias, residual, ldr, s_x, s_w, 0};
  if (out_dtype == ZK_I32) {
    if (epilogue != ZK_EPI_NONE)
      return fail(ZK_ERR_INVALID, "zk_gemm_i8: int32 output takes no epilogue");
    return launched(launch_mfma<I8Op, int32_t, false>(p, ZK_EPI_NONE, s), "zk_gemm_i8",
                    ZK_EPI_NONE);
  }
  if (!s_w) return fail(ZK_ERR_INVALID, "zk_gemm_i8: dequantised output needs s_w");
  if (!(s_x > 0.f)) return fail(ZK_ERR_INVALID, "zk_gemm_i8: s_x must be > 0");
  if (epilogue != ZK_EPI_NONE && !bias)
    return fail(ZK_ERR_INVALID, "zk_gemm_i8: epilogue needs a bias");
  if (epilogue == ZK_EPI_BIAS_RESIDUAL && (!residual || ldr < N))
    return fail(ZK_ERR_INVALID, "zk_gemm_i8: residual epilogue needs residual and ldr >= N");
  bool ok;
  if (out_dtype == ZK_F16) ok = launch_mfma<I8Op, f16, true>(p, epilogue, s);
  else if (out_dtype == ZK_F32) ok = launch_mfma<I8Op, float, true>(p, epilogue, s);
  else return fail(ZK_ERR_UNSUPPORTED, "zk_gemm_i8: out_dtype %d not supported", out_dtype);
  return launched(ok, "zk_gemm_i8", epilogue);
}

extern "C" int zk_gemm_i8_requant(const int8_t *A, const int8_t *W, int8_t *Q, int64_t M,
                                  int64_t N, int64_t K, int64_t lda, int64_t ldw,
                                  int64_t ldq, float s_x, const float *s_w,
                                  const void *bias, int epilogue, float s_out,
                                  void *stream) {
  int st = check_i8("zk_gemm_i8_requant", A, W, Q, M, N, K, lda, ldw, ldq, epilogue);
  if (st || M == 0 || N == 0) return st;
  if (epilogue == ZK_EPI_BIAS_RESIDUAL)
    return fail(ZK_ERR_INVALID, "zk_gemm_i8_requant: no residual epilogue for int8 output");
  if (!s_w) return fail(ZK_ERR_INVALID, "zk_gemm_i8_requant: s_w is required");
  if (!(s_x > 0.f) || !(s_out > 0.f))
    return fail(ZK_ERR_INVALID, "zk_gemm_i8_requant: s_x and s_out must be > 0");
  if (epilogue != ZK_EPI_NONE && !bias)
    return fail(ZK_ERR_INVALID, "zk_gemm_i8_requant: epilogue needs a bias");
  GemmParams p{A, W, Q, (int)M, (int)N, (int)K, lda, ldw, ldq, bias, nullptr, 0, s_x, s_w, 0};
  p.s_q = s_out;
  return launched(launch_mfma<I8Op, int8_t, true>(p, epilogue, as_stream(stream)),
                  "zk_gemm_i8_requant", epilogue);
}

extern "C" int zk_gemm_i8_requant_frag(const int8_t *A, const int8_t *W, int8_t *Q, int64_t M,
                                       int64_t N, int64_t K, int64_t lda, int64_t ldw,
                                       float s_x, const float *s_w, const void *bias,
                                       int epilogue, float s_out, void *stream) {
  const char *who = "zk_gemm_i8_requant_frag";
  int st = check_i8(who, A, W, Q, M, N, K, lda, ldw, N, epilogue);
  if (st || M == 0 || N == 0) return st;
  if (N % 128) return fail(ZK_ERR_UNSUPPORTED, "%s: N must be a multiple of 128", who);
  if (epilogue == ZK_EPI_BIAS_RESIDUAL)
    return fail(ZK_ERR_INVALID, "%s: no residual epilogue for int8 output", who);
  if (!s_w) return fail(ZK_ERR_INVALID, "%s: s_w is required", who);
  if (!(s_x > 0.f) || !(s_out > 0.f)) return fail(ZK_ERR_INVALID, "%s: s_x and s_out must be > 0", who);
  if (epilogue != ZK_EPI_NONE && !bias) return fail(ZK_ERR_INVALID, "%s: epilogue needs a bias", who);
  if (!aligned16(Q)) return fail(ZK_ERR_UNSUPPORTED, "%s: Q must be 16-byte aligned", who);
  GemmParams p{A, W, Q, (int)M, (int)N, (int)K, lda, ldw, N, bias, nullptr, 0, s_x, s_w, 0};
  p.s_q = s_out;
  p.c_pk = 1;
  const int cfg = frag_cfg(pick_cfg(p.M, p.N, p.K, false));
  return launched(launch_mfma<I8Op, int8_t, true>(p, epilogue, as_stream(stream), cfg), who,
                  epilogue);
}

extern "C" int zk_gemm_i8_res_stats_frag(const int8_t *A, const int8_t *W, void *C, int64_t M,
                                         int64_t N, int64_t K, int64_t ldw, int64_t ldc,
                                         float s_x, const float *s_w, const void *bias,
                                         const void *res, int64_t ldr, const float *res_ln,
                                         const void *res_gamma, const void *res_beta,
                                         float *part_out, void *stream) {
  const char *who = "zk_gemm_i8_res_stats_frag";
  int st = check_i8(who, A, W, C, M, N, K, K, ldw, ldc, ZK_EPI_BIAS);
  if (st || M == 0 || N == 0) return st;
  if (K % 128) return fail(ZK_ERR_UNSUPPORTED, "%s: K must be a multiple of 128", who);
  if (!aligned16(A)) return fail(ZK_ERR_UNSUPPORTED, "%s: A must be 16-byte aligned", who);
  if (!s_w || !(s_x > 0.f)) return fail(ZK_ERR_INVALID, "%s: s_w and s_x > 0 are required", who);
  if (ldc % 8 || !aligned16(C))
    return fail(ZK_ERR_UNSUPPORTED, "%s: ldc must be a multiple of 8 and C 16-byte aligned", who);
  GemmParams p{A, W, C, (int)M, (int)N, (int)K, K, ldw, ldc, bias, res, ldr, s_x, s_w, 0};
  p.a_pk = A;
  return res_stats_run<I8Op, true>(who, p, res_ln, res_gamma, res_beta, part_out, stream);
}

// Epilogue of the SIMT fp32 path, in place on C: the same operations, in the
// same order, as the MFMA kernel's epilogue.
template <int EPI>
__global__ __launch_bounds__(256) void f32_epilogue_kernel(float *__restrict__ C, int64_t ldc,
                                                           int64_t M, int64_t N,
                                                           const float *__restrict__ bias,
                                                           const float *__restrict__ res,
                                                           int64_t ldr) {
  const int64_t total = M * N, stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < total; i += stride) {
    const int64_t r = i / N, c = i % N;
    float v = epilogue<EPI>(C[r * ldc + c], bias[c]);
    if (EPI == ZK_EPI_BIAS_RESIDUAL) v += res[r * ldr + c];
    C[r * ldc + c] = v;
  }
}

static int gemm_f32_impl(const float *A, const float *B, float *C, int64_t M, int64_t N,
                         int64_t K, int64_t lda, int64_t ldb, int64_t ldc, int trans_b, void *ws,
                         int64_t ws_bytes, void *stream, const float *bias = nullptr,
                         const float *res = nullptr, int64_t ldr = 0, int epi = ZK_EPI_NONE,
                         const char *who = "zk_gemm_f32") {
  int st = check_dims(who, M, N, K);
  if (st) return st;
  if (M == 0 || N == 0) return ZK_OK;
  if (!A || !B || !C) return fail(ZK_ERR_INVALID, "%s: null pointer", who);
  if (lda < K || ldc < N || (trans_b ? ldb < K : ldb < N))
    return fail(ZK_ERR_INVALID, "%s: leading dimension too small", who);
  hipStream_t s = as_stream(stream);
  // The matrix kernel with fp32 products takes a W[N,K] operand with 16-byte
  // rows; buffer offsets of a 256-row tile must fit in 31 bits.
  const bool matrix = trans_b && K > 0 && K % 4 == 0 && lda % 4 == 0 && ldb % 4 == 0 &&
                      aligned16(A) && aligned16(B) &&
                      255 * (lda + ldb) * 4 + 2 * K * 4 < 0x7ffffff0LL;
  // the bf16-split kernel's offsets: 128 rows of A or W, 8 rows of B[K,N]. Where
  // 32 rows of B pass 31 bits (N above 17 million) few rows stay on the SIMT
  // kernel: M x K x 17.4e6, SIMT / split: 2 x 8 0.6 / 2.0 ms, 64 x 64 4.1 / 3.5,
  // 256 x 64 16.3 / 8.4.
  const bool span = 127 * lda * 4 + K * 4 < 0x7ffffff0LL &&
                    (trans_b ? 127 * ldb * 4 + K * 4
                             : (M < 64 ? 31 : 7) * ldb * 4 + N * 4) < 0x7ffffff0LL;
  const F32Plan fp =
      span ? plan_f32s(M, N, K, matrix ? F32Other::kMatrix : F32Other::kFma) : F32Plan{0, 1, 0};
  if (fp.tile) {
    F32sParams p{A, B, C, (int)M, (int)N, (int)K, lda, ldb, ldc, bias, res, ldr};
    const bool split = ws && fp.splits > 1 && ws_bytes >= f32s_ws_bytes(M, N, fp) && aligned16(ws);
    launch_f32s(p, trans_b, epi, fp, split ? (float *)ws : nullptr, s);
    return check_launch(who);
  }
  if (matrix) {
    GemmParams p{A, B, C, (int)M, (int)N, (int)K, lda, ldb, ldc, bias, res, ldr, 1.f, nullptr, 0};
    const SplitPlan sp = plan_split(M, N, K, 4);
    bool ok;
    if (ws && sp.splits > 1 && ws_bytes >= split_ws_bytes(M, N, sp) && aligned16(ws))
      ok = launch_split<F32Op, float>(p, epi, sp, (float *)ws, s);
    else
      ok = launch_mfma<F32Op, float, false>(p, epi, s);
    return launched(ok, who, epi);
  }
  if ((M + 63) / 64 > 65535)  // the SIMT kernel's grid; the others' have one dimension
    return fail(ZK_ERR_UNSUPPORTED, "%s: M too large", who);
  dim3 grid((unsigned)((N + 63) / 64), (unsigned)((M + 63) / 64));
  if (trans_b)
    gemm_f32_kernel<true><<<grid, 256, 0, s>>>(A, B, C, (int)M, (int)N, (int)K, lda, ldb, ldc);
  else
    gemm_f32_kernel<false><<<grid, 256, 0, s>>>(A, B, C, (int)M, (int)N, (int)K, lda, ldb, ldc);
  if (epi != ZK_EPI_NONE) {
    int64_t g = (M * N + 255) / 256;
    if (g > 4096) g = 4096;
#define ZK_E(E) f32_epilogue_kernel<E><<<(unsigned)g, 256, 0, s>>>(C, ldc, M, N, bias, res, ldr)
    switch (epi) {
      case ZK_EPI_BIAS: ZK_E(ZK_EPI_BIAS); break;
      case ZK_EPI_BIAS_GELU_ERF: ZK_E(ZK_EPI_BIAS_GELU_ERF); break;
      case ZK_EPI_BIAS_GELU_TANH: ZK_E(ZK_EPI_BIAS_GELU_TANH); break;
      case ZK_EPI_BIAS_RESIDUAL: ZK_E(ZK_EPI_BIAS_RESIDUAL); break;
      case ZK_EPI_BIAS_RELU: ZK_E(ZK_EPI_BIAS_RELU); break;
    }
#undef ZK_E
  }
  return check_launch(who);
}

extern "C" int zk_gemm_f32(const float *A, const float *B, float *C, int64_t M,
                           int64_t N, int64_t K, int64_t lda, int64_t ldb,
                           int64_t ldc, int trans_b, void *stream) {
  return gemm_f32_impl(A, B, C, M, N, K, lda, ldb, ldc, trans_b, nullptr, 0, stream);
}

extern "C" int zk_gemm_f32_ws(const float *A, const float *B, float *C, int64_t M, int64_t N,
                              int64_t K, int64_t lda, int64_t ldb, int64_t ldc, int trans_b,
                              void *workspace, int64_t ws_bytes, void *stream) {
  if (ws_bytes < 0) return fail(ZK_ERR_INVALID, "zk_gemm_f32_ws: negative workspace size");
  return gemm_f32_impl(A, B, C, M, N, K, lda, ldb, ldc, trans_b, workspace, ws_bytes, stream);
}

extern "C" int zk_linear_f32(const float *X, const float *W, float *Y, int64_t M, int64_t N,
                             int64_t K, int64_t ldx, int64_t ldw, int64_t ldy,
                             const float *bias, const float *residual, int64_t ldr,
                             int epilogue, void *workspace, int64_t ws_bytes, void *stream) {
  if (ws_bytes < 0) return fail(ZK_ERR_INVALID, "zk_linear_f32: negative workspace size");
  if (epilogue < ZK_EPI_NONE || epilogue > ZK_EPI_BIAS_RELU)
    return fail(ZK_ERR_INVALID, "zk_linear_f32: bad epilogue %d", epilogue);
  if (epilogue != ZK_EPI_NONE && !bias)
    return fail(ZK_ERR_INVALID, "zk_linear_f32: epilogue needs a bias");
  if (epilogue == ZK_EPI_BIAS_RESIDUAL && (!residual || ldr < N))
    return fail(ZK_ERR_INVALID, "zk_linear_f32: residual epilogue needs residual and ldr >= N");
  return gemm_f32_impl(X, W, Y, M, N, K, ldx, ldw, ldy, 1, workspace, ws_bytes, stream, bias,
                       residual, ldr, epilogue, "zk_linear_f32");
}

extern "C" int64_t zk_gemm_workspace_size(int64_t M, int64_t N, int64_t K, int dtype) {
  if (M <= 0 || N <= 0 || K <= 0) return 0;
  if (dtype == ZK_F16) return split_ws_bytes(M, N, plan_split(M, N, K, 2));
  if (dtype == ZK_F32) {
    // whatever layout and alignment the product will have
    int64_t most = split_ws_bytes(M, N, plan_split(M, N, K, 4));
    for (F32Other o : {F32Other::kMatrix, F32Other::kFma}) {
      const int64_t n = f32s_ws_bytes(M, N, plan_f32s(M, N, K, o));
      if (n > most) most = n;
    }
    return most;
  }
  return 0;
}
