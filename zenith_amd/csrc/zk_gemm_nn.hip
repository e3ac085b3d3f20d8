// zk_gemm_f16_nn: the fp16 GEMM on B[K,N] as wmma_matmul takes it. The main
// loop is gemm_mfma_kernel's; a slice of B goes to LDS as 64 rows of the
// tile's columns and its fragments come out of the transposing LDS read, so
// no transposed copy of B is made (4096^3: a 20 us launch that wrote 34 MB).
#include "zk_gemm_kernel.hpp"

namespace zk {
namespace {

template <int BM, int BN, int MS, int WM, int WN, typename OutT>
void launch_nn(GemmParams p, hipStream_t s) {
  const int grid = tile_grid(p, BM, BN);
  // the small tile's ring: as launch_64 in zk_gemm.hip
  if constexpr (BM == 64) {
    if (grid <= 512) {
      gemm_mfma_kernel<F16Op, BM, BN, MS, 128, 4, WM, WN, ZK_EPI_NONE, OutT, false, false, true>
          <<<grid, 64 * WM * WN, 0, s>>>(p);
      return;
    }
  }
  gemm_mfma_kernel<F16Op, BM, BN, MS, 128, 2, WM, WN, ZK_EPI_NONE, OutT, false, false, true>
      <<<grid, 64 * WM * WN, 0, s>>>(p);
}

// Tile by shape (us, one box, graph replays; 256x256 / 256x192 / 128x128 /
// 64x64): 4096^3 129 / 171 / 146 / 212; 4096x2304x768 30.6 / 27.3 / 28.5 /
// 29.8; 3000x2000x1504 43 / 38 / 31 / 43; 2048^3 50 / 44 / 30.7 / 30.6;
// 4096x768x768 24 / 21 / 13.6 / 12.6. The transpose that went before each of
// them took 5 to 20 us. Up to 128 rows a 256-row tile is at least half empty
// (256x192 / 128x128 or 64x64: 64x32000x768 21.8 / 14.4, 16x50264x768 36.2 / 21.4,
// 128x128000x4096 263 / 250; from 129 it is level or ahead: 129x32000x768 23.6 /
// 27.0).
template <typename OutT>
void run_nn(GemmParams p, hipStream_t s) {
  const int64_t tm = (p.M + 255) / 256, t256 = tm * ((p.N + 255) / 256),
                t192 = tm * ((p.N + 191) / 192),
                t128 = (int64_t)((p.M + 127) / 128) * ((p.N + 127) / 128);
  if (p.M > 128 && t256 >= 256 && (t192 + 255) / 256 * 3 >= (t256 + 255) / 256 * 4)
    launch_nn<256, 256, 32, 2, 4, OutT>(p, s);
  else if (p.M > 128 && t192 >= 160)
    launch_nn<256, 192, 32, 4, 2, OutT>(p, s);
  else if (t128 >= 256)
    launch_nn<128, 128, 32, 2, 2, OutT>(p, s);
  else
    launch_nn<64, 64, 16, 2, 2, OutT>(p, s);
}

}  // namespace
}  // namespace zk

using namespace zk;

extern "C" int zk_gemm_f16_nn(const void *A, const void *B, void *C, int64_t M, int64_t N,
                              int64_t K, int64_t lda, int64_t ldb, int64_t ldc, int out_dtype,
                              void *workspace, int64_t ws_bytes, void *stream) {
  const char *who = "zk_gemm_f16_nn";
  if (M < 0 || N < 0 || K < 0 || ws_bytes < 0) return fail(ZK_ERR_INVALID, "%s: negative size", who);
  if (M > 0x7fffffff || N > 0x7fffffff || K > 0x7fffffff)
    return fail(ZK_ERR_UNSUPPORTED, "%s: dimension exceeds int32", who);
  if (M == 0 || N == 0) return ZK_OK;
  if (!A || !B || !C) return fail(ZK_ERR_INVALID, "%s: null pointer", who);
  if (lda < K || ldb < N || ldc < N)
    return fail(ZK_ERR_INVALID, "%s: leading dimension too small", who);
  if (out_dtype != ZK_F16 && out_dtype != ZK_F32)
    return fail(ZK_ERR_UNSUPPORTED, "%s: out_dtype %d not supported", who, out_dtype);
  if (K == 0 || K % 8 || lda % 8 || ldb % 8 || !aligned16(A) || !aligned16(B))
    return fail(ZK_ERR_UNSUPPORTED,
                "%s: K, lda, ldb must be positive multiples of 8 and A, B 16-byte aligned", who);
  // 32-bit offsets: 256 rows of A, every row of B and those past K in the
  // last slice (at most 56; 192 leaves room)
  const int64_t lim = 0x7ffffff0LL;
  if (255 * lda * 2 + K * 2 >= lim || (K + 192) * ldb * 2 >= lim)
    return fail(ZK_ERR_UNSUPPORTED, "%s: operands too large for 32-bit addressing", who);
  GemmParams p{A, B, C, (int)M, (int)N, (int)K, lda, ldb, ldc, nullptr, nullptr, 0, 1.f, nullptr, 0};
  hipStream_t s = as_stream(stream);
  // the split of zk_gemm_f16_ws: whole, a product of few tiles can be faster
  // when timed alone (197x1000x768 6.7 us, 8.3 in 4 splits + reduction), but
  // its K-long fp32 sums round more (1.8e-7 of the result against 1.0e-7)
  const SplitPlan sp = plan_split(M, N, K, 2);
  if (workspace && sp.splits > 1 && ws_bytes >= split_ws_bytes(M, N, sp) && aligned16(workspace)) {
    GemmParams q = p;
    q.C = workspace;
    q.ldc = N;
    q.splits = sp.splits;
    q.nk_per = sp.nk_per;
    q.split_stride = M * N;
    launch_nn<64, 64, 16, 2, 2, float>(q, s);
    const float *ws = (const float *)workspace;
    if (out_dtype == ZK_F16)
      launch_reduce<f16>(ws, sp.splits, M * N, (int)M, (int)N, nullptr, nullptr, 0, (f16 *)C, ldc,
                         ZK_EPI_NONE, s);
    else
      launch_reduce<float>(ws, sp.splits, M * N, (int)M, (int)N, nullptr, nullptr, 0, (float *)C,
                           ldc, ZK_EPI_NONE, s);
  } else if (out_dtype == ZK_F16) {
    run_nn<f16>(p, s);
  } else {
    run_nn<float>(p, s);
  }
  return check_launch(who);
}
