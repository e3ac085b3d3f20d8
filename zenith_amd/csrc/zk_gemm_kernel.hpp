// The MFMA GEMM kernel behind the fp16 and int8 products and the small fp32
// ones (zk_gemm.hip describes it), in a header so that its instantiations
// can be spread over several sources.
#pragma once
#include <type_traits>

#include "zk_attn_tile.hpp"
#include "zk_splitk.hpp"

namespace zk {

struct GemmParams {
  const void *A;
  const void *B;
  void *C;
  int M, N, K;
  int64_t lda, ldb, ldc;
  const void *bias;
  const void *res;
  int64_t ldr;
  float s_x;
  const float *s_w;
  int tiles_n;
  int tiles_m;
  int group_m;
  float s_q;  // int8 output: scale of the re-quantisation
  // split-K: workgroup (tile t, split s) = blockIdx t * splits + s covers K
  // slices [s * nk_per, +nk_per) and writes its fp32 partial tile to
  // C + s * split_stride (C is then the workspace, ldc = N)
  int splits;
  int nk_per;
  int64_t split_stride;
  // fused QKV projection + attention (kEpiQkvAttn): sequences of `seq`
  // rows, `batch` of them, key-padding lengths, softmax scale * log2(e)
  int seq;
  int batch;
  const int32_t *valid_lens;
  float scale_log2;
  // LayerNorm of the A rows folded into the GEMM (kEpiLnIn*, and the fused
  // attention when ln_part is set): A holds the LN input x, the weight is
  // gamma-scaled (W'[n,k] = W[n,k] gamma[k]) and the epilogue forms
  //   rstd[m] (acc - mean[m] ln_s[n]) + ln_c[n],
  // ln_s = column sums of W', ln_c = beta . W^T + bias. mean / rstd come from
  // the per-row partial statistics ln_part [M][ln_nparts] of (mean, M2) over
  // kLnSeg-column segments; tile column 0 writes them to ln_out [M] if set.
  const float *ln_part;
  int ln_nparts;
  float ln_eps;
  const float *ln_s;
  const float *ln_c;
  float *ln_out;
  // kEpiResStats: the residual is LN(res) with res_ln [M] (mean, rstd) and
  // fp16 res_gamma / res_beta when res_ln is set; the fp16-rounded outputs'
  // per-row (mean, M2) over kLnSeg-column segments go to part_out
  // [M][N / kLnSeg].
  const float *res_ln;
  const void *res_gamma;
  const void *res_beta;
  float *part_out;
  // Fragment order, the layout of an fp16 MFMA operand of 32 rows: for row
  // block rb (rows 32 rb .. +31) and k-step ks (columns 16 ks .. +15) of an
  // R x K matrix, the 1 KB at byte (rb * K / 16 + ks) * 1024 holds lane l's
  // 16 bytes, X[32 rb + l % 32][16 ks + 8 (l / 32) .. +7], at byte 16 l.
  // a_pk: A in fragment order (kernels instantiated with APK, K a multiple
  // of 64; lda unused): each fragment is one 1 KB DMA into LDS.
  // c_pk: C written in fragment order (kEpiLnInGelu; ldc unused).
  const void *a_pk;
  int c_pk;
};

// Internal epilogues (not public ZK_EPI_* values): the fused QKV projection +
// attention; bias + residual (optionally LayerNorm-ed on the fly) with
// per-row partial statistics of the output; and the folded LayerNorm of the
// input rows, without or with erf-GELU.
constexpr int kEpiQkvAttn = 100;
constexpr int kEpiResStats = 101;
constexpr int kEpiLnIn = 102;
constexpr int kEpiLnInGelu = 103;

// Row statistics travel as (mean, M2) partials of kLnSeg-column segments
// (the 96-column wave tiles of the producing GEMM); a consumer holds at most
// kLnMaxParts of them per row in registers (rows of up to 1536 values).
constexpr int kLnSeg = 96;
constexpr int kLnMaxParts = 16;

// (mean, rstd) of a row of nparts x kLnSeg values from its partial
// (mean, M2) pairs (Chan et al.'s pairwise update for equal counts, in a
// fixed order).
__device__ __forceinline__ float2 ln_merge(const float2 (&pr)[kLnMaxParts], int nparts,
                                           float eps) {
  float sm = 0.f;
#pragma unroll
  for (int q = 0; q < kLnMaxParts; ++q)
    if (q < nparts) sm += pr[q].x;
  const float mean = sm / (float)nparts;
  float m2 = 0.f, dev = 0.f;
#pragma unroll
  for (int q = 0; q < kLnMaxParts; ++q)
    if (q < nparts) {
      const float d = pr[q].x - mean;
      m2 += pr[q].y;
      dev = fmaf(d, d, dev);
    }
  const float var = fmaf((float)kLnSeg, dev, m2) / ((float)kLnSeg * (float)nparts);
  return make_float2(mean, 1.0f / sqrtf(var + eps));
}

// MFMA step on 16 bytes per lane and operand. MS = 32: lane l supplies row
// l % 32, bytes [16 * (l / 32), +16) of the 32-byte k-step; the result
// register r of lane l is D[8 * (r / 4) + 4 * (l / 32) + r % 4][l % 32].
// MS = 16: lane l supplies row l % 16, bytes [16 * (l / 16), +16) of the
// 64-byte k-step; register r is D[4 * (l / 16) + r][l % 16].
template <int MS> struct F16Mma;
template <> struct F16Mma<32> {
  typedef f32x16 Acc;
  static constexpr int R = 16;
  static __device__ __forceinline__ Acc mma(f16x8 a, f16x8 b, Acc c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
  }
};
template <> struct F16Mma<16> {
  typedef f32x4 Acc;
  static constexpr int R = 4;
  static __device__ __forceinline__ Acc mma(f16x8 a, f16x8 b, Acc c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
  }
};
template <int MS> struct I8Mma;
template <> struct I8Mma<32> {
  typedef i32x16 Acc;
  static constexpr int R = 16;
  static __device__ __forceinline__ Acc mma(i32x4 a, i32x4 b, Acc c) {
    return __builtin_amdgcn_mfma_i32_32x32x32_i8(a, b, c, 0, 0, 0);
  }
};
template <> struct I8Mma<16> {
  typedef i32x4 Acc;
  static constexpr int R = 4;
  static __device__ __forceinline__ Acc mma(i32x4 a, i32x4 b, Acc c) {
    return __builtin_amdgcn_mfma_i32_16x16x64_i8(a, b, c, 0, 0, 0);
  }
};

// fp32 on the matrix cores: 16 bytes per lane and operand are four fp32
// values, k0 + 4 * (lane slot) + j, consumed by four chained fp32 MFMAs in
// which element j of every lane is the operand (16x16x4: lane quarter = k
// index). The four products together cover 16 consecutive k.
template <int MS> struct F32Mma;
template <> struct F32Mma<16> {
  typedef f32x4 Acc;
  static constexpr int R = 4;
  static __device__ __forceinline__ Acc mma(f32x4 a, f32x4 b, Acc c) {
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[0], b[0], c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[1], b[1], c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[2], b[2], c, 0, 0, 0);
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a[3], b[3], c, 0, 0, 0);
  }
};

struct F16Op {
  typedef f16x8 Frag;
  template <int MS> using Mma = F16Mma<MS>;
  static constexpr int kElem = 2;
};
struct F32Op {
  typedef f32x4 Frag;
  template <int MS> using Mma = F32Mma<MS>;
  static constexpr int kElem = 4;
};
struct I8Op {
  typedef i32x4 Frag;
  template <int MS> using Mma = I8Mma<MS>;
  static constexpr int kElem = 1;
};

template <int BKB>
__device__ __forceinline__ int lds_slot(int row, int c) {
  return BKB == 128 ? (c ^ ((row >> 1) & 7)) : (c ^ ((row >> 2) & 3));
}

// B[K,N] tiles (BNK): a slice of 64 rows of BN columns, 16-byte chunk c of
// row k in slot c ^ bnk_swz(k). A transposing fragment read gives each group
// of 16 lanes 2 chunks of 4 consecutive rows, and the LDS serves it in two
// passes that pair the groups (0, 1) and (2, 3), or (0, 2) and (1, 3): the
// rows of a group go to the four 64-byte quarters of the 256-byte bank period
// (rows of BN % 128 != 0 columns advance by half a period already), and
// groups 8 rows apart to the two halves of a quarter.
template <int BN>
__device__ __forceinline__ int bnk_swz(int k) {
  return (BN % 128 == 0 ? 4 * (k & 3) : 4 * ((k >> 1) & 1)) ^ (2 * (((k >> 3) ^ (k >> 4)) & 1));
}
// The B fragment of k-step ks and columns n .. n + MS - 1: two transposing
// reads of 4 k each. In each group of 16 lanes output lane i receives element
// i % 4 of source lanes i / 4, 4 + i / 4, ..: source lane s reads row s / 4,
// columns 4 (s % 4) .. +3, and lane i ends with column i of the group at 4
// consecutive k. Bs is restrict-qualified so that the reads carry alias
// information (without it each waits for every LDS DMA in flight).
template <int BN, int MS>
__device__ __forceinline__ f16x8 read_bnk(const f16 *__restrict__ Bs, int ks, int n, int lane) {
  static_assert(BN % 64 == 0, "B[K,N] tile");
  const int grp = lane >> 4, sl = lane & 15;
  const int k = MS == 32 ? ks * 16 + 8 * (grp >> 1) + (sl >> 2) : ks * 32 + 8 * grp + (sl >> 2);
  const int ch = (n + (MS == 32 ? 16 * (grp & 1) : 0)) / 8 + ((sl & 3) >> 1), in = 4 * (sl & 1);
  const f16x4 lo = lds_read_tr16(Bs + k * BN + ((ch ^ bnk_swz<BN>(k)) << 3) + in);
  const f16x4 hi = lds_read_tr16(Bs + (k + 4) * BN + ((ch ^ bnk_swz<BN>(k + 4)) << 3) + in);
  return f16x8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
}

constexpr int epi_pitch16(int w) {
  int p = (w + 3) / 4 * 4;
  while (p % 64 != 16 && p % 64 != 48) p += 4;
  return p;
}

template <class OP, int BM, int BN, int MS, int BKB, int ST, int WM = 2, int WN = 2>
struct GemmCfg {
  static constexpr int NW = WM * WN, NT = 64 * NW;
  static constexpr int WTM = BM / WM, WTN = BN / WN;
  static constexpr int TM = WTM / MS, TN = WTN / MS;
  static constexpr int CH = BKB / 16;          // 16-byte chunks per LDS row
  static constexpr int RPI = 1024 / BKB;       // rows per wavefront DMA instruction
  static constexpr int IA = BM / RPI / NW;     // DMA instructions per wave per slice
  static constexpr int IB = BN / RPI / NW;
  static constexpr int STAGE = (BM + BN) * BKB;
  static constexpr int KCH = MS == 32 ? 2 : 4;  // chunks per MFMA k-step
  static constexpr int KS = CH / KCH;          // MFMA k-steps per slice
  // fp32 words per epilogue LDS row, chosen so one register's worth of
  // writes (32 columns x 2 rows 4 apart for MS = 32; 16 columns x 4
  // consecutive rows for MS = 16) covers 64 distinct banks.
  static constexpr int EPITCH = MS == 32 ? (WTN % 16 == 8 ? WTN : WTN + 8 - WTN % 16 + (WTN % 16 > 8 ? 16 : 0))
                                         : epi_pitch16(WTN);
  static constexpr int EPI_BYTES = NW * MS * EPITCH * 4;
  static constexpr int SMEM = ST * STAGE > EPI_BYTES ? ST * STAGE : EPI_BYTES;
  static_assert(BKB == 64 || BKB == 128, "slice width");
  static_assert(WTM % MS == 0 && WTN % MS == 0, "wave tile must be a multiple of the MFMA block");
  static_assert(BM % (RPI * NW) == 0 && BN % (RPI * NW) == 0, "DMA split");
  static_assert(KS >= 2 && KS % 2 == 0, "k-steps per slice must be even");
  static_assert(ST >= 2 && (ST - 1) * (IA + IB) <= 63, "vmcnt range");
  static_assert(SMEM <= 160 * 1024, "LDS budget");
  static_assert(WTN % 8 == 0, "epilogue vectors");
};

// Scheduling hint for one k-step: NR LDS fragment reads spread evenly over
// NM MFMAs (a read, then its share of MFMAs), so read latency hides under
// matrix work instead of being waited for in front of it.
template <int NR, int NM, int R = 0>
__device__ __forceinline__ void interleave() {
  if constexpr (R < NR) {
    __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // DS read
    __builtin_amdgcn_sched_group_barrier(0x008, NM / NR + (R < NM % NR ? 1 : 0), 0);  // MFMA
    interleave<NR, NM, R + 1>();
  }
}

// Waves per SIMD the register allocation must allow: as many workgroups
// per CU as the LDS ring admits (NW / 4 waves per SIMD each), capped at 3.
constexpr int gemm_waves_per_eu(int smem_bytes, int nw) {
  return nw == 8 ? 2 : smem_bytes <= 53 * 1024 ? 3 : smem_bytes <= 80 * 1024 ? 2 : 1;
}

template <class OP, int BM, int BN, int MS, int BKB, int ST, int WM, int WN, int EPI, typename OutT,
          bool DEQ, bool APK = false, bool BNK = false>
__global__ __launch_bounds__(64 * WM * WN)
__attribute__((amdgpu_waves_per_eu(gemm_waves_per_eu(GemmCfg<OP, BM, BN, MS, BKB, ST, WM, WN>::SMEM,
                                                     WM * WN))))
void gemm_mfma_kernel(GemmParams p) {
  typedef GemmCfg<OP, BM, BN, MS, BKB, ST, WM, WN> G;
  typedef typename OP::template Mma<MS> MM;
  typedef typename OP::Frag Frag;
  constexpr int TM = G::TM, TN = G::TN, IA = G::IA, IB = G::IB, CH = G::CH;
  constexpr int WTM = G::WTM, WTN = G::WTN, KS = G::KS, KCH = G::KCH, R = MM::R;
  constexpr int NRD = TM + (BNK ? 2 : 1) * TN;  // LDS reads per k-step
  __shared__ __attribute__((aligned(1024))) char smem[G::SMEM];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // wave-uniform, in an SGPR
  const int wm = wave / WN, wn = wave % WN;
  int tm, tn;
  int split = 0, twg = blockIdx.x, nwg = gridDim.x;
  if (p.splits > 1) {
    split = blockIdx.x % p.splits;
    twg = blockIdx.x / p.splits;
    nwg = gridDim.x / p.splits;
  }
  tile_of(twg, nwg, p, tm, tn);
  const int m0 = tm * BM, n0 = tn * BN;
  // Folded LayerNorm: the partial statistics of row m0 + tid are loaded
  // into registers here, so that the loads overlap the main loop; they are
  // merged after it. (Issued after the first slices instead, as the
  // residual below is, they made the encoder 1% slower: a slice wait that
  // does not count them holds until these loads return.)
  constexpr bool LN_ROWS = EPI == kEpiLnIn || EPI == kEpiLnInGelu || EPI == kEpiQkvAttn;
  static_assert(BM <= 64 * WM * WN, "one thread per tile row");
  // Stands in for an absent operand (no statistics, no bias, no lengths) in
  // the unconditional loads below; their values then go unused.
  const void *any = APK ? p.a_pk : p.A;
  float2 ln_pr[LN_ROWS ? kLnMaxParts : 1];
  if constexpr (LN_ROWS) {
    const bool mine = p.ln_part && (int)threadIdx.x < BM && m0 + (int)threadIdx.x < p.M;
    const float2 *src = (const float2 *)p.ln_part + (int64_t)(m0 + threadIdx.x) * p.ln_nparts;
#pragma unroll
    for (int q = 0; q < kLnMaxParts; ++q)
      ln_pr[q] = mine && q < p.ln_nparts ? src[q] : make_float2(0.f, 0.f);
  }
  // The epilogue's per-column constants of this lane's TN columns: bias,
  // dequantisation scale, or the folded LayerNorm's column sums and offsets
  // (col_s: scale, col_c: offset). Loaded here with the row statistics, so
  // that their latency passes under the main loop instead of after the last
  // MFMA.
  constexpr bool LN_COLS = EPI == kEpiLnIn || EPI == kEpiLnInGelu;
  typedef typename std::conditional<std::is_same<OutT, int8_t>::value, f16, OutT>::type BiasT;
  // The raw values are loaded here, unconditionally (column 0 for columns
  // past N), and col_s / col_c formed from them after the main loop: a load
  // under a per-lane condition whose value is converted at once made the
  // wavefront wait for it before requesting its first slice (three to six
  // dependent loads in a row in the bias and dequantisation epilogues:
  // int8 FFN-down + statistics 19.0 -> 18.6 us, encoders 0.8-1.7% faster).
  BiasT col_bias[TN];
  float col_x[TN], col_y[TN];
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    const int col = n0 + wn * WTN + j * MS + lane % MS, cc = col < p.N ? col : 0;
    if constexpr (EPI == kEpiQkvAttn) {  // N is a whole number of 192-column tiles
      const bool ln = p.ln_part != nullptr, bias = p.bias != nullptr;
      col_x[j] = (ln ? p.ln_s : (const float *)any)[ln ? cc : 0];
      col_y[j] = (ln ? p.ln_c : (const float *)any)[ln ? cc : 0];
      col_bias[j] = (bias ? (const BiasT *)p.bias : (const BiasT *)any)[bias ? cc : 0];
    } else {
      if constexpr (EPI != ZK_EPI_NONE && !LN_COLS) col_bias[j] = ((const BiasT *)p.bias)[cc];
      if constexpr (DEQ) col_x[j] = p.s_w[cc];
      if constexpr (LN_COLS) {
        col_x[j] = p.ln_s[cc];
        col_y[j] = p.ln_c[cc];
      }
    }
  }
  float col_s[TN], col_c[TN];
  auto form_cols = [&]() {
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int col = n0 + wn * WTN + j * MS + lane % MS;
      col_s[j] = 1.f;
      col_c[j] = 0.f;
      if constexpr (EPI == kEpiQkvAttn) {
        const bool ln = p.ln_part != nullptr;
        col_s[j] = ln ? col_x[j] : 0.f;
        col_c[j] = ln ? col_y[j] : to_f(col_bias[j]);
      } else if (col < p.N) {
        if constexpr (EPI != ZK_EPI_NONE && !LN_COLS) col_c[j] = to_f(col_bias[j]);
        if constexpr (DEQ) col_s[j] = p.s_x * col_x[j];
        if constexpr (LN_COLS) {
          col_s[j] = col_x[j];
          col_c[j] = col_y[j];
        }
      }
    }
  };
  // kEpiResStats: the residual rows of the wave's first stripe (and their
  // LayerNorm statistics) are loaded into registers under the main loop,
  // issued right after the first slices; those of its other stripes right
  // after the main loop, all at once, instead of one dependent load per
  // vector in the epilogue. Every lane loads (out-of-range lanes from the
  // first element), so a stripe is exactly 2 NPV vector loads.
  constexpr int NPV0 = (MS * (WTN / 8) + 63) / 64;
  constexpr bool RES_PREF = EPI == kEpiResStats && std::is_same<OutT, f16>::value && NPV0 <= 6;
  constexpr int NPV = RES_PREF ? NPV0 : 1, NPT = RES_PREF ? G::TM : 1;
  f16x8 res_pv[NPT][NPV];
  float2 res_ms[NPT][NPV];
  auto load_res = [&](int i) {
    const f16 *rb = (const f16 *)p.res;
    const float2 *lb = p.res_ln ? (const float2 *)p.res_ln : (const float2 *)p.res;
#pragma unroll
    for (int k = 0; k < NPV; ++k) {
      const int v = lane + 64 * k, rl = v / (WTN / 8), cl = (v % (WTN / 8)) * 8;
      const int row = m0 + wm * WTM + i * MS + rl, col = n0 + wn * WTN + cl;
      const bool in = v < MS * (WTN / 8) && row < p.M && col + 8 <= p.N;
      // kept whatever `in` is (the epilogue reads only in-range vectors, and
      // res_ms only with res_ln), so that no lane's load is predicated away
      res_pv[i][k] = *(const f16x8 *)(rb + (in ? (int64_t)row * p.ldr + col : 0));
      res_ms[i][k] = lb[in && p.res_ln ? row : 0];
    }
  };
  // With res_ln, the residual LayerNorm's gamma and beta at this lane's
  // vector columns (the same for every stripe of the wave), all loaded
  // before any epilogue store (a load issued after a store could only be
  // waited for together with that store). The fp16 4-wave tiles (one wave
  // per SIMD, registers to spare) load them here, at kernel start, so that
  // their latency passes under the main loop; the others after it.
  constexpr bool EARLY_GB = RES_PREF && WM * WN == 4 && std::is_same<OP, F16Op>::value;
  f16x8 res_g[NPV], res_b[NPV];
  auto load_gb = [&]() {
#pragma unroll
    for (int k = 0; k < NPV; ++k) {
      const int col = n0 + wn * WTN + ((lane + 64 * k) % (WTN / 8)) * 8;
      const int64_t c = col + 8 <= p.N ? col : 0;
      res_g[k] = *(const f16x8 *)((const f16 *)p.res_gamma + c);
      res_b[k] = *(const f16x8 *)((const f16 *)p.res_beta + c);
    }
  };
  if constexpr (EARLY_GB) {
    if (p.res_ln) load_gb();
  }
  // The fused attention's sequence length for this wave's queries, loaded
  // at kernel start for the same reason.
  int attn_len = 0;
  if constexpr (EPI == kEpiQkvAttn) {
    const int b = m0 / p.seq + wave * 32 / p.seq;
    const bool vl = p.valid_lens != nullptr;
    attn_len = (vl ? p.valid_lens : (const int32_t *)any)[vl && b < p.batch ? b : 0];
  }
  const int kbytes = p.K * OP::kElem;
  const int64_t lda_b = p.lda * OP::kElem, ldb_b = p.ldb * OP::kElem;
  const int a_rows = min(BM, p.M - m0), b_rows = min(BN, p.N - n0);
  // APK: the tile's row blocks of the fragment-ordered A, one 1 KB fragment
  // per 32 bytes of a row (kbytes / 32 KB each)
  const int a_blocks = min(BM / 32, (p.M + 31) / 32 - m0 / 32);
  const __amdgpu_buffer_rsrc_t rA = __builtin_amdgcn_make_buffer_rsrc(
      APK ? (void *)((const char *)p.a_pk + (int64_t)(m0 / 32) * (kbytes / 32) * 1024)
          : (void *)((const char *)p.A + (int64_t)m0 * lda_b),
      (short)0, APK ? a_blocks * (kbytes / 32) * 1024 : (int)((a_rows - 1) * lda_b + kbytes),
      0x00020000);
  // BNK: B is [K,N], its descriptor ends with the 16-byte vector that holds the
  // last row's last column (inside the row's pitch, a multiple of 8): a 4-byte
  // word that straddles the end reads as zero, which for odd N would drop
  // that column's last product. Rows past K read as zero; columns past N read
  // what follows and are not stored.
  const __amdgpu_buffer_rsrc_t rB = __builtin_amdgcn_make_buffer_rsrc(
      (void *)((const char *)p.B + (BNK ? (int64_t)n0 * 2 : (int64_t)n0 * ldb_b)), (short)0,
      BNK ? (int)((p.K - 1) * ldb_b + (int64_t)(((p.N + 7) & ~7) - n0) * 2)
          : (int)((b_rows - 1) * ldb_b + kbytes),
      0x00020000);

  // DMA source offsets. Instruction g of this wave fills tile rows
  // [(wave * I + g) * RPI, +RPI); lane l lands at LDS slot l % CH of row
  // (l / CH) of that group and therefore fetches the logical chunk whose
  // swizzled slot that is.
  // APK: instruction g moves fragment f = wave * IA + g of the slice (row
  // block f / KS, k-step f % KS), 1 KB contiguous, to LDS byte f * 1024 of
  // the stage's A part, where lane l reads its 16 bytes of it back.
  int offA[IA], chA[IA], offB[IB], chB[IB];
#pragma unroll
  for (int g = 0; g < IA; ++g) {
    if constexpr (APK) {
      const int f = wave * IA + g;
      chA[g] = 0;
      offA[g] = ((f / KS) * (kbytes / 32) + f % KS) * 1024 + lane * 16;
    } else {
      const int row = (wave * IA + g) * G::RPI + lane / CH;
      const int c = lds_slot<BKB>(row, lane % CH);  // the swizzle is an involution
      chA[g] = c * 16;
      offA[g] = (int)(row * lda_b) + c * 16;
    }
  }
#pragma unroll
  for (int g = 0; g < IB; ++g) {
    if constexpr (BNK) {
      // the slice's rows of B, BN columns each, one after another
      const int at = (wave * IB + g) * 64 + lane, row = at / (BN / 8);
      chB[g] = 0;
      offB[g] = (int)(row * ldb_b) + ((at % (BN / 8)) ^ bnk_swz<BN>(row)) * 16;
    } else {
      const int row = (wave * IB + g) * G::RPI + lane / CH;
      const int c = lds_slot<BKB>(row, lane % CH);
      chB[g] = c * 16;
      offB[g] = (int)(row * ldb_b) + c * 16;
    }
  }
  // BNK: bytes of B per slice (BKB / 2 rows)
  const int slice_b = BNK ? (int)(BKB / 2 * ldb_b) : 0;
  typename MM::Acc acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < R; ++r) acc[i][j][r] = 0;

  // Fragment row of this lane inside an MS-row block, and the chunk offset
  // of its half / quarter of the k-step.
  const int frow = lane % MS, fch = lane / MS;
  // Fragments of two consecutive k-steps: k-step ks of every slice uses
  // buffer ks & 1 (KS is even), so the first k-step of the next slice can
  // be read while the last one of this slice is multiplied.
  Frag fa[2][TM], fb[2][TN];
  static_assert(!APK || (MS == 32 && !std::is_same<OP, F32Op>::value), "fragment-ordered A");
  constexpr int PER = IA + IB;  // DMA instructions per slice and wave
  auto rd = [&](int stage, int ks, int buf) {
    const char *As = smem + stage * G::STAGE;
    const char *Bs = As + BM * BKB;
    const int c = ks * KCH + fch;
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      if constexpr (APK) {
        fa[buf][i] = *(const Frag *)(As + (((wm * WTM + i * MS) / 32) * KS + ks) * 1024 + lane * 16);
      } else {
        const int row = wm * WTM + i * MS + frow;
        fa[buf][i] = *(const Frag *)(As + row * BKB + lds_slot<BKB>(row, c) * 16);
      }
    }
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      if constexpr (BNK) {
        fb[buf][j] = read_bnk<BN, MS>((const f16 *)Bs, ks, wn * WTN + j * MS, lane);
      } else {
        const int row = wn * WTN + j * MS + frow;
        fb[buf][j] = *(const Frag *)(Bs + row * BKB + lds_slot<BKB>(row, c) * 16);
      }
    }
  };
  auto mma_step = [&](int buf) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) acc[i][j] = MM::mma(fa[buf][i], fb[buf][j], acc[i][j]);
  };

  const int nk_all = (kbytes + BKB - 1) / BKB;
  const int kt0 = p.splits > 1 ? split * p.nk_per : 0;  // first slice of this split
  const int nk = p.splits > 1 ? max(0, min(nk_all - kt0, p.nk_per)) : nk_all;
  // One K slice of A and W: IA + IB wavefront instructions, each moving
  // 1 KB (64 lanes x 16 bytes) into consecutive LDS bytes. The host
  // compilation pass sees an empty statement: its semantic check of this
  // builtin with a run-time offset rejects the kernel, and clang would then
  // silently omit the kernel's launch stub.
#if defined(__HIP_DEVICE_COMPILE__)
#define ZK_ISSUE(kt, stage)                                                                   \
  do {                                                                                        \
    const int kb_ = ((kt) + kt0) * BKB;                                                       \
    char *as_ = smem + (stage) * G::STAGE, *bs_ = as_ + BM * BKB;                             \
    _Pragma("unroll") for (int g = 0; g < IA; ++g)                                            \
        __builtin_amdgcn_raw_ptr_buffer_load_lds(                                             \
            rA, ZK_LDS(as_ + (wave * IA + g) * 1024), 16,                                     \
            kb_ + chA[g] < kbytes ? offA[g] + (APK ? kb_ / BKB * KS * 1024 : kb_)            \
                                  : 0x7ffffff0,                                               \
            0, 0, 0);                                                                         \
    _Pragma("unroll") for (int g = 0; g < IB; ++g)                                            \
        __builtin_amdgcn_raw_ptr_buffer_load_lds(                                             \
            rB, ZK_LDS(bs_ + (wave * IB + g) * 1024), 16,                                     \
            BNK                       ? offB[g] + ((kt) + kt0) * slice_b                      \
            : kb_ + chB[g] < kbytes ? offB[g] + kb_                                           \
                                      : 0x7ffffff0,                                           \
            0, 0, 0);                                                                         \
  } while (0)
#else
#define ZK_ISSUE(kt, stage) ((void)(kt), (void)(stage))
#endif
  // res_first: the first stripe's residual rows are requested before the
  // first slice. Loads into registers and DMA loads into LDS complete in
  // order only among their own kind, so a slice wait (at most c loads in
  // flight) guarantees a slice only through the c DMA loads issued after
  // it, and holds for any load into registers still in flight. Issued after
  // the first slices, these loads made the first waits hold until they
  // returned (fp16 encoder 1.6% slower); allowed for as younger loads in
  // those waits, they could have let a wave read a slice before it landed
  // (as loads of A into registers beside the W DMA were seen to do).
  if constexpr (RES_PREF) {
    load_res(0);
    asm volatile("" ::: "memory");
  }
  {
    // Prologue: one slice per stage.
#pragma unroll
    for (int s = 0; s < ST; ++s)
      if (s < nk) ZK_ISSUE(s, s);
    // (the residual rows, loaded into registers before the prologue, are
    // not counted by the slice waits: see res_first)
    wait_slices<ST - 1, PER>(nk - 1);
    lds_barrier();
    rd(0, 0, 0);
    // Main loop over slices. Before the last k-step of slice kt every wave
    // waits for slice kt + 1 and meets at the barrier; by then the ring stage
    // of slice kt has been read completely (its last fragments are in
    // registers), so slice kt + ST is issued into it, and the first
    // fragments of slice kt + 1 are read under the last MFMAs of slice kt.
    auto steps_but_last = [&](int stage) {
#pragma unroll
      for (int ks = 0; ks + 1 < KS; ++ks) {
        rd(stage, ks + 1, (ks + 1) & 1);
        mma_step(ks & 1);
        interleave<NRD, TM * TN>();
      }
    };
    int stage = 0;
    for (int kt = 0; kt + 1 < nk; ++kt) {
      steps_but_last(stage);
      const int next = stage + 1 == ST ? 0 : stage + 1;
      wait_slices<ST - 2, PER>(nk - 2 - kt);
      lds_barrier();
      if (kt + ST < nk) ZK_ISSUE(kt + ST, stage);
      rd(next, 0, 0);
      mma_step(1);
      interleave<NRD, TM * TN>();
      stage = next;
    }
    steps_but_last(stage);  // last slice: nothing left to prefetch
    mma_step(1);
  }
#undef ZK_ISSUE
  if constexpr (RES_PREF) {
#pragma unroll
    for (int i = 1; i < NPT; ++i) load_res(i);
    if (!EARLY_GB && p.res_ln) load_gb();
  }
  __syncthreads();  // every wave is done reading the ring; it becomes epilogue space
  form_cols();
  if constexpr (EPI == kEpiQkvAttn) {
    // The tile is the Q, K and V columns of head tn (weights interleaved
    // per head: q, k, v, 64 rows each) for the 256 rows of the sequences
    // the tile holds. They go into LDS as fp16 with their bias, [part][row]
    // [64] with the K/V tile swizzle, and the tile's attention runs from
    // there: Q, K and V never reach HBM.
    static_assert(std::is_same<OP, F16Op>::value && BM == 256 && BN == 192 && MS == 32 &&
                      WM == 4 && WN == 2, "fused QKV attention tile");
    constexpr int HD = 64;
    f16 *qkv = (f16 *)smem;  // 3 x 256 x 64 halves = 96 KB, inside the ring
    const int h32 = lane >> 5;
    // With ln_part the rows of X are the LayerNorm input: Q, K, V are
    // rstd (acc - mean s) + c (see GemmParams), (mean, rstd) per row in LDS.
    float2 *lnt = (float2 *)(smem + 3 * BM * HD * 2);
    static_assert(3 * BM * HD * 2 + BM * 8 <= G::SMEM, "LN table does not fit");
    const bool ln = p.ln_part != nullptr;
    if (ln) {
      if ((int)threadIdx.x < BM) {
        const float2 ms = ln_merge(ln_pr, p.ln_nparts, p.ln_eps);
        lnt[threadIdx.x] = ms;
        if (p.ln_out && tn == 0 && m0 + (int)threadIdx.x < p.M)
          ((float2 *)p.ln_out)[m0 + threadIdx.x] = ms;
      }
      __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      float2 ms[16];
#pragma unroll
      for (int r = 0; r < 16; ++r)
        ms[r] = ln ? lnt[wm * WTM + i * 32 + 8 * (r >> 2) + 4 * h32 + (r & 3)]
                   : make_float2(0.f, 1.f);
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const int cb = wn * WTN + j * 32;  // first tile column of the block
        const int d = cb % HD + (lane & 31), n = n0 + cb + (lane & 31);
        const float sv = col_s[j], cv = col_c[j];  // column n's constants
        f16 *dst = qkv + (cb / HD) * (BM * HD);
        // one formula for both cases (no per-element select): without ln,
        // (mean, rstd) = (0, 1) and sv = 0 make it fma(1, fma(-0, 0, acc), c),
        // i.e. acc + c. The outer fma and the fp16 conversion compile to one
        // v_fma_mixlo_f16, which rounds once, to fp16.
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int row = wm * WTM + i * 32 + 8 * (r >> 2) + 4 * h32 + (r & 3);
          const float v = fmaf(ms[r].y, fmaf(-ms[r].x, sv, acc[i][j][r]), cv);
          dst[row * HD + (((d >> 3) ^ kv_swz(row)) << 3) + (d & 7)] = (f16)v;
        }
      }
    }
    __syncthreads();
    // Wave w owns the 32 queries of tile rows [32 w, 32 w + 32); their
    // sequence's keys are tile rows [sq * seq, +seq).
    const int qr = wave * 32 + (lane & 31);
    const int sq = wave * 32 / p.seq;
    const int b = m0 / p.seq + sq;
    if (b < p.batch) {
      // opaque until here, so that the select below is not formed (and
      // waited for) right after the load at kernel start
      asm volatile("" : "+v"(attn_len));
      int L = p.valid_lens ? attn_len : p.seq;
      L = L < 0 ? 0 : (L > p.seq ? p.seq : L);
      f16x8 qf[HD / 16];
#pragma unroll
      for (int c = 0; c < HD / 16; ++c)
        qf[c] = *(const f16x8 *)(qkv + qr * HD + (((2 * c + h32) ^ kv_swz(qr)) << 3));
      const f16 *Kt = qkv + BM * HD + sq * p.seq * HD, *Vt = Kt + BM * HD;
      f32x16 o[HD / 32];
#pragma unroll
      for (int dt = 0; dt < HD / 32; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[dt][r] = 0.f;
      float m = -__builtin_inff(), l = 0.f;
      // At most two 64-key tiles (sequences of 64 or 128 tokens), both in
      // LDS: the second tile's Q.K^T is issued before the first tile's
      // softmax, so that its MFMAs can run under that VALU work (the same
      // arithmetic per tile as attn32_tile, in the same order).
      const int ntiles = (L + 63) / 64;
      if (ntiles > 0) {
        // Both tiles are processed whatever the length (a wave-uniform branch
        // would let the compiler hoist the exponentials above it and lose the
        // interleaving): with 64-token sequences tile 1 is tile 0 again, and
        // wherever L <= 64 every key of tile 1 lies at or past L, so its
        // probabilities are 0 and m, l and o stay exactly as they were.
        const int off1 = p.seq > 64 ? 64 * HD : 0;
        f32x16 s0[2], s1[2];
        f16x8 pf0[2][2], pf1[2][2];
        attn32_qk<HD, true, HD>(Kt, qf, lane, s0);
        const float mneg = attn32_softmax_max<HD, false>(s0, 0, L, p.scale_log2, NoMask{},
                                                         false, lane, o, m, l);
        // tile 1's 8 K-fragment reads and 8 MFMAs among tile 0's exponentials
        attn32_qk<HD, true, HD>(Kt + off1, qf, lane, s1);
        attn32_softmax_exp<HD>(s0, p.scale_log2, mneg, l, pf0);
        __builtin_amdgcn_sched_group_barrier(0x100, 8, 0);  // DS reads
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // MFMA
          __builtin_amdgcn_sched_group_barrier(0x402, 8, 0);  // VALU incl. exp
        }
        // tile 0's P.V (16 transposing reads, 8 MFMAs) among tile 1's
        // exponentials; tile 1's rescale of o, if any, after it
        float alpha;
        bool resc;
        const float mneg1 = attn32_max_defer(s1, 1, L, p.scale_log2, lane, m, l, alpha, resc);
        attn32_softmax_exp<HD>(s1, p.scale_log2, mneg1, l, pf1);
        attn32_pv<HD, true, HD>(Vt, pf0, lane, o);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);  // DS reads
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // MFMA
          __builtin_amdgcn_sched_group_barrier(0x402, 8, 0);  // VALU incl. exp
        }
        if (resc) {
#pragma unroll
          for (int dt = 0; dt < HD / 32; ++dt)
#pragma unroll
            for (int r = 0; r < 16; ++r) o[dt][r] *= alpha;
        }
        attn32_pv<HD, true, HD>(Vt + off1, pf1, lane, o);
      }
      const int grow = m0 + qr;
      const float inv = l > 0.f ? 1.0f / l : 0.f;
      // (f16)as_f32(o inv) in both layouts: the product rounded to fp32, then
      // to fp16, so that no build fuses it into one rounding in one of them
      if (p.c_pk) {
        // ctx in fragment order (the out-projection's A): the wave's 32 rows
        // are one row block, head tn's 64 columns four 1 KB k-steps. Lane l
        // holds columns 8 g + 4 (l / 32) .. +3 of each 32-column group; one
        // v_permlane32_swap per register pair hands each half of the wave
        // the other half's 4 columns, so that lane l holds columns
        // 8 (l / 32) .. +7 of a k-step (16 bytes, one store per k-step).
        char *F = (char *)p.C + ((int64_t)((m0 + wave * 32) / 32) * (p.ldc / 16) + tn * (HD / 16)) * 1024 +
                  lane * 16;
#pragma unroll
        for (int dt = 0; dt < HD / 32; ++dt)
#pragma unroll
          for (int kh = 0; kh < 2; ++kh) {
            u32x2 a, b;  // columns 16 kh + 4 (l / 32) and 16 kh + 8 + 4 (l / 32), 4 each
#pragma unroll
            for (int e = 0; e < 2; ++e) {
              const f16 a0 = (f16)as_f32(o[dt][8 * kh + 2 * e] * inv);
              const f16 a1 = (f16)as_f32(o[dt][8 * kh + 2 * e + 1] * inv);
              const f16 b0 = (f16)as_f32(o[dt][8 * kh + 4 + 2 * e] * inv);
              const f16 b1 = (f16)as_f32(o[dt][8 * kh + 4 + 2 * e + 1] * inv);
              a[e] = (unsigned)__builtin_bit_cast(unsigned short, a0) |
                     ((unsigned)__builtin_bit_cast(unsigned short, a1) << 16);
              b[e] = (unsigned)__builtin_bit_cast(unsigned short, b0) |
                     ((unsigned)__builtin_bit_cast(unsigned short, b1) << 16);
            }
            // upper lanes' a <-> lower lanes' b: the lower half then holds
            // columns 0-7 of the k-step in (a, b), the upper half 8-15
            u32x4 v;
#pragma unroll
            for (int e = 0; e < 2; ++e) {
              const auto sw = __builtin_amdgcn_permlane32_swap(a[e], b[e], false, false);
              v[e] = sw[0];
              v[e + 2] = sw[1];
            }
            if (grow < p.M) store_nt((u32x4 *)(F + (dt * 2 + kh) * 1024), v);
          }
      } else if (grow < p.M) {
        f16 *O = (f16 *)p.C + (int64_t)grow * p.ldc + tn * HD;
#pragma unroll
        for (int dt = 0; dt < HD / 32; ++dt)
#pragma unroll
          for (int g = 0; g < 4; ++g) {
            f16x4 out;
#pragma unroll
            for (int e = 0; e < 4; ++e) out[e] = (f16)as_f32(o[dt][4 * g + e] * inv);
            *(f16x4 *)(O + dt * 32 + 8 * g + 4 * h32) = out;
          }
      }
    }
  } else {
    // Epilogue: per wave, one MS-row stripe at a time.
    constexpr bool RES_STATS = EPI == kEpiResStats;
    constexpr bool LN_IN = EPI == kEpiLnIn || EPI == kEpiLnInGelu;
    constexpr bool RESID = EPI == ZK_EPI_BIAS_RESIDUAL || RES_STATS;
    float *ws = (float *)smem + wave * MS * G::EPITCH;
    // LN_IN: (mean, rstd) of the tile's rows, in LDS beyond the stripes
    float2 *lnt = (float2 *)(smem + G::EPI_BYTES);
    if constexpr (LN_IN) {
      static_assert(G::EPI_BYTES + BM * 8 <= G::SMEM, "LN table does not fit");
      if ((int)threadIdx.x < BM) {
        const float2 ms = ln_merge(ln_pr, p.ln_nparts, p.ln_eps);
        lnt[threadIdx.x] = ms;
        if (p.ln_out && tn == 0 && m0 + (int)threadIdx.x < p.M)
          ((float2 *)p.ln_out)[m0 + threadIdx.x] = ms;
      }
      __syncthreads();
    }
    // int8 output (re-quantisation): bias and residual are fp16; the value is
    // rounded to fp16 first, so the result equals quantising the fp16 output.
    constexpr bool Q8 = std::is_same<OutT, int8_t>::value;
    OutT *C = (OutT *)p.C + (p.splits > 1 ? split * p.split_stride : 0);
    const BiasT *res = (const BiasT *)p.res;
    const float inv_q = Q8 ? 1.0f / p.s_q : 1.0f;
    const bool vec_ok = (p.ldc % 8 == 0) && (Q8 ? aligned8(p.C) : aligned16(p.C)) &&
                        (!RESID || ((p.ldr % 8 == 0) && aligned16(p.res)));
    // this lane's column constants, loaded at kernel start: bias (or LN_IN's
    // offset c) and scale (DEQ's s_x s_w, LN_IN's column sum s)
    const float *bj = col_c, *sj = col_s;
    // the residual's value at (row, col) (RES_STATS with res_ln: its LayerNorm)
    auto resid = [&](int row, int col, float r) {
      if constexpr (RES_STATS) {
        if (p.res_ln) {
          const float2 ms = ((const float2 *)p.res_ln)[row];
          return fmaf((r - ms.x) * ms.y, to_f(((const f16 *)p.res_gamma)[col]),
                      to_f(((const f16 *)p.res_beta)[col]));
        }
      }
      return r;
    };
    constexpr int VPR = WTN / 8;  // 8-column vectors per stripe row
    // fragment-ordered output (p.c_pk): the folded-LayerNorm GELU epilogue of
    // the fp16 32x32 tiles and the re-quantising int8 ones (FFN-up, whose
    // output is FFN-down's A)
    constexpr bool CPK = MS == 32 && ((EPI == kEpiLnInGelu && std::is_same<OutT, f16>::value &&
                                       WTN % 16 == 0) ||
                                      (Q8 && WTN % 32 == 0));
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      // LN_IN: (mean, rstd) of the rows this lane's registers hold
      float2 msr[LN_IN ? R : 1];
      if constexpr (LN_IN) {
#pragma unroll
        for (int r = 0; r < R; ++r)
          msr[r] = lnt[wm * WTM + i * MS + (MS == 32 ? 8 * (r >> 2) + 4 * fch + (r & 3) : 4 * fch + r)];
      }
#pragma unroll
      for (int j = 0; j < TN; ++j) {
#pragma unroll
        for (int r = 0; r < R; ++r) {
          const int rl = MS == 32 ? 8 * (r >> 2) + 4 * fch + (r & 3) : 4 * fch + r;
          float *dst = ws + rl * G::EPITCH + j * MS + frow;
          if constexpr (std::is_same<OutT, int32_t>::value) {
            *(int *)dst = acc[i][j][r];
          } else if constexpr (LN_IN) {
            // rstd (acc - mean s) + c, then the activation
            const float t = fmaf(msr[r].y, fmaf(-msr[r].x, sj[j], (float)acc[i][j][r]), bj[j]);
            *dst = EPI == kEpiLnInGelu ? gelu_erf_fast(t) : t;
          } else {
            const float v = DEQ ? (float)acc[i][j][r] * sj[j] : (float)acc[i][j][r];
            *dst = epilogue<RES_STATS ? (int)ZK_EPI_BIAS : EPI>(v, bj[j]);
          }
        }
      }
      const int row0 = m0 + wm * WTM + i * MS, col0 = n0 + wn * WTN;
      auto store_vec = [&](int v, int k) {
        const int rl = v / VPR, cl = (v % VPR) * 8;
        const int row = row0 + rl, col = col0 + cl;
        if (row >= p.M || col >= p.N) return;
        float *src = ws + rl * G::EPITCH + cl;
        OutT *dst = C + (int64_t)row * p.ldc + col;
        if (vec_ok && col + 8 <= p.N) {
          const f32x4 lo = *(const f32x4 *)src, hi = *(const f32x4 *)(src + 4);
          if constexpr (std::is_same<OutT, int32_t>::value) {
            *(f32x4 *)dst = lo;  // raw bits of the int32 accumulators
            *(f32x4 *)(dst + 4) = hi;
          } else {
            float o[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
            if constexpr (RESID) {
              const BiasT *rp = res + (int64_t)row * p.ldr + col;
              if constexpr (std::is_same<BiasT, f16>::value) {
                const f16x8 rv = RES_PREF ? res_pv[RES_PREF ? i : 0][k] : *(const f16x8 *)rp;
                if (RES_STATS && p.res_ln) {
                  // LN(res): one (mean, rstd) per row, gamma / beta as vectors
                  const float2 ms = RES_PREF ? res_ms[RES_PREF ? i : 0][k]
                                             : ((const float2 *)p.res_ln)[row];
                  const f16x8 g = RES_PREF ? res_g[k] : *(const f16x8 *)((const f16 *)p.res_gamma + col);
                  const f16x8 bb = RES_PREF ? res_b[k] : *(const f16x8 *)((const f16 *)p.res_beta + col);
#pragma unroll
                  for (int e = 0; e < 8; ++e)
                    o[e] += fmaf(((float)rv[e] - ms.x) * ms.y, (float)g[e], (float)bb[e]);
                } else {
#pragma unroll
                  for (int e = 0; e < 8; ++e) o[e] += (float)rv[e];
                }
              } else {
#pragma unroll
                for (int e = 0; e < 8; ++e) o[e] += resid(row, col + e, to_f(rp[e]));
              }
            }
            if constexpr (std::is_same<OutT, f16>::value) {
              f16x8 h;
#pragma unroll
              for (int e = 0; e < 8; ++e) h[e] = (f16)o[e];
              store_nt((f16x8 *)dst, h);
              if constexpr (RES_STATS) {  // the stored values, for the statistics
                *(f32x4 *)src = f32x4{(float)h[0], (float)h[1], (float)h[2], (float)h[3]};
                *(f32x4 *)(src + 4) = f32x4{(float)h[4], (float)h[5], (float)h[6], (float)h[7]};
              }
            } else if constexpr (Q8) {
              float of[8];  // rounded to fp16 first: the fp16 output's quantisation
#pragma unroll
              for (int e = 0; e < 8; ++e) of[e] = (float)(f16)o[e];
              store_nt((u32x2 *)dst, quant8(of, p.s_q, inv_q));
            } else {
              *(f32x4 *)dst = f32x4{o[0], o[1], o[2], o[3]};
              *(f32x4 *)(dst + 4) = f32x4{o[4], o[5], o[6], o[7]};
            }
          }
        } else {
          for (int e = 0; e < 8 && col + e < p.N; ++e) {
            if constexpr (std::is_same<OutT, int32_t>::value) {
              dst[e] = ((const int *)src)[e];
            } else {
              float o = src[e];
              if (RESID) o += resid(row, col + e, to_f(res[(int64_t)row * p.ldr + col + e]));
              if constexpr (Q8) dst[e] = quant1((float)(f16)o, p.s_q, inv_q);
              else dst[e] = (OutT)o;
              if constexpr (RES_STATS) src[e] = (float)(OutT)o;
            }
          }
        }
      };
      if constexpr (CPK) {
        if (p.c_pk) {
          // C in fragment order: the stripe (32 rows, a whole row block) is a
          // run of the consumer's 1 KB A fragments of KC columns (16 fp16 or
          // 32 int8); lane l stores row l % 32, columns KE (l / 32) .. +KE-1
          // of its fragment: 16 bytes
          constexpr int KC = Q8 ? 32 : 16, KE = KC / 2;
          const int rl = lane & 31;
          const int64_t blk = (int64_t)(row0 / 32) * (p.N / KC) + col0 / KC;
#pragma unroll
          for (int kc = 0; kc < WTN / KC; ++kc) {
            const int cl = kc * KC + (lane >> 5) * KE;
            if (row0 + rl < p.M && col0 + cl < p.N) {
              const float *src = ws + rl * G::EPITCH + cl;
              char *dst = (char *)p.C + ((blk + kc) * 64 + lane) * 16;
              if constexpr (Q8) {
                // rounded to fp16 first, as the row-major stores do
                float of[2][8];
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                  const f32x4 lo = *(const f32x4 *)(src + 8 * h), hi = *(const f32x4 *)(src + 8 * h + 4);
#pragma unroll
                  for (int e = 0; e < 4; ++e) {
                    of[h][e] = (float)(f16)lo[e];
                    of[h][e + 4] = (float)(f16)hi[e];
                  }
                }
                const u32x2 q0 = quant8(of[0], p.s_q, inv_q), q1 = quant8(of[1], p.s_q, inv_q);
                store_nt((u32x4 *)dst, u32x4{q0[0], q0[1], q1[0], q1[1]});
              } else {
                const f32x4 lo = *(const f32x4 *)src, hi = *(const f32x4 *)(src + 4);
                f16x8 h;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                  h[e] = (f16)lo[e];
                  h[e + 4] = (f16)hi[e];
                }
                store_nt((f16x8 *)dst, h);
              }
            }
          }
          continue;
        }
      }
      if constexpr (RES_PREF) {
#pragma unroll
        for (int k = 0; k < NPV; ++k)
          if (lane + 64 * k < MS * VPR) store_vec(lane + 64 * k, k);
      } else {
        for (int v = lane; v < MS * VPR; v += 64) store_vec(v, 0);
      }
      if constexpr (RES_STATS) {
        // (mean, M2) of every kLnSeg-column segment of the stripe's rows,
        // from the stored (rounded) values. Two neighbouring lanes per (row,
        // segment), each over half of it; the halves are merged by Chan's
        // rule: M2 = M2a + M2b + (mean_a - mean_b)^2 * n / 4.
        static_assert(WTN % kLnSeg == 0 && kLnSeg % 8 == 0, "statistics segments");
        constexpr int SEG = WTN / kLnSeg, HALF = kLnSeg / 2;
        for (int v = lane; v < 2 * MS * SEG; v += 64) {  // 2 MS SEG is even: pairs stay together
          const int pr = v >> 1, hf = v & 1;
          const int rl = pr / SEG, sg = pr % SEG;
          const int row = row0 + rl;
          const bool ok = row < p.M && col0 + kLnSeg * sg < p.N;
          float mean = 0.f, m2 = 0.f;
          if (ok) {
            const f32x4 *x4 = (const f32x4 *)(ws + rl * G::EPITCH + kLnSeg * sg + HALF * hf);
            float sum = 0.f;
#pragma unroll
            for (int q = 0; q < HALF / 4; ++q) {
              const f32x4 t = x4[q];
              sum += (t[0] + t[1]) + (t[2] + t[3]);
            }
            mean = sum * (1.0f / HALF);
#pragma unroll
            for (int q = 0; q < HALF / 4; ++q) {
              const f32x4 t = x4[q];
#pragma unroll
              for (int e = 0; e < 4; ++e) {
                const float d = t[e] - mean;
                m2 = fmaf(d, d, m2);
              }
            }
          }
          const float mo = lane_xor1(mean), m2o = lane_xor1(m2);
          if (ok && hf == 0) {
            const float d = mo - mean;
            ((float2 *)p.part_out)[(int64_t)row * (p.N / kLnSeg) + col0 / kLnSeg + sg] =
                make_float2(0.5f * (mean + mo), m2 + m2o + d * d * (0.25f * kLnSeg));
          }
        }
      }
    }
  }
}

}  // namespace zk
