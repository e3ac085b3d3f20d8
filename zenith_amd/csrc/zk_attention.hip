// Flash-attention forward (non-causal, optional key-padding mask).
//
// fp16 path (MFMA). A workgroup of NW wavefronts owns NW*32 query rows of
// one (batch, head); every wavefront owns 32 of them. Keys are walked in
// tiles of 64: K and V are staged in LDS as [key][d] with 16-byte stores (or
// DMA'd there, fa_fwd_f16_ring_kernel); the V^T fragments of the P.V product
// come out of the transposing LDS read.
// The wavefront computes S^T = K . Q^T with 32x32x16 MFMAs, so each lane
// ends up holding 32 keys of ONE query column (lane % 32): the row max and
// row sum of the online softmax are then a register loop plus a single
// swap with lane ^ 32, and the per-query rescale factor is lane-uniform.
// The exponentiated scores, rounded to fp16, are already laid out as the B
// operand of O^T += V^T . P^T, so P never leaves registers. Statistics and
// accumulation are fp32; exp2 with the softmax scale folded into log2(e).
// Key tiles at or beyond the sequence's valid length are never loaded; keys
// >= valid length inside the last tile get probability exactly 0, and a
// query with no valid key produces 0 (mask rule of the reference's masked
// attention primitive).
//
// For D = 64 and at most 128 queries, fa_fwd_f16_q16_kernel below does the
// same arithmetic with 16 queries per wavefront on 16x16x32 MFMAs.
//
// fp32 path: fp32 matrix instructions, 16 queries per wavefront
// (fa_fwd_f32_kernel).
#include <type_traits>

#include "zk_attn_tile.hpp"

namespace zk {

// (query block, head, batch) of this workgroup. The gridDim.x query blocks of
// one (batch, head) read the same K and V. Workgroups go to the 8 XCDs
// round-robin by linear id, so when B*H is a multiple of 8 the blocks of one
// head are given ids 8 apart: they run on one XCD and share its L2. At b32
// s128 this cut the L2-miss reads from 31.5 MB to 18.9 MB (Q, K and V once).
struct AttnTile {
  int qb, h, b;
};
__device__ __forceinline__ AttnTile attn_tile() {
  const int64_t gx = gridDim.x, nh = gridDim.y, nbh = nh * gridDim.z;
  if (gx == 1 || nbh % 8 != 0) return {(int)blockIdx.x, (int)blockIdx.y, (int)blockIdx.z};
  const int64_t bid = blockIdx.x + gx * (blockIdx.y + nh * blockIdx.z);
  const int64_t grp = bid / (8 * gx), rem = bid % (8 * gx);
  const int64_t bh = grp * 8 + rem % 8;
  return {(int)(rem / 8), (int)(bh % nh), (int)(bh / nh)};
}

// The 16-query kernel's transposing V read gives each 16-lane group 4 rows x
// 2 chunks (group g: rows 4g .. 4g+3), and the LDS serves a 64-bit read in
// two passes, one pairing the groups (0, 2) and (1, 3). kv_swz puts rows r
// and r + 8 in the same slots, which costs each such read an extra pass.
// kv_swz16 keeps the two chunks of a row in one aligned slot pair 2h, 2h+1
// with h distinct over the even (and the odd) rows of groups {0,1}, {2,3},
// {0,2} and {1,3}, and (h, low bit) distinct over all 16 rows for the K
// fragment reads. LDS bank-conflict cycles of the b32 s128 launch: 1.97e5
// with kv_swz, 0 with kv_swz16 (the encoder's time is unchanged).
__device__ __forceinline__ int kv_swz16(int r) {
  return 2 * (((r >> 1) & 3) ^ ((r >> 2) & 2)) + ((r >> 3) & 1);
}

// PAD: the stored head_dim p.D (a multiple of 8) is below the compiled D;
// dims >= p.D of Q, K and V are read as zeros (they add nothing to Q.K^T and
// produce output columns that are not stored).
// MASK: p.mask is applied on top of the valid lengths. A tile can then be
// fully masked for a query that has seen no valid key yet (running max still
// -inf); the rescale factor and the exponent are guarded for that case.
template <int D, int NW, bool PAD = false, bool MASK = false, bool LEAN = false>
__global__ __launch_bounds__(NW * 64) void fa_fwd_f16_kernel(AttnParams p) {
  constexpr int KT = 64;
  constexpr int NT = NW * 64;
  constexpr bool SWZ = D == 64;  // swizzled unpadded rows (else padded rows)
  constexpr int KLD = SWZ ? D : D + 8;  // K and V tile row pitch (halves)
  constexpr int DV = D / 8;    // 16-byte vectors per K/V row
  constexpr int PER = KT * DV / NT;
  static_assert(KT * DV % NT == 0, "tile/thread mismatch");
  __shared__ __attribute__((aligned(16))) f16 Ks[KT * KLD];
  __shared__ __attribute__((aligned(16))) f16 Vs[KT * KLD];

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, h32 = lane >> 5;
  const AttnTile tile = attn_tile();
  const int b = tile.b, h = tile.h;
  const int L = valid_len(p, b);
  const f16 *Qb = (const f16 *)p.Q + b * p.sq[0] + h * p.sq[1];
  const f16 *Kb = (const f16 *)p.K + b * p.sk[0] + h * p.sk[1];
  const f16 *Vb = (const f16 *)p.V + b * p.sv[0] + h * p.sv[1];
  f16 *Ob = (f16 *)p.O + b * p.so[0] + h * p.so[1];

  const int qrow = tile.qb * (NW * 32) + wave * 32 + (lane & 31);
  const bool qvalid = qrow < p.Sq;
  const uint8_t *mrow = MASK ? mask_row(p, b, h, qvalid ? qrow : 0) : nullptr;
  f16x8 qf[D / 16];
#pragma unroll
  for (int c = 0; c < D / 16; ++c)
    qf[c] = qvalid && (!PAD || c * 16 + h32 * 8 < p.D)
                ? *(const f16x8 *)(Qb + qrow * p.sq[2] + c * 16 + h32 * 8)
                : f16x8{0, 0, 0, 0, 0, 0, 0, 0};

  f32x16 o[D / 32];
#pragma unroll
  for (int dt = 0; dt < D / 32; ++dt)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[dt][r] = 0.f;
  float m = -__builtin_inff(), l = 0.f;

  const int ntiles = (L + KT - 1) / KT;
  f16x8 kr[PER], vr[PER];
  auto load_kv = [&](int t) {
#pragma unroll
    for (int v = 0; v < PER; ++v) {
      const int idx = tid + v * NT;
      const int kk = t * KT + idx / DV;  // K: 16-byte vectors row-contiguous
      const bool in = kk < p.Sk && (!PAD || (idx % DV) * 8 < p.D);
      kr[v] = in ? *(const f16x8 *)(Kb + kk * p.sk[2] + (idx % DV) * 8)
                 : f16x8{0, 0, 0, 0, 0, 0, 0, 0};
      // V like K (8 lanes per 128-byte row, coalesced)
      vr[v] = in ? *(const f16x8 *)(Vb + kk * p.sv[2] + (idx % DV) * 8)
                 : f16x8{0, 0, 0, 0, 0, 0, 0, 0};
    }
  };
  auto stash_kv = [&]() {
#pragma unroll
    for (int v = 0; v < PER; ++v) {
      const int idx = tid + v * NT;
      const int row = idx / DV, ch = SWZ ? (idx % DV) ^ kv_swz(row) : idx % DV;
      *(f16x8 *)(Ks + row * KLD + ch * 8) = kr[v];
      *(f16x8 *)(Vs + row * KLD + ch * 8) = vr[v];
    }
  };

  // MASK, D <= 64: the mask bytes of a tile are requested with its K and V, one
  // tile ahead. A wavefront whose queries keep no key of the tile skips it,
  // and one whose queries keep all of them does not apply the mask (the
  // tiles of a padding or causal mask but the few on its edge). b8 h12 s384
  // 23.7 -> 17.1 us, b16 h12 s512 57 -> 35, b4 h12 s1024 54 -> 36. At D = 128
  // the registers for it cost more than it gives (b8 h12 s512 35 -> 46): the
  // bytes are read where they are used, as in LEAN (see the launch).
  // A masked key's V counts with probability 0 where its tile is walked and not
  // at all where it is skipped: rows of V that hold an infinity or NaN must not
  // be relied on to reach the output, nor not to.
  constexpr bool AHEAD = MASK && D <= 64 && !LEAN;
  uint32_t raw[8], mw[2];
  if (ntiles > 0) {
    load_kv(0);
    if constexpr (AHEAD) mask_load32(p, mrow, 0, lane, raw);
  }
  for (int t = 0; t < ntiles; ++t) {
    __syncthreads();  // every wavefront is done with the previous tile
    stash_kv();
    bool any = true, apply = false;
    if constexpr (AHEAD) {
      const uint32_t bits = mask_bits32(raw);
      any = __builtin_amdgcn_ballot_w64(bits != 0) != 0;
      apply = __builtin_amdgcn_ballot_w64(bits != 0xffffffffu) != 0;
      const auto both = __builtin_amdgcn_permlane32_swap(bits, bits, false, false);
      mw[0] = both[0] >> h32;  // keys 0 .. 31 of the tile, 4 h32 on
      mw[1] = both[1] >> h32;  // keys 32 .. 63
    }
    __syncthreads();
    if (t + 1 < ntiles) {
      load_kv(t + 1);
      if constexpr (AHEAD) mask_load32(p, mrow, t + 1, lane, raw);
    }
    if constexpr (AHEAD) {
      if (any)
        attn32_tile<D, SWZ, KLD, true>(Ks, Vs, qf, t, L, p.scale_log2,
                                       [&](int w) {
                                         return (mw[w >> 2] >> (2 * (w & 3))) & 0x01010101u;
                                       },
                                       apply, lane, o, m, l);
    } else if constexpr (MASK) {
      attn32_tile<D, SWZ, KLD, true>(
          Ks, Vs, qf, t, L, p.scale_log2,
          [&](int w) {
            return mask4(p, mrow, t * KT + 32 * (w >> 2) + 8 * (w & 3) + 4 * h32);
          },
          true, lane, o, m, l);
    } else {
      attn32_tile<D, SWZ, KLD, false>(Ks, Vs, qf, t, L, p.scale_log2, NoMask{}, false, lane, o, m,
                                      l);
    }
  }

  if (qvalid) {
    const float inv = l > 0.f ? 1.0f / l : 0.f;
#pragma unroll
    for (int dt = 0; dt < D / 32; ++dt)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        if (PAD && dt * 32 + 8 * g + 4 * h32 >= p.D) continue;
        f16x4 out;
#pragma unroll
        for (int j = 0; j < 4; ++j) out[j] = (f16)(o[dt][4 * g + j] * inv);
        *(f16x4 *)(Ob + qrow * p.so[2] + dt * 32 + 8 * g + 4 * h32) = out;
      }
  }
}

// fp16, D = 64, key-padding lengths only (no boolean mask): the arithmetic
// of fa_fwd_f16_kernel with NW (4 or 8) wavefronts of 32 queries, but K and V go
// global -> LDS by DMA (buffer_load ... lds, 16 bytes per lane, nothing
// staged in registers) into a ring of ST stages of one 64-key tile each
// (8 KB of K, then 8 KB of V), so that up to ST - 1 tiles are in flight
// while one is multiplied. One wavefront instruction moves 8 rows of the K or
// the V tile, lane l landing in slot l % 8 of row l / 8 of them, so it fetches the logical chunk whose
// kv_swz slot that is. Keys at or beyond Sk lie past the buffer's end and
// read as 0; keys in [valid length, Sk) are loaded and given probability 0,
// as in fa_fwd_f16_kernel. The host launches it only when every byte offset
// fits 31 bits. (A boolean mask is read from global memory inside the tile
// loop, and that load could only be waited for together with the DMA of the
// tiles in flight before it; fa_fwd_f16_kernel serves that case.)
template <int NW, int ST>
__global__ __launch_bounds__(NW * 64) void fa_fwd_f16_ring_kernel(AttnParams p) {
  constexpr int D = 64, KT = 64, TILE = KT * D * 2, IPW = 8 / NW;
  __shared__ __attribute__((aligned(1024))) char ring[ST * 2 * TILE];

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, h32 = lane >> 5;
  const AttnTile tile = attn_tile();
  const int b = tile.b, h = tile.h;
  const int L = valid_len(p, b);
  const f16 *Qb = (const f16 *)p.Q + b * p.sq[0] + h * p.sq[1];
  const f16 *Kb = (const f16 *)p.K + b * p.sk[0] + h * p.sk[1];
  const f16 *Vb = (const f16 *)p.V + b * p.sv[0] + h * p.sv[1];
  f16 *Ob = (f16 *)p.O + b * p.so[0] + h * p.so[1];

  const int qrow = tile.qb * (NW * 32) + wave * 32 + (lane & 31);
  const bool qvalid = qrow < p.Sq;
  f16x8 qf[D / 16];
#pragma unroll
  for (int c = 0; c < D / 16; ++c)
    qf[c] = qvalid ? *(const f16x8 *)(Qb + qrow * p.sq[2] + c * 16 + h32 * 8)
                   : f16x8{0, 0, 0, 0, 0, 0, 0, 0};
  f32x16 o[D / 32];
#pragma unroll
  for (int dt = 0; dt < D / 32; ++dt)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[dt][r] = 0.f;
  float m = -__builtin_inff(), l = 0.f;

  const int ntiles = (L + KT - 1) / KT;
  const int rsk = (int)(p.sk[2] * 2), rsv = (int)(p.sv[2] * 2);  // row strides, bytes
  const __amdgpu_buffer_rsrc_t rK = __builtin_amdgcn_make_buffer_rsrc(
      (void *)Kb, (short)0, (p.Sk - 1) * rsk + D * 2, 0x00020000);
  const __amdgpu_buffer_rsrc_t rV = __builtin_amdgcn_make_buffer_rsrc(
      (void *)Vb, (short)0, (p.Sk - 1) * rsv + D * 2, 0x00020000);
  int offK[IPW], offV[IPW];
#pragma unroll
  for (int i = 0; i < IPW; ++i) {
    const int trow = (wave * IPW + i) * 8 + (lane >> 3), chunk = (lane & 7) ^ kv_swz(trow);
    offK[i] = trow * rsk + chunk * 16;
    offV[i] = trow * rsv + chunk * 16;
  }
  // 2 IPW instructions per tile and wavefront. The host compilation pass sees
  // an empty statement (its check of this builtin with a run-time offset
  // rejects the kernel).
  auto issue = [&](int t, int stage) {
#if defined(__HIP_DEVICE_COMPILE__)
    char *ks = ring + stage * 2 * TILE + wave * IPW * 1024;
#pragma unroll
    for (int i = 0; i < IPW; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rK, ZK_LDS(ks + i * 1024), 16,
                                               offK[i] + t * KT * rsk, 0, 0, 0);
#pragma unroll
    for (int i = 0; i < IPW; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rV, ZK_LDS(ks + TILE + i * 1024), 16,
                                               offV[i] + t * KT * rsv, 0, 0, 0);
#else
    (void)t, (void)stage;
#endif
  };
#pragma unroll
  for (int s = 0; s < ST; ++s)
    if (s < ntiles) issue(s, s);
  if (ntiles > 0) {
    wait_slices<ST - 1, 2 * IPW>(ntiles - 1);
    lds_barrier();
  }
  int stage = 0;
  for (int t = 0; t < ntiles; ++t) {
    const char *ks = ring + stage * 2 * TILE;
    attn32_tile<D, true, D, false>((const f16 *)ks, (const f16 *)(ks + TILE), qf, t, L,
                                   p.scale_log2, NoMask{}, false, lane, o, m, l);
    if (t + 1 < ntiles) {
      // tile t + 1 has landed (up to ST - 2 younger tiles still in flight),
      // and after the barrier every wavefront is done reading tile t, whose
      // stage then receives tile t + ST
      wait_slices<ST - 2, 2 * IPW>(ntiles - 2 - t);
      lds_barrier();
      if (t + ST < ntiles) issue(t + ST, stage);
      stage = stage + 1 == ST ? 0 : stage + 1;
    }
  }

  if (qvalid) {
    const float inv = l > 0.f ? 1.0f / l : 0.f;
#pragma unroll
    for (int dt = 0; dt < D / 32; ++dt)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        f16x4 out;
#pragma unroll
        for (int j = 0; j < 4; ++j) out[j] = (f16)(o[dt][4 * g + j] * inv);
        *(f16x4 *)(Ob + qrow * p.so[2] + dt * 32 + 8 * g + 4 * h32) = out;
      }
  }
}

__device__ __forceinline__ f16x8 load8_f16(const f16 *p) { return *(const f16x8 *)p; }
__device__ __forceinline__ f16x8 load8_f16(const float *p) {
  const f32x4 lo = *(const f32x4 *)p, hi = *(const f32x4 *)(p + 4);
  return f16x8{(f16)lo[0], (f16)lo[1], (f16)lo[2], (f16)lo[3],
               (f16)hi[0], (f16)hi[1], (f16)hi[2], (f16)hi[3]};
}

// fp16, D = 64, 16 queries per wavefront on 16x16x32 MFMAs, NW wavefronts
// per workgroup. Same arithmetic as fa_fwd_f16_kernel (fp32 statistics, exp2
// with the scale folded in, lazy rescaling, P rounded to fp16), with half
// the per-wavefront dependency chain and twice the wavefronts.
// S^T = K . Q^T: lane l supplies K[key 16 kb + l%16][dims 8 (l/16) + 32 ks ..]
// and Q[query l%16][same dims], and receives S^T[16 kb + 4 (l/16) + r][l%16].
// O^T += V^T . P^T over 32 keys per step: k-slot 8 g + j (g = l / 16) is key
// 4 g + j for j < 4 and 16 + 4 g + (j - 4) otherwise, so the B operand is the
// lane's own probabilities of key blocks 2 st and 2 st + 1, and the V^T
// operand comes from two transposing reads 16 keys apart.
// IO: f16, or float for tensors in fp32 that are rounded to fp16 as they are
// loaded (and the fp16 output widened as it is stored).
template <int NW, int TPS = 1, bool MASK = false, typename IO = f16>
__global__ __launch_bounds__(NW * 64) void fa_fwd_f16_q16_kernel(AttnParams p) {
  constexpr int D = 64, KT = 64, NT = NW * 64, DV = D / 8;
  constexpr int PER = TPS * KT * DV / NT;  // TPS key tiles per LDS stage
  static_assert(TPS * KT * DV % NT == 0 && PER >= 1, "tile/thread mismatch");
  __shared__ __attribute__((aligned(16))) f16 Ks[TPS * KT * D];
  __shared__ __attribute__((aligned(16))) f16 Vs[TPS * KT * D];

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int g = lane >> 4, c16 = lane & 15;
  const AttnTile tile = attn_tile();
  const int b = tile.b, h = tile.h;
  const int L = valid_len(p, b);
  const IO *Qb = (const IO *)p.Q + b * p.sq[0] + h * p.sq[1];
  const IO *Kb = (const IO *)p.K + b * p.sk[0] + h * p.sk[1];
  const IO *Vb = (const IO *)p.V + b * p.sv[0] + h * p.sv[1];
  IO *Ob = (IO *)p.O + b * p.so[0] + h * p.so[1];

  const int qrow = tile.qb * (NW * 16) + wave * 16 + c16;
  const bool qvalid = qrow < p.Sq;
  const uint8_t *mrow = MASK ? mask_row(p, b, h, qvalid ? qrow : 0) : nullptr;
  f16x8 qf[2];
#pragma unroll
  for (int ks = 0; ks < 2; ++ks)
    qf[ks] = qvalid ? load8_f16(Qb + qrow * p.sq[2] + 32 * ks + 8 * g)
                    : f16x8{0, 0, 0, 0, 0, 0, 0, 0};

  f32x4 o[4];
#pragma unroll
  for (int db = 0; db < 4; ++db) o[db] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m = -__builtin_inff(), l = 0.f;

  const int ntiles = (L + KT - 1) / KT;
  const int nstages = (ntiles + TPS - 1) / TPS;
  f16x8 kr[PER], vr[PER];
  auto load_kv = [&](int stg) {
#pragma unroll
    for (int v = 0; v < PER; ++v) {
      const int idx = tid + v * NT;
      const int kk = stg * TPS * KT + idx / DV;
      kr[v] = kk < p.Sk ? load8_f16(Kb + kk * p.sk[2] + (idx % DV) * 8)
                        : f16x8{0, 0, 0, 0, 0, 0, 0, 0};
      vr[v] = kk < p.Sk ? load8_f16(Vb + kk * p.sv[2] + (idx % DV) * 8)
                        : f16x8{0, 0, 0, 0, 0, 0, 0, 0};
    }
  };
  auto stash_kv = [&]() {
#pragma unroll
    for (int v = 0; v < PER; ++v) {
      const int idx = tid + v * NT;
      const int row = idx / DV, ch = (idx % DV) ^ kv_swz16(idx / DV);
      *(f16x8 *)(Ks + row * D + ch * 8) = kr[v];
      *(f16x8 *)(Vs + row * D + ch * 8) = vr[v];
    }
  };
  // V^T source address of this lane: key 4 g + l%16 / 4 (+ 32 st, + 16),
  // dims 16 db + 4 (l % 4); with the swizzle, chunk 2 db + (l%4)/2 of a row
  // r is in slot chunk ^ kv_swz16(r), and kv_swz16 ignores the +32 st / +16.
  const int r0 = 4 * g + (c16 >> 2);
  const int fv = kv_swz16(r0), vhalf = (c16 & 3) >> 1, vin = 4 * (c16 & 1);

  if (nstages > 0) load_kv(0);
  for (int stg = 0; stg < nstages; ++stg) {
    __syncthreads();
    stash_kv();
    __syncthreads();
    if (stg + 1 < nstages) load_kv(stg + 1);
    for (int sub = 0; sub < TPS; ++sub) {
      const int t = stg * TPS + sub;
      if (t >= ntiles) break;  // wave-uniform; no barrier in this loop
      const f16 *Kt = Ks + sub * KT * D;
      const f16 *Vt = Vs + sub * KT * D;

      f32x4 s4[4];
#pragma unroll
      for (int kb = 0; kb < 4; ++kb) {
        s4[kb] = f32x4{0.f, 0.f, 0.f, 0.f};
        const int row = 16 * kb + c16;
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
          const f16x8 kf = *(const f16x8 *)(Kt + row * D + (((4 * ks + g) ^ kv_swz16(row)) << 3));
          s4[kb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf, qf[ks], s4[kb], 0, 0, 0);
        }
      }
      if (t * KT + KT > L) {
#pragma unroll
        for (int kb = 0; kb < 4; ++kb)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (t * KT + 16 * kb + 4 * g + r >= L) s4[kb][r] = -__builtin_inff();
      }
      if constexpr (MASK) {
#pragma unroll
        for (int kb = 0; kb < 4; ++kb) {
          const uint32_t m4 = mask4(p, mrow, t * KT + 16 * kb + 4 * g);
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (((m4 >> (8 * r)) & 0xffu) == 0) s4[kb][r] = -__builtin_inff();
        }
      }
      float tmax = -__builtin_inff();
#pragma unroll
      for (int kb = 0; kb < 4; ++kb)
        tmax = smax(smax(tmax, s4[kb][0]), smax(s4[kb][1], smax(s4[kb][2], s4[kb][3])));
      const auto smax_op = [](float a, float b) { return smax(a, b); };
      tmax = bfly<16>(tmax, smax_op);
      // finite unless MASK (without a mask, key t*KT < L is valid)
      tmax = bfly<32>(tmax, smax_op) * p.scale_log2;
      if (__builtin_amdgcn_ballot_w64(tmax > m + 8.0f) != 0) {
        const float m_new = fmaxf(m, tmax);
        const float alpha = MASK && m_new == -__builtin_inff() ? 1.0f
                                                               : __builtin_amdgcn_exp2f(m - m_new);
        m = m_new;
        l *= alpha;
#pragma unroll
        for (int db = 0; db < 4; ++db)
#pragma unroll
          for (int r = 0; r < 4; ++r) o[db][r] *= alpha;
      }
      const float mneg = MASK && m == -__builtin_inff() ? 0.0f : -m;
      float psum = 0.f;
      f16x8 pf[2];
#pragma unroll
      for (int kb = 0; kb < 4; ++kb)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float e = __builtin_amdgcn_exp2f(fmaf(s4[kb][r], p.scale_log2, mneg));
          psum += e;
          pf[kb >> 1][4 * (kb & 1) + r] = (f16)e;
        }
      psum = bfly<16>(psum, OpAdd{});
      psum = bfly<32>(psum, OpAdd{});
      l += psum;
#pragma unroll
      for (int db = 0; db < 4; ++db)
#pragma unroll
        for (int st = 0; st < 2; ++st) {
          const f16 *row = Vt + (32 * st + r0) * D + ((((2 * db + vhalf) ^ fv)) << 3) + vin;
          const f16x4 lo = lds_read_tr16(row);
          const f16x4 hi = lds_read_tr16(row + 16 * D);
          const f16x8 vf = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
          o[db] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vf, pf[st], o[db], 0, 0, 0);
        }
    }
  }

  if (qvalid) {
    const float inv = l > 0.f ? 1.0f / l : 0.f;
#pragma unroll
    for (int db = 0; db < 4; ++db) {
      f16x4 out;
#pragma unroll
      for (int r = 0; r < 4; ++r) out[r] = (f16)(o[db][r] * inv);
      if constexpr (std::is_same<IO, float>::value)
        *(f32x4 *)(Ob + qrow * p.so[2] + 16 * db + 4 * g) =
            f32x4{(float)out[0], (float)out[1], (float)out[2], (float)out[3]};
      else
        *(f16x4 *)(Ob + qrow * p.so[2] + 16 * db + 4 * g) = out;
    }
  }
}

// ---------------------------------------------------------------- fp32 ----
// fp32 attention on the fp32 matrix instructions (v_mfma_f32_16x16x4_f32,
// 64 FLOP per cycle and SIMD, twice the FMA pipe's rate). 16 queries per
// wavefront; a workgroup of four wavefronts owns 16 * 4 / KS queries and
// splits each 64-key stage KS ways between the wavefronts of one query
// group, whose partial (m, l, O) are merged through LDS at the end.
// S^T = K . Q^T in blocks of 16 keys: lane l (g = l / 16) reads 16 bytes,
// dims 16 c + 4 g .. +3 of key (or query) l % 16, and the four products of
// element j cover dims 16 c + 4 g + j. It receives scores of keys 4 g + r of
// query l % 16 in register r, which is the B operand of the product over
// keys {4 g + r : g} of O^T += V^T . P^T: P never leaves registers. The
// V^T operand is read VW (2 or 4) consecutive dims at a time from the row-
// major V tile: row i of output block dt is dim VW i + dt of the group, so a
// lane ends with VW consecutive dims and stores them as one vector.
// LDS rows of D + 4 floats: 16 rows of a K fragment read start 4 banks apart,
// and a V read covers whole rows; both are conflict-free.
// Bound: the fp32 matrix rate where the grid fills the 1024 SIMDs, else one
// wavefront's chain of stages, which KS shortens. b4 h12 s256 d64: 103 us on
// the FMA pipe (D / 32 lanes per query, K and V broadcast from LDS) -> 16.5 us,
// 49 TFLOP/s; b16 h12 s256 130 -> 38 us, b4 h16 s1024 d128 1305 -> 315 us (110
// TFLOP/s).
// Stored head dims p.D <= D are zero-padded (dims >= p.D are read as zeros and
// not stored). VEC: every row of Q, K, V and O starts on 16 bytes and
// p.D % 4 == 0; otherwise elements are loaded and stored one by one. Keys at
// or past the valid length are read as zeros.
template <int D, int KS, bool MASK, bool VEC>
__global__ __launch_bounds__(256, 2) void fa_fwd_f32_kernel(AttnParams p) {
  constexpr int QW = 4 / KS, KB = 4 / KS;  // query groups; key blocks per wave and stage
  constexpr int KT = 64, PITCH = D + 4, DV = D / 4, PER = KT * DV / 256;
  constexpr int VW = D % 64 == 0 ? 4 : 2, NG = D / (16 * VW);
  constexpr int SMEM = 2 * KT * PITCH;
  // merge: (m, l, O) of the KS - 1 other wavefronts of every query group
  constexpr int MW = D / 4 + 2;
  static_assert(QW * (KS - 1) * 64 * MW <= SMEM, "merge space");
  __shared__ __attribute__((aligned(16))) float smem[SMEM];
  float *Ks = smem, *Vs = smem + KT * PITCH;

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int g = lane >> 4, c16 = lane & 15;
  const int ks = wave % KS, qw = wave / KS;
  const AttnTile tile = attn_tile();
  const int b = tile.b, h = tile.h;
  const int L = valid_len(p, b);
  const float *Qb = (const float *)p.Q + b * p.sq[0] + h * p.sq[1];
  const float *Kb = (const float *)p.K + b * p.sk[0] + h * p.sk[1];
  const float *Vb = (const float *)p.V + b * p.sv[0] + h * p.sv[1];
  float *Ob = (float *)p.O + b * p.so[0] + h * p.so[1];
  // 4 consecutive floats of a row, zero from dim p.D on (or everywhere)
  auto load4 = [&](const float *row, int d, bool in) {
    f32x4 v = {0.f, 0.f, 0.f, 0.f};
    if constexpr (VEC) {
      if (in && d < p.D) v = *(const f32x4 *)(row + d);
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (in && d + j < p.D) v[j] = row[d + j];
    }
    return v;
  };

  const int qrow = (tile.qb * QW + qw) * 16 + c16;
  const bool qvalid = qrow < p.Sq;
  const uint8_t *mrow = MASK ? mask_row(p, b, h, qvalid ? qrow : 0) : nullptr;
  f32x4 qf[D / 16];
#pragma unroll
  for (int c = 0; c < D / 16; ++c)
    qf[c] = load4(Qb + (qvalid ? qrow : 0) * p.sq[2], 16 * c + 4 * g, qvalid);
  f32x4 o[D / 16];
#pragma unroll
  for (int i = 0; i < D / 16; ++i) o[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m = -__builtin_inff(), l = 0.f;  // l: this lane's keys only until the end

  const int nst = (L + KT - 1) / KT;
  f32x4 kr[PER], vr[PER];
  auto load_kv = [&](int t) {
#pragma unroll
    for (int v = 0; v < PER; ++v) {
      const int idx = tid + v * 256, key = t * KT + idx / DV, d = (idx % DV) * 4;
      const bool in = key < L;
      kr[v] = load4(Kb + (in ? key : 0) * p.sk[2], d, in);
      vr[v] = load4(Vb + (in ? key : 0) * p.sv[2], d, in);
    }
  };
  if (nst > 0) load_kv(0);
  for (int t = 0; t < nst; ++t) {
    __syncthreads();  // every wavefront is done with the previous stage
#pragma unroll
    for (int v = 0; v < PER; ++v) {
      const int idx = tid + v * 256, at = (idx / DV) * PITCH + (idx % DV) * 4;
      *(f32x4 *)(Ks + at) = kr[v];
      *(f32x4 *)(Vs + at) = vr[v];
    }
    __syncthreads();
    if (t + 1 < nst) load_kv(t + 1);
    const int kw = ks * KB * 16, k0 = t * KT + kw;  // this wavefront's first key
    if (k0 >= L) continue;  // wave-uniform; no barrier is skipped

    // NC independent chains per score, 32 dims each, added at the end: a
    // chain's rounding error grows with its length
    constexpr int NC = D / 32;
    f32x4 sc[NC][KB];
#pragma unroll
    for (int n = 0; n < NC; ++n)
#pragma unroll
      for (int kb = 0; kb < KB; ++kb) sc[n][kb] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int c2 = 0; c2 < 2; ++c2)
#pragma unroll
      for (int n = 0; n < NC; ++n) {
        const int c = 2 * n + c2;
        f32x4 kf[KB];
#pragma unroll
        for (int kb = 0; kb < KB; ++kb)
          kf[kb] = *(const f32x4 *)(Ks + (kw + 16 * kb + c16) * PITCH + 16 * c + 4 * g);
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int kb = 0; kb < KB; ++kb)
            sc[n][kb] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[kb][j], qf[c][j], sc[n][kb], 0,
                                                             0, 0);
      }
    f32x4 s[KB];
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) {
      if constexpr (NC == 1) s[kb] = sc[0][kb];
      else if constexpr (NC == 2) s[kb] = sc[0][kb] + sc[1][kb];
      else if constexpr (NC == 3) s[kb] = (sc[0][kb] + sc[1][kb]) + sc[2][kb];
      else s[kb] = (sc[0][kb] + sc[1][kb]) + (sc[2][kb] + sc[3][kb]);
    }
    float tmin = __builtin_inff();  // of all keys, kept or not
#pragma unroll
    for (int kb = 0; kb < KB; ++kb)
#pragma unroll
      for (int r = 0; r < 4; ++r) tmin = smin(tmin, s[kb][r]);
    if (k0 + KB * 16 > L) {  // the stage that straddles the valid length
#pragma unroll
      for (int kb = 0; kb < KB; ++kb)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (k0 + 16 * kb + 4 * g + r >= L) s[kb][r] = -__builtin_inff();
    }
    if constexpr (MASK) {
#pragma unroll
      for (int kb = 0; kb < KB; ++kb) {
        const uint32_t m4 = mask4(p, mrow, k0 + 16 * kb + 4 * g);
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (((m4 >> (8 * r)) & 0xffu) == 0) s[kb][r] = -__builtin_inff();
      }
    }
    float tmax = -__builtin_inff();
#pragma unroll
    for (int kb = 0; kb < KB; ++kb)
#pragma unroll
      for (int r = 0; r < 4; ++r) tmax = fmaxf(tmax, s[kb][r]);
    tmax = bfly<16>(tmax, OpMax{});
    tmax = bfly<32>(tmax, OpMax{}) * p.scale_log2;  // the scale is positive
    if (__builtin_amdgcn_ballot_w64(tmax > m) != 0) {
      const float m_new = fmaxf(m, tmax);
      // a query whose keys so far are all masked keeps m = -inf: no rescale
      const float alpha =
          m_new == -__builtin_inff() ? 1.0f : exp2f(m - m_new);
      m = m_new;
      l *= alpha;
#pragma unroll
      for (int i = 0; i < D / 16; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) o[i][r] *= alpha;
    }
    const float mneg = m == -__builtin_inff() ? 0.0f : -m;  // exp2(-inf + 0) = 0
#pragma unroll
    for (int kb = 0; kb < KB; ++kb)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        s[kb][r] = __builtin_amdgcn_exp2f(fmaf(s[kb][r], p.scale_log2, mneg));
        l += s[kb][r];
      }
#pragma unroll
    for (int kb = 0; kb < KB; ++kb)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        typedef float VF __attribute__((ext_vector_type(VW)));
        const float *row = Vs + (kw + 16 * kb + 4 * g + r) * PITCH + VW * c16;
#pragma unroll
        for (int n = 0; n < NG; ++n) {
          const VF vf = *(const VF *)(row + 16 * VW * n);
#pragma unroll
          for (int dt = 0; dt < VW; ++dt)
            o[n * VW + dt] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[dt], s[kb][r],
                                                                 o[n * VW + dt], 0, 0, 0);
        }
      }
    // v_exp_f32 makes results below 2^-126 zero, exp2f goes down to the
    // subnormals: such a key still counts where its V is large. What the
    // instruction left out of this stage is formed again and added here, after
    // it and one key block at a time, which costs stages that need none 0.4% on
    // average (D = 64: 2%; b4 h12 s256 14.9 -> 15.3 us). Scores so far apart that
    // every stage takes it (q 15 times N(0, 1)): b4 h12 s256 26.5 us, b4 h16 s1024
    // d128 560 (299 otherwise; 1340 on the FMA pipe). exp2f throughout costs 3
    // to 9%, a branch before the products 5 to 7% of the short chains, a second
    // pass over all keys at the end 1.6%; with the scores held or the blocks
    // unrolled here D = 128 spills.
    if (__builtin_expect(
            __builtin_amdgcn_ballot_w64(fmaf(tmin, p.scale_log2, mneg) < -125.f) != 0, 0)) {
#pragma unroll 1
      for (int kb = 0; kb < KB; ++kb) {
        f32x4 c1[NC], x;
#pragma unroll
        for (int n = 0; n < NC; ++n) {
          c1[n] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int c = 2 * n; c < 2 * n + 2; ++c) {
            const f32x4 kf = *(const f32x4 *)(Ks + (kw + 16 * kb + c16) * PITCH + 16 * c + 4 * g);
#pragma unroll
            for (int j = 0; j < 4; ++j)
              c1[n] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[j], qf[c][j], c1[n], 0, 0, 0);
          }
        }
        if constexpr (NC == 1) x = c1[0];
        else if constexpr (NC == 2) x = c1[0] + c1[1];
        else if constexpr (NC == 3) x = (c1[0] + c1[1]) + c1[2];
        else x = (c1[0] + c1[1]) + (c1[2] + c1[3]);
        const int key = 16 * kb + 4 * g;  // of this wavefront's
        uint32_t m4 = 0x01010101u;
        if constexpr (MASK) m4 = mask4(p, mrow, k0 + key);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const bool kept = k0 + key + r < L && ((m4 >> (8 * r)) & 0xffu) != 0;
          const float y = fmaf(x[r], p.scale_log2, mneg);
          const float e = kept && y < -125.f ? exp2f(y) - __builtin_amdgcn_exp2f(y) : 0.f;
          l += e;
          typedef float VF __attribute__((ext_vector_type(VW)));
          const float *row = Vs + (kw + key + r) * PITCH + VW * c16;
#pragma unroll
          for (int n = 0; n < NG; ++n) {
            const VF vf = *(const VF *)(row + 16 * VW * n);
#pragma unroll
            for (int dt = 0; dt < VW; ++dt)
              o[n * VW + dt] =
                  __builtin_amdgcn_mfma_f32_16x16x4f32(vf[dt], e, o[n * VW + dt], 0, 0, 0);
          }
        }
      }
    }
  }
  l = bfly<16>(l, OpAdd{});
  l = bfly<32>(l, OpAdd{});

  if constexpr (KS > 1) {
    // Merge in the order ks = 0, 1, ..: every wavefront's O and l at the
    // common maximum (a wavefront that saw no key has m = -inf, l = 0).
    __syncthreads();  // the tiles are no longer read
    float *mine = smem + (qw * (KS - 1) + ks - 1) * 64 * MW + lane;
    if (ks > 0) {
      mine[0] = m;
      mine[64] = l;
#pragma unroll
      for (int i = 0; i < D / 16; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) mine[(2 + 4 * i + r) * 64] = o[i][r];
    }
    __syncthreads();
    if (ks > 0) return;
    float mt = m;
#pragma unroll
    for (int k = 0; k < KS - 1; ++k) mt = fmaxf(mt, mine[(k + 1) * 64 * MW]);
    const float mref = mt == -__builtin_inff() ? 0.0f : mt;
    const float f0 = exp2f(m - mref);
    l *= f0;
#pragma unroll
    for (int i = 0; i < D / 16; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) o[i][r] *= f0;
#pragma unroll
    for (int k = 0; k < KS - 1; ++k) {
      const float *part = mine + (k + 1) * 64 * MW;
      const float f = exp2f(part[0] - mref);
      l = fmaf(part[64], f, l);
#pragma unroll
      for (int i = 0; i < D / 16; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) o[i][r] = fmaf(part[(2 + 4 * i + r) * 64], f, o[i][r]);
    }
  }
  if (!qvalid) return;
  const float inv = l > 0.f ? 1.0f / l : 0.f;
  float *orow = Ob + qrow * p.so[2];
#pragma unroll
  for (int n = 0; n < NG; ++n)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int d = 16 * VW * n + VW * (4 * g + r);
      typedef float VF __attribute__((ext_vector_type(VW)));
      VF v;
#pragma unroll
      for (int dt = 0; dt < VW; ++dt) v[dt] = o[n * VW + dt][r] * inv;
      if constexpr (VEC) {
        if (d < p.D) *(VF *)(orow + d) = v;
      } else {
#pragma unroll
        for (int dt = 0; dt < VW; ++dt)
          if (d + dt < p.D) orow[d + dt] = v[dt];
      }
    }
}

template <bool MASK, typename IO>
static void launch_q16(const AttnParams &p, hipStream_t s) {
  if ((unsigned)((p.Sq + 63) / 64) * (unsigned)p.H * (unsigned)p.B < 256) {
    dim3 grid((unsigned)((p.Sq + 15) / 16), (unsigned)p.H, (unsigned)p.B);
    fa_fwd_f16_q16_kernel<1, 1, MASK, IO><<<grid, 64, 0, s>>>(p);
  } else {
    dim3 grid((unsigned)((p.Sq + 63) / 64), (unsigned)p.H, (unsigned)p.B);
    fa_fwd_f16_q16_kernel<4, 1, MASK, IO><<<grid, 256, 0, s>>>(p);
  }
}

template <int D, bool PAD = false, bool MASK = false>
static void launch_f16_m(const AttnParams &p, hipStream_t s) {
  // 4 wavefronts x 32 queries per workgroup: at seq 128 one workgroup holds a
  // whole (batch, head), so K and V are read from HBM once.
  // Up to 128 queries (BERT s128), D = 64: 16-query wavefronts, 4 per
  // workgroup. The shorter per-wave chain and the doubled wave count win
  // where the kernel is latency-bound (encoder 0.5% faster per step at b32
  // s128); at s512 the 32-query kernel's lower LDS traffic per query wins.
  if constexpr (D == 64 && !PAD) {
    if (p.Sq <= 128) {
      // one 64-key tile per LDS stage, the next one loading under the
      // current one's MFMAs. Staging both tiles of a 128-key sequence at once
      // (TPS = 2) was 0.7% slower per encoder step, fp16 and INT8-FFN, in
      // both-order A/Bs on two boxes. A few (batch, head) pairs (one to
      // four 128-token sequences: 96 to 384 workgroups of one wavefront
      // instead of 24 to 96 of four) take one wavefront per workgroup, so
      // that more CUs share the work.
      launch_q16<MASK, f16>(p, s);
      return;
    }
  }
  // D = 64 with lengths only, from 128 queries: K and V DMA'd into a 3-stage
  // ring. 128 queries (4 wavefronts) per workgroup, or 256 where these give at
  // least three workgroups per CU and the last block of 256 is more than half
  // full. 256 / 128 queries, us: b32 h12 s512 40.5 / 41.1 (lengths U{S/2..S}),
  // b16 h16 s1024 79.3 / 80.8; b16 h12 s512 27.2 / 24.6 (384 workgroups of 256
  // leave half the CUs one, half two), b8 h12 s1024 42.0 / 37.7, b8 h12 s768
  // 31.4 / 27.6, b12 h12 s384 18.1 / 14.3 (a quarter of 2 x 256 is padding), b2
  // h12 s512 12.4 / 9.5. Against the kernel that stages through registers:
  // b32 h12 s256 17.8 -> 17.1, b16 h12 s200 10.2 -> 10.0.
  if constexpr (D == 64 && !PAD && !MASK) {
    const int64_t rs = 2 * (p.sk[2] > p.sv[2] ? p.sk[2] : p.sv[2]);
    if (p.Sq >= 128 && rs >= 0 && ((int64_t)p.Sk + 64) * rs + 128 < (int64_t(1) << 31)) {
      const int64_t w8 = (int64_t)((p.Sq + 255) / 256) * p.H * p.B;
      if (w8 >= 768 && (p.Sq - 1) % 256 >= 128) {
        dim3 grid((unsigned)((p.Sq + 255) / 256), (unsigned)p.H, (unsigned)p.B);
        fa_fwd_f16_ring_kernel<8, 3><<<grid, 512, 0, s>>>(p);
      } else {
        dim3 grid((unsigned)((p.Sq + 127) / 128), (unsigned)p.H, (unsigned)p.B);
        fa_fwd_f16_ring_kernel<4, 3><<<grid, 256, 0, s>>>(p);
      }
      return;
    }
  }
  // Masks at D = 64: a CU holds two workgroups of 128 queries (200 registers),
  // four of 64, or three of 128 that read their mask bytes inside the tile
  // (LEAN, 162). Past one round of the first the others where they still fit in
  // one. us, random / causal / lengths mask, h12: b16 s300, 576 workgroups of 128
  // or 960 of 64: 26.8 / 22.8 / 23.3 -> 19.6 / 17.7 / 18.2; b24 s192 19.1 / 17.0 /
  // 17.7 -> 13.8 / 12.2 / 13.0; LEAN: b20 s300 27.6 / 25.6 / 26.1 -> 22.5, b12 s500
  // 40.1 / 36.3 / 34.0 -> 32.5. Rows of whole 64-byte lines gain less from it
  // than from skipping tiles (b16 s384 32.6 / 26.4 / 28.7, LEAN 30.5).
  if constexpr (MASK && D == 64) {
    const int64_t bh = (int64_t)p.H * p.B, w4 = (p.Sq + 127) / 128 * bh, w2 = (p.Sq + 63) / 64 * bh;
    if (w4 > 512 && w2 <= 1024) {
      dim3 grid((unsigned)((p.Sq + 63) / 64), (unsigned)p.H, (unsigned)p.B);
      fa_fwd_f16_kernel<D, 2, PAD, MASK><<<grid, 128, 0, s>>>(p);
      return;
    }
    if (p.Sq >= 128 && w4 > 512 && w4 <= 768 && p.Sk % 64 != 0) {
      dim3 grid((unsigned)((p.Sq + 127) / 128), (unsigned)p.H, (unsigned)p.B);
      fa_fwd_f16_kernel<D, 4, PAD, MASK, true><<<grid, 256, 0, s>>>(p);
      return;
    }
  }
  if (p.Sq >= 128) {
    dim3 grid((unsigned)((p.Sq + 127) / 128), (unsigned)p.H, (unsigned)p.B);
    fa_fwd_f16_kernel<D, 4, PAD, MASK><<<grid, 256, 0, s>>>(p);
  } else {
    dim3 grid((unsigned)((p.Sq + 63) / 64), (unsigned)p.H, (unsigned)p.B);
    fa_fwd_f16_kernel<D, 2, PAD, MASK><<<grid, 128, 0, s>>>(p);
  }
}

template <int D, bool PAD = false>
static void launch_f16(const AttnParams &p, hipStream_t s) {
  if (p.mask) launch_f16_m<D, PAD, true>(p, s);
  else launch_f16_m<D, PAD, false>(p, s);
}

template <int D, int KS, bool MASK>
static void launch_f32_ks(const AttnParams &p, bool vec, hipStream_t s) {
  constexpr int QPB = 16 * 4 / KS;
  dim3 grid((unsigned)((p.Sq + QPB - 1) / QPB), (unsigned)p.H, (unsigned)p.B);
  if (vec) fa_fwd_f32_kernel<D, KS, MASK, true><<<grid, 256, 0, s>>>(p);
  else fa_fwd_f32_kernel<D, KS, MASK, false><<<grid, 256, 0, s>>>(p);
}

template <int D>
static void launch_f32(const AttnParams &p, hipStream_t s) {
  // 16-byte accesses: every row start of Q, K, V and O on 16 bytes
  bool vec = p.D % 4 == 0 && aligned16(p.Q) && aligned16(p.K) && aligned16(p.V) && aligned16(p.O);
  for (int i = 0; i < 3; ++i)
    vec = vec && p.sq[i] % 4 == 0 && p.sk[i] % 4 == 0 && p.sv[i] % 4 == 0 && p.so[i] % 4 == 0;
  const int64_t w64 = (int64_t)((p.Sq + 63) / 64) * p.H * p.B;  // workgroups without a key split
  // Key split: 64 queries per workgroup once that gives two workgroups per CU
  // (b16 h12 s256: 38 us whole, 42 in 2 splits, 51 in 4), fewer queries and
  // the keys split 2 or 4 ways where the grid would leave SIMDs idle (b8 h12
  // s256: 25.4 / 23.5 / 28.5 us; b2 h12 s300 d80: 24.9 / 17.2 / 17.9; b1 h12
  // s128: 8.7 / 6.8 / 5.9).
  const int ks = w64 >= 512 ? 1 : w64 >= 160 ? 2 : 4;
#define ZK_F32(KS) \
  (p.mask ? launch_f32_ks<D, KS, true>(p, vec, s) : launch_f32_ks<D, KS, false>(p, vec, s))
  if (ks == 4) ZK_F32(4);
  else if (ks == 2) ZK_F32(2);
  else ZK_F32(1);
#undef ZK_F32
}

}  // namespace zk

using namespace zk;

static int attn_impl(const char *who, const void *Q, const void *K, const void *V, void *O,
                     int64_t batch, int64_t heads, int64_t seq_q, int64_t seq_k,
                     int64_t head_dim, const int64_t *strides, const int32_t *valid_lens,
                     const uint8_t *mask, const int64_t *mask_strides, float scale, int dtype,
                     void *stream, bool f32_io = false) {
  if (batch < 0 || heads < 0 || seq_q < 0 || seq_k < 0 || head_dim <= 0)
    return fail(ZK_ERR_INVALID, "%s: bad size", who);
  if (batch == 0 || heads == 0 || seq_q == 0) return ZK_OK;
  if (!Q || !K || !V || !O || !strides) return fail(ZK_ERR_INVALID, "%s: null pointer", who);
  if (batch > 65535 || heads > 65535 || seq_q > 0x7fffffff || seq_k > 0x7fffffff)
    return fail(ZK_ERR_UNSUPPORTED, "%s: size exceeds launch limits", who);
  // any head_dim up to 128, the reference's HEAD_DIM_MAX (flash_attention.cu:26)
  if (head_dim > 128)
    return fail(ZK_ERR_UNSUPPORTED, "%s: head_dim %lld > 128", who, (long long)head_dim);
  if (!(scale > 0.0f) || scale == __builtin_inff())
    return fail(ZK_ERR_INVALID, "%s: scale must be finite and > 0", who);
  for (int i = 0; i < 12; ++i)
    if (strides[i] < 0) return fail(ZK_ERR_INVALID, "%s: negative stride", who);
  AttnParams p;
  p.Q = Q; p.K = K; p.V = V; p.O = O;
  p.B = (int)batch; p.H = (int)heads; p.Sq = (int)seq_q; p.Sk = (int)seq_k;
  p.D = (int)head_dim;
  for (int i = 0; i < 3; ++i) {
    p.sq[i] = strides[i]; p.sk[i] = strides[3 + i];
    p.sv[i] = strides[6 + i]; p.so[i] = strides[9 + i];
  }
  p.valid_lens = valid_lens;
  p.mask = mask;
  p.sm[0] = p.sm[1] = p.sm[2] = 0;
  if (mask) {
    if (!mask_strides) return fail(ZK_ERR_INVALID, "%s: mask without strides", who);
    for (int i = 0; i < 3; ++i) {
      if (mask_strides[i] < 0) return fail(ZK_ERR_INVALID, "%s: negative mask stride", who);
      if (mask_strides[i] % 4)
        return fail(ZK_ERR_UNSUPPORTED, "%s: mask strides must be multiples of 4", who);
      p.sm[i] = mask_strides[i];
    }
    if (reinterpret_cast<uintptr_t>(mask) & 3u)
      return fail(ZK_ERR_UNSUPPORTED, "%s: mask must be 4-byte aligned", who);
  }
  p.scale_log2 = scale * 1.4426950408889634f;
  hipStream_t s = as_stream(stream);
  if (f32_io) {
    if (head_dim != 64 || seq_q > 128)
      return fail(ZK_ERR_UNSUPPORTED, "%s: head_dim must be 64 and seq_q at most 128", who);
    bool ok = aligned16(Q) && aligned16(K) && aligned16(V) && aligned16(O);
    for (int i = 0; i < 12; ++i) ok = ok && strides[i] % 4 == 0;
    if (!ok) return fail(ZK_ERR_UNSUPPORTED, "%s: rows must start on 16 bytes", who);
    launch_q16<false, float>(p, s);
  } else if (dtype == ZK_F16) {
    for (int i = 0; i < 12; ++i)
      if (strides[i] % 8)
        return fail(ZK_ERR_UNSUPPORTED, "%s: fp16 strides must be multiples of 8", who);
    if (!aligned16(Q) || !aligned16(K) || !aligned16(V) || !aligned16(O))
      return fail(ZK_ERR_UNSUPPORTED, "%s: fp16 tensors must be 16-byte aligned", who);
    if (head_dim % 8)
      return fail(ZK_ERR_UNSUPPORTED, "%s: fp16 head_dim must be a multiple of 8 (got %lld)",
                  who, (long long)head_dim);
    // compiled widths 32 / 64 / 128; narrower head_dims are zero-padded
    if (head_dim == 32) launch_f16<32>(p, s);
    else if (head_dim == 64) launch_f16<64>(p, s);
    else if (head_dim == 128) launch_f16<128>(p, s);
    else if (head_dim < 32) launch_f16<32, true>(p, s);
    else if (head_dim < 64) launch_f16<64, true>(p, s);
    else launch_f16<128, true>(p, s);
  } else if (dtype == ZK_F32) {
    if (head_dim <= 32) launch_f32<32>(p, s);
    else if (head_dim <= 64) launch_f32<64>(p, s);
    else if (head_dim <= 96) launch_f32<96>(p, s);
    else launch_f32<128>(p, s);
  } else {
    return fail(ZK_ERR_UNSUPPORTED, "%s: dtype %d not supported", who, dtype);
  }
  return check_launch(who);
}

extern "C" int zk_flash_attn_fwd(const void *Q, const void *K, const void *V, void *O,
                                 int64_t batch, int64_t heads, int64_t seq_q, int64_t seq_k,
                                 int64_t head_dim, const int64_t *strides,
                                 const int32_t *valid_lens, float scale, int dtype,
                                 void *stream) {
  return attn_impl("zk_flash_attn_fwd", Q, K, V, O, batch, heads, seq_q, seq_k, head_dim,
                   strides, valid_lens, nullptr, nullptr, scale, dtype, stream);
}

extern "C" int zk_flash_attn_fwd_masked(const void *Q, const void *K, const void *V, void *O,
                                        int64_t batch, int64_t heads, int64_t seq_q,
                                        int64_t seq_k, int64_t head_dim, const int64_t *strides,
                                        const int32_t *valid_lens, const uint8_t *mask,
                                        const int64_t *mask_strides, float scale, int dtype,
                                        void *stream) {
  if (!mask) return fail(ZK_ERR_INVALID, "zk_flash_attn_fwd_masked: null mask");
  return attn_impl("zk_flash_attn_fwd_masked", Q, K, V, O, batch, heads, seq_q, seq_k,
                   head_dim, strides, valid_lens, mask, mask_strides, scale, dtype, stream);
}

extern "C" int zk_flash_attn_fwd_f16_io32(const void *Q, const void *K, const void *V, void *O,
                                          int64_t batch, int64_t heads, int64_t seq_q,
                                          int64_t seq_k, int64_t head_dim, const int64_t *strides,
                                          const int32_t *valid_lens, float scale, void *stream) {
  return attn_impl("zk_flash_attn_fwd_f16_io32", Q, K, V, O, batch, heads, seq_q, seq_k, head_dim,
                   strides, valid_lens, nullptr, nullptr, scale, ZK_F16, stream, true);
}
