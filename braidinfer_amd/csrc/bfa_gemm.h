// Main loop of the 16x16x32-MFMA GEMMs on 16-bit operands (linear_gemm.hip, qkv_prefill.hip):
// acc = W X^T of one BM x BN tile over a range of 64-deep K stages, both
// operands through a ring of LDS stages filled by DMA.
#pragma once

#include <hip/hip_runtime.h>

#include "bfa_device.h"

namespace bfa {

typedef __attribute__((ext_vector_type(8))) __bf16 gemm_bf16x8_t;
typedef __attribute__((ext_vector_type(8))) _Float16 gemm_f16x8_t;
typedef __attribute__((ext_vector_type(4))) float gemm_f32x4_t;

template <int DT>
__device__ __forceinline__ gemm_f32x4_t gemm_mfma(const uint4& a, const uint4& b, gemm_f32x4_t c) {
  if constexpr (DT == BFA_DTYPE_BF16)
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(gemm_bf16x8_t, a),
                                                   __builtin_bit_cast(gemm_bf16x8_t, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(gemm_f16x8_t, a),
                                                  __builtin_bit_cast(gemm_f16x8_t, b), c, 0, 0, 0);
}

// LDS tile rows are 64 elements = 8 granules of 16 bytes; granule g of row r
// sits at slot g ^ ((r / 2) & 7), so a 16-lane phase of a fragment read (one
// granule of 16 consecutive rows) hits 16 distinct bank groups.
__device__ __forceinline__ int gemm_swz(int r, int g) { return r * 8 + (g ^ ((r >> 1) & 7)); }

// s_waitcnt vmcnt(N), the other counters untouched (gfx9 encoding).
template <int N>
__device__ __forceinline__ void gemm_wait_vm() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  __builtin_amdgcn_s_waitcnt((N & 15) | (7 << 4) | (15 << 8) | ((N >> 4) << 14));
}

// Waits until at most `later` (< NS) stages of DPW copies each are in flight.
template <int DPW, int NS>
__device__ __forceinline__ void gemm_wait_stages(int later) {
  static_assert(NS >= 2 && NS <= 6 && DPW * (NS - 1) < 64, "vmcnt range");
  if (NS > 5 && later >= 5) gemm_wait_vm<(NS > 5 ? 5 : 0) * DPW>();
  else if (NS > 4 && later >= 4) gemm_wait_vm<(NS > 4 ? 4 : 0) * DPW>();
  else if (NS > 3 && later >= 3) gemm_wait_vm<(NS > 3 ? 3 : 0) * DPW>();
  else if (NS > 2 && later >= 2) gemm_wait_vm<(NS > 2 ? 2 : 0) * DPW>();
  else if (later >= 1) gemm_wait_vm<DPW>();
  else gemm_wait_vm<0>();
}

// Workgroup b of `count` -> work item: XCD x holds workgroups x, x + 8, ... and
// walks a contiguous range of items.
__device__ __forceinline__ int gemm_band(int b, int count) {
  const int x = b & 7;
  return x * (count >> 3) + min(x, count & 7) + (b >> 3);
}

// Tile t, column by column inside groups of 8 row tiles, so that the tiles one
// XCD works on at a time share operand rows and weight columns in its L2.
__device__ __forceinline__ void gemm_tile(int tiles_m, int tiles_n, int t, int& tm, int& tn) {
  const int group = t / (8 * tiles_n), first = group * 8;
  const int gs = min(tiles_m - first, 8), r = t - group * 8 * tiles_n;
  tn = r / gs;
  tm = first + (r - tn * gs);
}

// Tile of RW x CW waves, each MA 16-token by 4 16-column blocks, with NS stages
// in the LDS ring.  The weight is the MFMA's first operand: of each block a lane
// holds token lane % 16 and the four weight rows 4 (lane / 16) + v of the wave's
// 64; which matrix row the tile's weight row c stands for is the caller's
// wrow(c), so that a lane's values can be neighbours in the output.
template <int MA, int RW, int CW, int NS, int DT>
struct GemmTile {
  static constexpr int NW = RW * CW, NB = 4;
  static constexpr int BM = RW * MA * 16, BN = CW * NB * 16;
  static constexpr int STAGE = (BM + BN) * 8;              // 16-byte granules
  static constexpr int AB = BM / 8, BB = BN / 8;           // 1 KiB copies per stage
  static constexpr int ADPW = (AB + NW - 1) / NW, BDPW = (BB + NW - 1) / NW, DPW = ADPW + BDPW;
  static constexpr int LDS_U4 = NS * STAGE;
  using Acc = gemm_f32x4_t[MA][NB];

  // a: operand rows (m of them, lda apart) and w: weight rows (ldw apart), both
  // at the first K stage; byte offsets below 4 GiB; nk >= 1 stages.  `early` is
  // called once the first stages are under way.
  template <class WROW, class EARLY>
  __device__ __forceinline__ static void run(Acc& acc, uint4* lds, const uint16_t* a, const uint16_t* w, int64_t m,
                                             int64_t lda, int64_t ldw, int64_t m0, int nk, int wid, int lane,
                                             WROW wrow, EARLY early) {
    const int wr = wid / CW, wc = wid % CW;
    // Copy i of a wave moves tile rows 8 b .. 8 b + 7, b = min(i NW + wid, last)
    // (the clamp repeats a block where the waves do not divide them: the same
    // bytes to the same place); a lane fetches the granule that lands at its slot.
    uint32_t aoff[ADPW], boff[BDPW], alds[ADPW], blds[BDPW];
    const uint32_t base = lds_addr(lds);
#pragma unroll
    for (int i = 0; i < ADPW; ++i) {
      const int b = min(i * NW + wid, AB - 1), r = b * 8 + (lane >> 3);
      aoff[i] = static_cast<uint32_t>((min(m0 + r, m - 1) * lda + ((lane & 7) ^ ((r >> 1) & 7)) * 8) * 2);
      alds[i] = base + b * 1024;
    }
#pragma unroll
    for (int i = 0; i < BDPW; ++i) {
      const int b = min(i * NW + wid, BB - 1), r = b * 8 + (lane >> 3);
      boff[i] = static_cast<uint32_t>((wrow(r) * ldw + ((lane & 7) ^ ((r >> 1) & 7)) * 8) * 2);
      blds[i] = base + (AB + b) * 1024;
    }
    auto issue = [&](int st, int slot) {
      const uint32_t so = static_cast<uint32_t>(slot) * (STAGE * 16);
#pragma unroll
      for (int i = 0; i < ADPW; ++i) dma16(a + static_cast<int64_t>(st) * 64, aoff[i], alds[i] + so);
#pragma unroll
      for (int i = 0; i < BDPW; ++i) dma16(w + static_cast<int64_t>(st) * 64, boff[i], blds[i] + so);
    };
#pragma unroll
    for (int i = 0; i < MA; ++i)
#pragma unroll
      for (int j = 0; j < NB; ++j) acc[i][j] = gemm_f32x4_t{};

    const int fr = lane & 15, fg = lane >> 4;
    auto load = [&](int slot, int ks, uint4 (&fa)[MA], uint4 (&fb)[NB]) {
      const uint4* st = lds + slot * STAGE;
#pragma unroll
      for (int j = 0; j < NB; ++j) fb[j] = st[BM * 8 + gemm_swz(wc * 64 + j * 16 + fr, ks * 4 + fg)];
#pragma unroll
      for (int i = 0; i < MA; ++i) fa[i] = st[gemm_swz(wr * MA * 16 + i * 16 + fr, ks * 4 + fg)];
    };
    auto mul = [&](const uint4 (&fa)[MA], const uint4 (&fb)[NB]) {
#pragma unroll
      for (int i = 0; i < MA; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j) acc[i][j] = gemm_mfma<DT>(fb[j], fa[i], acc[i][j]);
    };

    // A stage's second half is read while its first half is multiplied; then the
    // wave waits for the next stage's copies (vmcnt counts this wave's, in order,
    // so the later stages stay in flight), and a barrier publishes them and
    // proves that every wave holds the rest of this stage in registers, so its
    // buffer takes stage kt + NS at once; the next stage's first half is read
    // under the second half's MFMAs.
#pragma unroll
    for (int st = 0; st < NS; ++st)
      if (st < nk) issue(st, st);
    early();
    gemm_wait_stages<DPW, NS>(min(NS - 1, nk - 1));
    __syncthreads();
    uint4 fa0[MA], fb0[NB], fa1[MA], fb1[NB];
    load(0, 0, fa0, fb0);
    int kt = 0, slot = 0;
    for (; kt + 1 < nk; ++kt) {
      const int next = slot + 1 == NS ? 0 : slot + 1;
      load(slot, 1, fa1, fb1);
      mul(fa0, fb0);
      gemm_wait_stages<DPW, NS>(min(NS - 2, nk - 2 - kt));
      __syncthreads();
      if (kt + NS < nk) issue(kt + NS, slot);
      load(next, 0, fa0, fb0);
      mul(fa1, fb1);
      slot = next;
    }
    load(slot, 1, fa1, fb1);
    mul(fa0, fb0);
    mul(fa1, fb1);
  }
};

// Split-K partial tiles, register order, 1 KiB per store:
// [split tile][split][wave][token block][column block][lane].  Token blocks
// past the last token are not stored.
template <int MA, int NB>
__device__ __forceinline__ void gemm_store_part(float* part, int64_t unit, int nw, int wid, int lane, int blocks,
                                                const gemm_f32x4_t (&acc)[MA][NB]) {
  gemm_f32x4_t* p = reinterpret_cast<gemm_f32x4_t*>(part) + (unit * nw + wid) * (MA * NB * 64) + lane;
#pragma unroll
  for (int i = 0; i < MA; ++i) {
    if (i >= blocks) break;
#pragma unroll
    for (int j = 0; j < NB; ++j) p[(i * NB + j) * 64] = acc[i][j];
  }
}

// The sum over splits, in split order, of one wave's 16-token x 64-column block:
// p its first partial, `stride` apart; four splits' loads are out at a time.
__device__ __forceinline__ void gemm_sum_part(const gemm_f32x4_t* p, int64_t stride, int splits, gemm_f32x4_t (&acc)[4]) {
#pragma unroll
  for (int j = 0; j < 4; ++j) acc[j] = p[j * 64];
  int s = 1;
  for (; s + 4 <= splits; s += 4) {
    gemm_f32x4_t t[4][4];
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int j = 0; j < 4; ++j) t[u][j] = p[(s + u) * stride + j * 64];
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[j] += t[u][j];
  }
  for (; s < splits; ++s)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[j] += p[s * stride + j * 64];
}

}  // namespace bfa
