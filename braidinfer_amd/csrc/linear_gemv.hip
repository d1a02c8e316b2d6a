// Linear layers of up to 16 tokens (64 for a small weight) in one launch, where
// that is faster than split-K (linear_gemv_ok):
// y = x W^T with the layer's epilogue (bias, residual, or SiLU(gate) * up), 16-bit
// operands, fp32 sums.
//
// A weight stream: bound by HBM where the weight is large, by the latency of one
// launch where it is small.  A workgroup owns 16 or 32 weight rows for the whole
// of K, so there are no partial sums to write, read back and reduce in a second
// launch; its waves take the 64-deep K steps in turn (the workgroup reads NWV x
// 128 contiguous bytes of each row at a time) straight into MFMA fragments: in a
// step lane l holds the 32 bytes at 32 (l / 16) of row, or token, l % 16, so two
// loads cover whole 128-byte lines and both operands agree on which k a slot is.
// The waves' sums meet in the LDS, in wave order.  Loads past a wave's last step
// are skipped, not clamped: the repeated ones cost as much as new ones (gate_up
// at one token 50.9 us with them).
//
// Against the split-K kernels and their reduction (graph-replayed, weights from
// HBM, one token / 16 tokens): Llama-3-8B gate_up 49.9 -> 41.3 us (5.7 TB/s) /
// 55.5 -> 48.7, down 30.9 -> 24.9 / 33.8 -> 31.9, o_proj 11.7 -> 9.8 / 13.3 ->
// 12.0; TinyLlama 15.6 -> 12.1, 12.7 -> 10.2, 8.4 -> 6.1; Qwen3-0.6B 8.9 -> 5.5,
// 12.3 -> 6.6, 9.5 -> 5.7 us.
#include "bfa_gemm.h"
#include "bfa_host.h"
#include "bfa_linear.h"
#include "bfa_qkv.h"

namespace bfa {

__device__ __forceinline__ uint4 gemv_u4(const u32x4_t& v) { return make_uint4(v.x, v.y, v.z, v.w); }

// NR blocks of 16 weight rows per workgroup, MT of 16 tokens.  Plain: consecutive
// columns.  SwiGLU: NR = 1 8 gate rows and their 8 up rows, NR = 2 16 gate rows
// and 16 up.
template <int DT, int NWV, int NR, int MT, bool SWIGLU>
__global__ __launch_bounds__(NWV * 64) void linear_gemv_kernel(LinArgs q) {
  // K steps per batch; the next batch's loads (16, 18, 16, 20 or 24 per lane)
  // are in flight under a batch's products
  constexpr int U = NR + MT == 2 ? 4 : NR + MT == 3 ? 3 : 2;
  __shared__ gemm_f32x4_t red[NR * MT][NWV][64];
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, g = lane >> 4;
  const int64_t n0 = static_cast<int64_t>(blockIdx.x) * (SWIGLU ? 8 * NR : 16 * NR);
  const u32x4_t* wp[NR];
  const u32x4_t* xp[MT];
#pragma unroll
  for (int b = 0; b < NR; ++b) {
    int64_t row;
    if (SWIGLU && NR == 1) row = min(n0 + (r & 7), q.n - 1) + (r >= 8 ? q.n : 0);
    else if (SWIGLU) row = min(n0 + r, q.n - 1) + (b ? q.n : 0);
    else row = min(n0 + 16 * b + r, q.n - 1);
    wp[b] = reinterpret_cast<const u32x4_t*>(q.w + row * q.ldw + g * 16 + wid * 64);
  }
#pragma unroll
  for (int i = 0; i < MT; ++i)
    xp[i] = reinterpret_cast<const u32x4_t*>(q.a + min<int64_t>(16 * i + r, q.m - 1) * q.lda + g * 16 + wid * 64);
  struct Frag {
    u32x4_t w[NR][2], x[MT][2];
  };
  auto load = [&](int s) {  // this wave's s-th step
    Frag f;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
      for (int b = 0; b < NR; ++b) f.w[b][h] = wp[b][static_cast<int64_t>(s) * (8 * NWV) + h];
#pragma unroll
      for (int i = 0; i < MT; ++i) f.x[i][h] = xp[i][static_cast<int64_t>(s) * (8 * NWV) + h];
    }
    return f;
  };
  constexpr int AH = MT > 1 ? 1 : 2;  // accumulators per block: two chains where one block is too few
  gemm_f32x4_t acc[NR][MT][AH] = {};
  auto mul = [&](const Frag& f) {
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int b = 0; b < NR; ++b)
#pragma unroll
        for (int i = 0; i < MT; ++i)
          acc[b][i][h % AH] = gemm_mfma<DT>(gemv_u4(f.w[b][h]), gemv_u4(f.x[i][h]), acc[b][i][h % AH]);
  };

  // The epilogue's blocks (weight block b, token block i) go to the waves in
  // turn: token 16 i + r, columns c0 .. c0 + 3.  The bias and residual of a
  // wave's first block are requested ahead of the stream (SwiGLU has neither).
  constexpr int EB = SWIGLU ? MT : NR * MT;
  struct Side {
    uint32_t bw[4], rw[4];
  };
  auto side = [&](int e) {
    Side d = {};
    const int64_t t = min<int64_t>(16 * (e % MT) + r, q.m - 1);
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int64_t c = min(n0 + 16 * (e / MT) + 4 * g + v, q.n - 1);
      if (q.bias) d.bw[v] = ld_word(q.bias, q.bias_dt, c);
      if (q.res) d.rw[v] = ld_word(q.res, q.res_dt, t * q.ldr + c);
    }
    return d;
  };
  Side sd = {};
  if (!SWIGLU && wid < EB) sd = side(wid);

  const int steps = wid < q.kt ? (q.kt - 1 - wid) / NWV + 1 : 0;  // of this wave
  const int full = steps / U * U, rest = steps - full;
  Frag f[2][U], tail[U - 1];
  if (full > 0) {
#pragma unroll
    for (int u = 0; u < U; ++u) f[0][u] = load(u);
  }
#pragma unroll
  for (int u = 0; u < U - 1; ++u)
    if (u < rest) tail[u] = load(full + u);
  int s = 0;
  for (; s + 2 * U <= full; s += 2 * U) {
#pragma unroll
    for (int u = 0; u < U; ++u) f[1][u] = load(s + U + u);
#pragma unroll
    for (int u = 0; u < U; ++u) mul(f[0][u]);
    if (s + 2 * U < full) {
#pragma unroll
      for (int u = 0; u < U; ++u) f[0][u] = load(s + 2 * U + u);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) mul(f[1][u]);
  }
  if (s < full) {
#pragma unroll
    for (int u = 0; u < U; ++u) mul(f[0][u]);
  }
#pragma unroll
  for (int u = 0; u < U - 1; ++u)
    if (u < rest) mul(tail[u]);
#pragma unroll
  for (int b = 0; b < NR; ++b)
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      gemm_f32x4_t t = acc[b][i][0];
      if constexpr (AH == 2) t += acc[b][i][1];
      red[b * MT + i][wid][lane] = t;
    }
  __syncthreads();
  auto sum = [&](int e) {
    gemm_f32x4_t t = red[e][0][lane];
#pragma unroll
    for (int w = 1; w < NWV; ++w) t += red[e][w][lane];
    return t;
  };
  for (int e = wid; e < EB; e += NWV) {
    const int t = 16 * (e % MT) + r;
    const int64_t c0 = n0 + 16 * (SWIGLU ? 0 : e / MT) + 4 * g;
    if constexpr (SWIGLU) {
      const gemm_f32x4_t gate = sum(e);
      gemm_f32x4_t up;
      if constexpr (NR == 1) {  // gate rows 0-7 are the lanes below 32, up rows 8-15 those above
#pragma unroll
        for (int v = 0; v < 4; ++v) up[v] = __shfl(gate[v], (lane + 32) & 63);
      } else {
        up = sum(MT + e);
      }
      if ((NR == 1 && lane >= 32) || t >= q.m) continue;
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const float y = round_to(silu_fast(round_to(gate[v], q.proj_dt)), q.proj_dt) * round_to(up[v], q.proj_dt);
        if (c0 + v < q.n) store_any(q.out, q.out_dt, static_cast<int64_t>(t) * q.ldo + c0 + v, y);
      }
    } else {
      if (e != wid) sd = side(e);
      const gemm_f32x4_t p = sum(e);
      if (t >= q.m) continue;
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int64_t c = min(c0 + v, q.n - 1);
        float y = p[v];
        if (q.bias) y = y + word_value(sd.bw[v], q.bias_dt, q.bias, c);
        y = round_to(y, q.proj_dt);
        if (q.res) y = y + word_value(sd.rw[v], q.res_dt, q.res, t * q.ldr + c);
        y = round_to(y, q.mid_dt);
        if (c0 + v < q.n) store_any(q.out, q.out_dt, static_cast<int64_t>(t) * q.ldo + c0 + v, y);
      }
    }
  }
}

namespace {

template <int DT, int NWV, int NR, int MT, bool SWIGLU>
void launch_form(const LinArgs& q, hipStream_t st) {
  const dim3 grid(static_cast<unsigned>(cdiv(q.n, SWIGLU ? 8 * NR : 16 * NR)));
  hipLaunchKernelGGL((linear_gemv_kernel<DT, NWV, NR, MT, SWIGLU>), grid, dim3(NWV * 64), 0, st, q);
}

// Waves and weight blocks of a workgroup.  Plain: one weight block, so that as many
// CUs as there are blocks of columns stream (two blocks: Llama-3-8B down_proj at one
// token 24.9 -> 32.6 us), in 4 waves, 8 for a long K and up to 16 tokens.  SwiGLU
// has twice the rows: two blocks, which halve the token reads per weight byte
// (gate_up at 16 tokens 60.9 -> 48.7 us), but one for up to 4 tokens of a weight of
// 32 MiB and more (41.3 against 42.7 us).
struct GemvForm {
  int nwv, nr;
};
GemvForm gemv_form(int64_t m, int64_t n, int64_t k, bool swiglu) {
  if (swiglu) return {4, m <= 4 && n * k * 4 >= (int64_t(32) << 20) ? 1 : 2};
  return {m <= 16 && k >= 128 * 64 ? 8 : 4, 1};
}

template <int DT>
void launch_dt(const LinArgs& q, hipStream_t st) {
  const int mt = static_cast<int>(cdiv(q.m, 16));
  const GemvForm f = gemv_form(q.m, q.n, q.k, q.swiglu != 0);
  if (q.swiglu) {
    if (f.nr == 1) return launch_form<DT, 4, 1, 1, true>(q, st);
    if (mt == 1) return launch_form<DT, 4, 2, 1, true>(q, st);
    if (mt == 2) return launch_form<DT, 4, 2, 2, true>(q, st);
    if (mt == 3) return launch_form<DT, 4, 2, 3, true>(q, st);
    return launch_form<DT, 4, 2, 4, true>(q, st);
  }
  if (f.nwv == 8) return launch_form<DT, 8, 1, 1, false>(q, st);
  if (mt == 1) return launch_form<DT, 4, 1, 1, false>(q, st);
  if (mt == 2) return launch_form<DT, 4, 1, 2, false>(q, st);
  if (mt == 3) return launch_form<DT, 4, 1, 3, false>(q, st);
  return launch_form<DT, 4, 1, 4, false>(q, st);
}

}  // namespace

// Neither kernel is always ahead: a workgroup walks the whole of K, so a long K on
// few columns leaves most CUs idle (1 token, K 65536, 128 columns 74 against 44 us
// split; 64 tokens, K 8192, 1024 columns 39 against 17), and from some thousand
// workgroups their start costs more than their stream (K 1024, 128256 columns 69
// against 47 us).  So both times are estimated, in us, from what was measured of
// either on 2753 shapes (1 to 64 tokens, K 64 to 65536, 16 to 128256 columns):
//   here   3 + the longer of one workgroup's K steps and a CU's share of all of
//          them; a step takes 0.31 at one token and 0.0125 more for each other
//   split  5.4 (6 from 17 tokens) + 0.14 (0.083) per split that the reduction
//          reads, 1.7 times that with SwiGLU, + the weight at 5.6 (6.9) TB/s, the
//          partials' round trip and the outputs
// each within 10 % for 8 in 10 shapes.  On those shapes the choice is within 3 % of
// the faster one or ahead of split-K in all but one in ninety, 20 % behind at worst
// (always taking this kernel up to 16 tokens, and up to 64 for 16 MiB, was behind
// in one of three, by up to 8 times).
// From 17 tokens only weights of up to 16 MiB are weighed.  Overrides:
// BFA_TUNE_LINEAR_GEMV, and any of the split-K kernels' own keeps them.
bool linear_gemv_ok(int64_t m, int64_t wrows, int64_t k, bool swiglu, int64_t splits) {
  if (m > 64 || k % 64 != 0) return false;
  const int o = tuning(BFA_TUNE_LINEAR_GEMV);
  if (o >= 0) return o != 0;
  if (tuning(BFA_TUNE_DECODE_KS) >= 0 || tuning(BFA_TUNE_DECODE_WG) >= 0 || tuning(BFA_TUNE_DECODE_SPLITS) >= 0)
    return false;
  const double mb = static_cast<double>(wrows) * k * 2e-6, outs = static_cast<double>(m) * wrows * 1e-6;
  if (m > 16 && wrows * k * 2 > (int64_t(16) << 20)) return false;
  const int64_t n = swiglu ? wrows / 2 : wrows;
  const GemvForm f = gemv_form(m, n, k, swiglu);
  const double steps = static_cast<double>(cdiv(k / 64, f.nwv));
  const int64_t wgs = cdiv(n, swiglu ? 8 * f.nr : 16);
  const double cu = wgs > 256 ? static_cast<double>(cdiv(wgs, 256)) : static_cast<double>(wgs) / 256;  // per CU, at most
  double step = 0.31 + 0.0125 * static_cast<double>(m - 1), busy = step;  // alone on a CU, with others
  if (f.nr == 2) busy = step += 0.2;
  if (f.nwv == 8) busy += 0.43, step *= 1.8;
  const double here = 3 + std::max(steps * step, cu * ((m > 48 ? 1.7 : 0.7) + steps * busy));
  const double sp = static_cast<double>(splits) * (swiglu ? 1.7 : 1);
  const double split = m <= 16 ? 5.4 + 0.14 * sp + 0.18 * mb + 2.5 * outs : 6.0 + 0.083 * sp + 0.145 * mb + outs;
  return here <= 0.965 * (split + 2.5 * static_cast<double>(splits) * outs);
}

void launch_linear_gemv(LinArgs q, int dt, hipStream_t st) {
  q.kt = static_cast<int>(q.k / 64);
  if (dt == BFA_DTYPE_BF16) launch_dt<BFA_DTYPE_BF16>(q, st);
  else launch_dt<BFA_DTYPE_F16>(q, st);
}

}  // namespace bfa
