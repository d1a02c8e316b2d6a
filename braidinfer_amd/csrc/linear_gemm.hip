// Linear-layer GEMM for 65 and more tokens: y = x W^T with the layer's own
// epilogue (bias, residual, or SiLU(gate) * up), 16-bit operands, fp32 sums.
//
// What bounds it: from about a thousand tokens the matrix cores (under their
// load the chip is power limited), below that the weight stream and the number
// of CUs that have a tile.  A workgroup of RW x CW waves owns a BM x BN tile
// and runs the ring of bfa_gemm.h.  The tile sizes (bfa_gemm_plan.h) differ in how well they fill
// the 256 CUs, which decides more than the loop does (Llama-3-8B, 300 tokens:
// gate_up on 128 x 256 tiles is 336 tiles, two rounds of which the second is
// nearly empty; on 160 x 256 it is one round of 224).  What whole rounds of
// tiles do not fill is split over K: the last tiles go to several workgroups
// each, whose fp32 partial tiles linear_reduce_kernel sums, in split order, into
// the same epilogue.
//
// Measured against the projection GEMM's tiles with linear epilogues, which
// these replace (Llama-3-8B, weights from HBM, same box): gate_up+SiLU*mul 94 ->
// 56 us at 100 tokens, 158 -> 76 us at 300 (927 TFLOP/s; a plain library GEMM
// 76 us), 1235 -> 1119 us at 6000; down_proj+residual 165 -> 35 us, 153 -> 52 us
// and 728 -> 572 us (1232 TFLOP/s).
#include "bfa_gemm.h"
#include "bfa_host.h"
#include "bfa_linear.h"
#include "bfa_qkv.h"

namespace bfa {

// Output columns of the wave's 64 weight rows: row 16 j + 4 g + v feeds
//   plain    column 16 g + 4 j + v                          (a lane: 16 consecutive)
//   SwiGLU   gate (j < 2) or up column 8 g + 4 (j % 2) + v  (a lane: 8 of each)
// so that a lane's values are neighbours in one token's output row and go out in
// 16-byte stores straight from the accumulators.
template <bool SWIGLU>
__device__ __forceinline__ int64_t lin_weight_row(const LinArgs& q, int64_t n0, int c) {
  const int w = c >> 6, j = (c >> 4) & 3, g = (c >> 2) & 3, v = c & 3;
  if constexpr (SWIGLU) {
    const int64_t o = min(n0 + w * 32 + g * 8 + (j & 1) * 4 + v, q.n - 1);
    return j < 2 ? o : q.n + o;
  } else {
    return min(n0 + w * 64 + g * 16 + j * 4 + v, q.n - 1);
  }
}

// Eight neighbouring outputs (columns c .. c + 7) of one token, where proj_dt,
// out_dt and res_dt are DT, mid_dt DT or fp32, the rows vec and n a multiple of 8.
template <int DT, bool SWIGLU>
__device__ __forceinline__ void lin_out8(const LinArgs& q, int64_t row, int64_t c, const float (&a)[8],
                                         const float (&u)[8], const uint4& res) {
  using E = Elem<DT>;
  if (c >= q.n) return;
  const uint32_t rw[4] = {res.x, res.y, res.z, res.w};
  float y[8];
#pragma unroll
  for (int t = 0; t < 8; ++t) {
    if constexpr (SWIGLU) {
      y[t] = E::round(silu_fast(E::round(a[t]))) * E::round(u[t]);
    } else {
      float v = a[t];
      if (q.bias) v = v + load_any(q.bias, q.bias_dt, c + t);
      v = E::round(v);
      if (q.res) v = v + E::to_f32(static_cast<uint16_t>((t & 1) ? rw[t >> 1] >> 16 : rw[t >> 1] & 0xffffu));
      y[t] = v;
    }
  }
  store8<DT>(static_cast<uint16_t*>(q.out) + row * q.ldo + c, y);
}

// One token's 16 projection values of a lane; c0 its first output column.
template <int DT, bool SWIGLU>
__device__ __forceinline__ void lin_finish(const LinArgs& q, int64_t row, int64_t c0, const gemm_f32x4_t (&acc)[4],
                                           const uint4 (&res)[2]) {
  const float lo[8] = {acc[0][0], acc[0][1], acc[0][2], acc[0][3], acc[1][0], acc[1][1], acc[1][2], acc[1][3]};
  const float hi[8] = {acc[2][0], acc[2][1], acc[2][2], acc[2][3], acc[3][0], acc[3][1], acc[3][2], acc[3][3]};
  if constexpr (SWIGLU) {
    lin_out8<DT, true>(q, row, c0, lo, hi, res[0]);
  } else {
    lin_out8<DT, false>(q, row, c0, lo, lo, res[0]);
    lin_out8<DT, false>(q, row, c0 + 8, hi, hi, res[1]);
  }
}

// The general form (any dtypes, any n and row stride) passes a wave's blocks
// through the LDS, a few at a time, and walks their rows in a loop.  In registers
// its code, once per block, outgrew the unroller: the accumulators went to scratch,
// in the main loop too (3000 tokens, K 2048, n = 8004 951 us, against 147 on the
// projection GEMM's tiles; 120 like this).  A block is 16 tokens of 16 granules of
// 4 values, granule G of token r at G ^ r (a lane writes 4 granules of one token):
// plain, the wave's 64 columns in order; SwiGLU, its 32 gate columns, then its 32
// up columns.
template <bool SWIGLU>
__device__ __forceinline__ void lin_stage(gemm_f32x4_t* block, int lane, const gemm_f32x4_t (&acc)[4]) {
  const int r = lane & 15, g = lane >> 4;
#pragma unroll
  for (int j = 0; j < 4; ++j)
    block[r * 16 + ((SWIGLU ? (j >> 1) * 8 + 2 * g + (j & 1) : 4 * g + j) ^ r)] = acc[j];
}

// One output from its sum (SwiGLU: and its up sum), bias and residual.
template <bool SWIGLU>
__device__ __forceinline__ float lin_value(const LinArgs& q, float a, float u, float bias, float res) {
  if constexpr (SWIGLU) {
    return round_to(silu_fast(round_to(a, q.proj_dt)), q.proj_dt) * round_to(u, q.proj_dt);
  } else {
    if (q.bias) a = a + bias;
    return round_to(round_to(a, q.proj_dt) + res, q.mid_dt);
  }
}

// `rows` staged tokens of a wave, the first one row0, its first output column c0,
// where output rows take 4-byte accesses of 16-bit elements (W = 2 columns a lane:
// gate_up of 3000 tokens, K 256, 8004 columns 82 -> 69 us) or none (W = 1): the
// wave's accesses lie next to each other.  A lane keeps its
// columns, so it reads the bias once; the residual of the next rows is on its way
// during these rows' work.
template <bool SWIGLU, int W>
__device__ __forceinline__ void lin_rows_narrow(const LinArgs& q, int64_t row0, int64_t c0,
                                                const gemm_f32x4_t* staged, int rows, int lane) {
  constexpr int LPR = (SWIGLU ? 32 : 64) / W, STEP = 64 / LPR, U = 8 / W;  // lanes per row; U steps at a time
  const float* f = reinterpret_cast<const float*>(staged);
  const int col = lane % LPR * W;
  const int64_t c = c0 + col;
  if (c >= q.n) return;
  const bool whole = c + W <= q.n;
  float bias[W] = {};
  if (!SWIGLU && q.bias) {
#pragma unroll
    for (int w = 0; w < W; ++w) bias[w] = load_any(q.bias, q.bias_dt, min(c + w, q.n - 1));
  }
  struct Res {
    uint32_t v[U][W];
  };
  auto load_res = [&](int t) {
    Res d{};
    if (!SWIGLU && q.res) {
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int w = 0; w < W; ++w)
          d.v[u][w] = ld_word(q.res, q.res_dt, (row0 + min(t + u * STEP, rows - 1)) * q.ldr + min(c + w, q.n - 1));
    }
    return d;
  };
  Res cur = load_res(lane / LPR);
  for (int t0 = lane / LPR; t0 < rows; t0 += U * STEP) {
    const Res next = load_res(t0 + U * STEP);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int t = t0 + u * STEP;
      if (t >= rows) break;
      const int r = t & 15, o = t * 64 + (col & 3);
      const float* a = f + o + 4 * ((col >> 2) ^ r);
      const float* up = SWIGLU ? f + o + 4 * ((8 + (col >> 2)) ^ r) : a;
      float y[W];
#pragma unroll
      for (int w = 0; w < W; ++w) {
        const int64_t i = (row0 + t) * q.ldr + min(c + w, q.n - 1);
        const float res = !SWIGLU && q.res ? word_value(cur.v[u][w], q.res_dt, q.res, i) : 0.f;
        y[w] = lin_value<SWIGLU>(q, a[w], up[w], bias[w], res);
      }
      const int64_t i = (row0 + t) * q.ldo + c;
      if constexpr (W == 2) {
        if (whole) {
          const uint32_t b = pack_bf16x2(y[0], y[1]);
          const uint32_t h = Elem<BFA_DTYPE_F16>::from_f32(y[0]) |
                             (static_cast<uint32_t>(Elem<BFA_DTYPE_F16>::from_f32(y[1])) << 16);
          *reinterpret_cast<uint32_t*>(static_cast<uint16_t*>(q.out) + i) = q.out_dt == BFA_DTYPE_BF16 ? b : h;
          continue;
        }
      }
      store_any(q.out, q.out_dt, i, y[0]);
    }
    cur = next;
  }
}

// Rows that take 16-byte accesses: eight columns a lane; else lin_rows_narrow.
template <bool SWIGLU>
__device__ __forceinline__ void lin_rows(const LinArgs& q, int64_t row0, int64_t c0, const gemm_f32x4_t* staged,
                                         int rows, int lane) {
  constexpr int COLS = SWIGLU ? 32 : 64;
  rows = static_cast<int>(min<int64_t>(rows, q.m - row0));
  if (rows <= 0) return;
  if (q.vec) {
    constexpr int G8 = COLS / 8, STEP = 64 / G8;
    const int g = 2 * (lane % G8);
    const int64_t c = c0 + 4 * g;
    if (c >= q.n) return;
    const bool whole = c + 8 <= q.n;
    float bias[8] = {};
    if (!SWIGLU && q.bias) {
#pragma unroll
      for (int v = 0; v < 8; ++v) bias[v] = load_any(q.bias, q.bias_dt, min(c + v, q.n - 1));
    }
    struct Res {
      uint4 lo, hi;  // 16-bit: lo alone
    };
    auto load_res = [&](int t) {
      Res d{};
      if (!SWIGLU && q.res && whole) {
        const char* p = static_cast<const char*>(q.res);
        const int64_t e = (row0 + min(t, rows - 1)) * q.ldr + c;
        d.lo = *reinterpret_cast<const uint4*>(p + e * (q.res_dt == BFA_DTYPE_F32 ? 4 : 2));
        if (q.res_dt == BFA_DTYPE_F32) d.hi = *reinterpret_cast<const uint4*>(p + e * 4 + 16);
      }
      return d;
    };
    Res cur = load_res(lane / G8);
    for (int t = lane / G8; t < rows; t += STEP) {
      const Res next = load_res(t + STEP);
      const int r = t & 15;
      const int64_t row = row0 + t;
      const gemm_f32x4_t* s = staged + t * 16;
      const gemm_f32x4_t a0 = s[g ^ r], a1 = s[(g + 1) ^ r];
      const gemm_f32x4_t u0 = SWIGLU ? s[(8 + g) ^ r] : a0, u1 = SWIGLU ? s[(9 + g) ^ r] : a1;
      const uint32_t w[8] = {cur.lo.x, cur.lo.y, cur.lo.z, cur.lo.w, cur.hi.x, cur.hi.y, cur.hi.z, cur.hi.w};
      float y[8];
#pragma unroll
      for (int v = 0; v < 8; ++v) {
        float res = 0.f;
        if (!SWIGLU && q.res) {
          const uint32_t h = (v & 1) ? w[v >> 1] >> 16 : w[v >> 1] & 0xffffu;
          if (!whole) res = load_any(q.res, q.res_dt, row * q.ldr + min(c + v, q.n - 1));
          else if (q.res_dt == BFA_DTYPE_F32) res = __uint_as_float(w[v]);
          else res = q.res_dt == BFA_DTYPE_BF16 ? bf16_bits_to_f32(h) : f16_bits_to_f32(h);
        }
        y[v] = lin_value<SWIGLU>(q, v < 4 ? a0[v & 3] : a1[v & 3], v < 4 ? u0[v & 3] : u1[v & 3], bias[v], res);
      }
      cur = next;
      if (whole) {
        if (q.out_dt == BFA_DTYPE_BF16) store8<BFA_DTYPE_BF16>(static_cast<uint16_t*>(q.out) + row * q.ldo + c, y);
        else if (q.out_dt == BFA_DTYPE_F16) store8<BFA_DTYPE_F16>(static_cast<uint16_t*>(q.out) + row * q.ldo + c, y);
        else store8<BFA_DTYPE_F32>(static_cast<float*>(q.out) + row * q.ldo + c, y);
      } else {
#pragma unroll
        for (int v = 0; v < 8; ++v)
          if (c + v < q.n) store_any(q.out, q.out_dt, row * q.ldo + c + v, y[v]);
      }
    }
    return;
  }
  if (q.pairs) lin_rows_narrow<SWIGLU, 2>(q, row0, c0, staged, rows, lane);
  else lin_rows_narrow<SWIGLU, 1>(q, row0, c0, staged, rows, lane);
}

// The lane's residual elements, ahead of their use (columns past n are clamped;
// their results are not stored).
template <bool SWIGLU>
__device__ __forceinline__ void lin_residual(const LinArgs& q, int64_t row, int64_t c0, uint4 (&res)[2]) {
  res[0] = res[1] = make_uint4(0, 0, 0, 0);
  if constexpr (!SWIGLU) {
    if (q.res) {
#pragma unroll
      for (int h = 0; h < 2; ++h)
        res[h] = *reinterpret_cast<const uint4*>(static_cast<const uint16_t*>(q.res) + row * q.ldr +
                                                 min(c0 + 8 * h, q.n - 8));
    }
  }
}

// The first q.full workgroups take whole tiles; each of the tiles after those
// goes to q.splits workgroups, one K range each (q.full is a multiple of 8 or
// covers every tile, so both parts keep their XCDs).
template <int MA, int RW, int CW, int NS, int DT, bool SAME, bool SWIGLU>
__global__ __launch_bounds__(RW * CW * 64, 2) void linear_gemm_kernel(LinArgs q) {
  using T = GemmTile<MA, RW, CW, NS, DT>;
  __shared__ uint4 lds[T::LDS_U4];
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wr = wid / CW, wc = wid % CW;
  const int b = blockIdx.x;
  const bool part = b >= q.full;
  const int rest = q.tiles_m * q.tiles_n - q.full;
  const int u = part ? gemm_band(b - q.full, rest * q.splits) : gemm_band(b, q.full);
  const int split = part ? u / rest : 0, tile = part ? q.full + (u - split * rest) : u, ns = part ? q.splits : 1;
  int tm, tn;
  gemm_tile(q.tiles_m, q.tiles_n, tile, tm, tn);
  const int64_t m0 = static_cast<int64_t>(tm) * T::BM;
  const int64_t n0 = static_cast<int64_t>(tn) * (SWIGLU ? T::BN / 2 : T::BN);
  const int k0 = static_cast<int>(static_cast<int64_t>(q.kt) * split / ns);
  const int nk = static_cast<int>(static_cast<int64_t>(q.kt) * (split + 1) / ns) - k0;
  typename T::Acc acc;
  T::run(acc, lds, q.a + static_cast<int64_t>(k0) * 64, q.w + static_cast<int64_t>(k0) * 64, q.m, q.lda, q.ldw, m0, nk,
         wid, lane, [&](int c) { return lin_weight_row<SWIGLU>(q, n0, c); }, [] {});

  const int64_t wm0 = m0 + wr * MA * 16;
  if (part) {
    gemm_store_part<MA, 4>(q.part, static_cast<int64_t>(tile - q.full) * q.splits + split, T::NW, wid, lane,
                           static_cast<int>(cdiv(q.m - wm0, 16)), acc);
    return;
  }
  if constexpr (!SAME) {
    constexpr int HB = T::LDS_U4 / (T::NW * 256) < MA ? T::LDS_U4 / (T::NW * 256) : MA;  // blocks of 4 KiB at a time
    static_assert(HB >= 1, "a block per wave takes the ring's place");
    gemm_f32x4_t* staged = reinterpret_cast<gemm_f32x4_t*>(lds) + wid * (HB * 256);
    __syncthreads();  // the ring's last reads are done
#pragma unroll
    for (int h = 0; h < MA; h += HB) {
#pragma unroll
      for (int i = 0; i < HB && h + i < MA; ++i) lin_stage<SWIGLU>(staged + i * 256, lane, acc[h + i]);
      asm volatile("" ::: "memory");  // the wave's own LDS writes precede its reads, and these the next writes
      lin_rows<SWIGLU>(q, wm0 + h * 16, n0 + wc * (SWIGLU ? 32 : 64), staged, min(HB, MA - h) * 16, lane);
      asm volatile("" ::: "memory");
    }
    return;
  }
  const int64_t c0 = n0 + (SWIGLU ? wc * 32 + (lane >> 4) * 8 : wc * 64 + (lane >> 4) * 16);
  const int64_t r0 = wm0 + (lane & 15);
  // the residual rows of half the blocks are requested together (of all of
  // them, the 256 x 256 tile spills 16 registers)
  constexpr int H = (MA + 1) / 2;
#pragma unroll
  for (int h = 0; h < MA; h += H) {
    uint4 res[H][2];
#pragma unroll
    for (int i = 0; i < H; ++i) lin_residual<SWIGLU>(q, min(r0 + (h + i) * 16, q.m - 1), c0, res[i]);
#pragma unroll
    for (int i = 0; i < H && h + i < MA; ++i)
      if (r0 + (h + i) * 16 < q.m) lin_finish<DT, SWIGLU>(q, r0 + (h + i) * 16, c0, acc[h + i], res[i]);
  }
}

// One wave per 16-token x 64-column block of a split tile.
template <int DT, bool SAME, bool SWIGLU>
__global__ __launch_bounds__(256) void linear_reduce_kernel(LinArgs q, int ma, int rw, int cw, int items) {
  const int item = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (item >= items) return;
  const int lane = threadIdx.x & 63;
  const int per = rw * cw * ma, rest = item / per, in = item - rest * per;
  const int w = in / ma, i = in - w * ma, wr = w / cw, wc = w - wr * cw;
  int tm, tn;
  gemm_tile(q.tiles_m, q.tiles_n, q.full + rest, tm, tn);
  const int64_t row0 = (static_cast<int64_t>(tm) * rw * ma + wr * ma + i) * 16, row = row0 + (lane & 15);
  if (row0 >= q.m) return;  // no partials there
  const int64_t w0 = (static_cast<int64_t>(tn) * cw + wc) * (SWIGLU ? 32 : 64);  // the wave's first output column
  const int64_t c0 = w0 + (lane >> 4) * (SWIGLU ? 8 : 16);
  uint4 res[2];
  if constexpr (SAME) lin_residual<SWIGLU>(q, min(row, q.m - 1), c0, res);
  gemm_f32x4_t acc[4];
  const int64_t stride = static_cast<int64_t>(per) * 256;
  gemm_sum_part(reinterpret_cast<const gemm_f32x4_t*>(q.part) + (static_cast<int64_t>(rest) * q.splits * per + in) * 256 + lane,
                stride, q.splits, acc);
  if constexpr (SAME) {
    if (row < q.m) lin_finish<DT, SWIGLU>(q, row, c0, acc, res);
  } else {
    __shared__ gemm_f32x4_t blocks[4][256];
    gemm_f32x4_t* staged = blocks[threadIdx.x >> 6];
    lin_stage<SWIGLU>(staged, lane, acc);
    asm volatile("" ::: "memory");  // the wave's own LDS writes precede its reads
    lin_rows<SWIGLU>(q, row0, w0, staged, 16, lane);
  }
}

// ------------------------------------------------------------------- host
namespace {

template <int DT, bool SAME>
void launch_form(const GemmPlan& p, const LinArgs& q, hipStream_t st) {
  const int rest = q.tiles_m * q.tiles_n - q.full;
  const dim3 grid(static_cast<unsigned>(q.full + rest * q.splits));
  gemm_tile_dispatch(p.tile, [&](auto t) {
    using S = decltype(t);
    const dim3 block(S::RW * S::CW * 64);
    if (q.swiglu) hipLaunchKernelGGL((linear_gemm_kernel<S::MA, S::RW, S::CW, S::NS, DT, SAME, true>), grid, block, 0, st, q);
    else hipLaunchKernelGGL((linear_gemm_kernel<S::MA, S::RW, S::CW, S::NS, DT, SAME, false>), grid, block, 0, st, q);
  });
  if (rest > 0) {
    const GemmTileInfo& t = kGemmTiles[p.tile];
    const int items = rest * t.rw * t.cw * t.ma;
    const dim3 rgrid(static_cast<unsigned>(cdiv(items, 4)));
    if (q.swiglu) hipLaunchKernelGGL((linear_reduce_kernel<DT, SAME, true>), rgrid, dim3(256), 0, st, q, t.ma, t.rw, t.cw, items);
    else hipLaunchKernelGGL((linear_reduce_kernel<DT, SAME, false>), rgrid, dim3(256), 0, st, q, t.ma, t.rw, t.cw, items);
  }
}

}  // namespace

GemmPlan linear_plan(int64_t m, int64_t n, int64_t k, bool swiglu, bool split) {
  return gemm_plan(m, swiglu ? 2 * n : n, k, 4.0, 4.0, split ? INT64_MAX : 0);
}

void launch_linear_gemm(const GemmPlan& p, LinArgs q, int dt, hipStream_t st) {
  q.tiles_m = p.tiles_m;
  q.tiles_n = p.tiles_n;
  q.full = p.full;
  q.splits = p.splits;
  q.kt = static_cast<int>(q.k / 64);
  q.pairs = q.out_dt != BFA_DTYPE_F32 && q.ldo % 2 == 0 && reinterpret_cast<uintptr_t>(q.out) % 4 == 0;
  // (the sum's own rounding is fp32's, none, or the output's)
  const bool same = q.vec && q.n % 8 == 0 && q.proj_dt == dt && q.out_dt == dt &&
                    (q.swiglu || ((q.mid_dt == dt || q.mid_dt == BFA_DTYPE_F32) && (!q.res || q.res_dt == dt)));
  if (dt == BFA_DTYPE_BF16) {
    if (same) launch_form<BFA_DTYPE_BF16, true>(p, q, st);
    else launch_form<BFA_DTYPE_BF16, false>(p, q, st);
  } else {
    if (same) launch_form<BFA_DTYPE_F16, true>(p, q, st);
    else launch_form<BFA_DTYPE_F16, false>(p, q, st);
  }
}

}  // namespace bfa
