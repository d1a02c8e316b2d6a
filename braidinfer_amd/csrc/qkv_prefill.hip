// QKV projection above 64 tokens with head_dim 64 or 128: the GEMM of
// bfa_gemm.h with the projection's whole row epilogue (row scale, bias, rounding,
// per-head q/k RMSNorm, RoPE, store, paged KV append) in its registers.
//
// Bound by the matrix cores from a few thousand tokens, by the CUs that have a
// tile and by the epilogue below that.  A wave's 64 weight rows are 32 columns of
// a head's first half and the 32 that RoPE pairs with them, so a lane holds both
// of a pair, eight neighbouring pairs per token: no pass through the LDS, and
// 16-byte stores.  A head of 128 is two waves wide; only its sum of squares
// crosses them.  Tile choice and split K as for the linear layers
// (bfa_gemm_plan.h).
//
// Measured against the kernel that staged its accumulators through the LDS, on
// tiles of its own (fused RMSNorm + QKV + RoPE, same box): Llama-3-8B 300 tokens
// 46 -> 32 us, 3000 214 -> 154 us, 8192 382 -> 367 us; TinyLlama 8192 128 -> 101
// us; Qwen3 with q/k norm 3000 59 -> 45 us, 8192 119 -> 108 us.
#include "bfa_gemm.h"
#include "bfa_host.h"
#include "bfa_qkv.h"
#include "bfa_qkv_prefill.h"

namespace bfa {

// Weight row of the tile's row c (wave c / 64; its rows 16 j + 4 g + v): column
// 8 g + 4 (j % 2) + v of the wave's 32 in the first (j < 2) or second half.
template <int HD>
__device__ __forceinline__ int64_t qkv_weight_row(int64_t n, int64_t n0, int c) {
  constexpr int WPH = HD / 64;  // waves per head
  const int w = c >> 6, j = (c >> 4) & 3, g = (c >> 2) & 3, v = c & 3;
  return min(n0 + (w / WPH) * HD + (w % WPH) * 32 + (j >> 1) * (HD / 2) + g * 8 + (j & 1) * 4 + v, n - 1);
}

// Per-token values of a tile (or of a reduction block), filled from registers
// once the LDS ring is free.
template <int ROWS, int SUMS>
struct QkvTab {
  int64_t slot[ROWS];  // cache slot, -1: not appended
  int32_t pos[ROWS];   // -1: outside the table
  float scale[ROWS];
  float sum[SUMS];     // [wave][token of the wave]: sums of squares
};
struct QkvTok {
  int64_t slot, rawpos;
  float scale;
};

// Everything a token's epilogue needs, requested ahead of its use.
__device__ __forceinline__ QkvTok qkv_token(const QkvEpi& e, int64_t row) {
  QkvTok t{-1, 0, 1.f};
  if (e.row_scale) t.scale = e.row_scale[row];
  if (e.cs)
    t.rawpos = e.pos_is_i64 ? static_cast<const int64_t*>(e.positions)[row]
                            : static_cast<const int32_t*>(e.positions)[row];
  if (e.cache) t.slot = append_slot(e.app, append_key(e.app, row));
  return t;
}

template <class TAB>
__device__ __forceinline__ void qkv_tab_put(TAB& tab, int r, const QkvEpi& e, const QkvTok& t) {
  tab.slot[r] = t.slot;
  tab.scale[r] = t.scale;
  tab.pos[r] = e.cs ? epi_pos_check(e, t.rawpos) : 0;
}

// Eight neighbouring 16-bit elements in one word group.
template <int DT>
__device__ __forceinline__ u32x4_t qkv_pack8(const float (&y)[8]) {
  uint32_t w[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    if constexpr (DT == BFA_DTYPE_BF16) w[t] = pack_bf16x2(y[2 * t], y[2 * t + 1]);
    else w[t] = Elem<DT>::from_f32(y[2 * t]) | (static_cast<uint32_t>(Elem<DT>::from_f32(y[2 * t + 1])) << 16);
  }
  return u32x4_t{w[0], w[1], w[2], w[3]};
}

// Run-time dtype: 16-byte stores where the rows allow them (vec), else 8-byte
// (16-bit) or 16-byte (fp32) ones.
__device__ __forceinline__ void qkv_store8(void* p, int dt, int64_t i, const float (&y)[8], int vec) {
  if (dt == BFA_DTYPE_F32) {
    store8<BFA_DTYPE_F32>(static_cast<float*>(p) + i, y);
    return;
  }
  u32x4_t w;
  if (dt == BFA_DTYPE_BF16) w = qkv_pack8<BFA_DTYPE_BF16>(y);
  else w = qkv_pack8<BFA_DTYPE_F16>(y);
  uint16_t* d = static_cast<uint16_t*>(p) + i;
  if (vec) {
    *reinterpret_cast<u32x4_t*>(d) = w;
  } else {
    reinterpret_cast<uint2*>(d)[0] = make_uint2(w.x, w.y);
    reinterpret_cast<uint2*>(d)[1] = make_uint2(w.z, w.w);
  }
}

// Rounds a lane's eight values to DT (compile time) or dt: to bf16 two at a time.
// Rounding both ways and selecting cost the run-time form up to 9 % of a call
// (Qwen3 in fp16, 4096 tokens 58.3 -> 53.1 us).
template <int DT>
__device__ __forceinline__ void qkv_rnd8(float (&v)[8], int dt) {
  if constexpr (DT < 0) {  // (uniform)
    if (dt == BFA_DTYPE_BF16) qkv_rnd8<BFA_DTYPE_BF16>(v, dt);
    else if (dt == BFA_DTYPE_F16) qkv_rnd8<BFA_DTYPE_F16>(v, dt);
    return;
  }
#pragma unroll
  for (int t = 0; t < 8; t += 2) {
    if constexpr (DT == BFA_DTYPE_BF16) {
      const uint32_t w = pack_bf16x2(v[t], v[t + 1]);
      v[t] = __uint_as_float(w << 16);
      v[t + 1] = __uint_as_float(w & 0xffff0000u);
    } else if constexpr (DT >= 0) {
      v[t] = Elem<DT>::round(v[t]);
      v[t + 1] = Elem<DT>::round(v[t + 1]);
    }
  }
}

// Elements i .. i + 7 of a small vector of run-time dtype: all the loads
// (branch-free, ld_word) before the first conversion.
__device__ __forceinline__ void qkv_vec8(const void* p, int dt, int64_t i, float (&v)[8]) {
  uint32_t w[8];
#pragma unroll
  for (int t = 0; t < 8; ++t) w[t] = ld_word(p, dt, i + t);
#pragma unroll
  for (int t = 0; t < 8; ++t) v[t] = word_value(w[t], dt, p, i + t);
}

// The rows of a wave: MA blocks of 16 tokens from `row0` (table index `trow`),
// columns [32 sub + 8 g, + 8) and their RoPE partners of head `head`.  Every wave
// of the workgroup calls it (the q/k norm of a 128-wide head has a barrier); a
// wave whose head lies past the last one stores nothing.  mine / other: this
// wave's sums of squares and those of the wave with the rest of the head.
template <int HD, int EDT, int MA, class TAB>
__device__ __forceinline__ void qkv_rows(gemm_f32x4_t (&acc)[MA][4], const QkvEpi& e, const QkvPrefillArgs& q,
                                         int64_t row0, int trow, int64_t head, int sub, int lane, const TAB& tab,
                                         float* mine, const float* other) {
  using D = QkvDt<EDT>;
  const int fr = lane & 15, c = sub * 32 + (lane >> 4) * 8;
  const bool live = head < e.hq + 2 * e.hkv;
  const int64_t h = min(head, e.hq + 2 * e.hkv - 1);
  const int kd = head_kind(e, h);
  const int64_t gc = h * HD + c;  // first column; its partner is gc + HD / 2
  constexpr bool NORM = EDT == EDT_RT || EDT == EDT_BF16;  // the fp32 forms have no q/k norm
  const bool norm = NORM && (e.qn_w != nullptr || e.kn_w != nullptr);
  const void* nw = !NORM ? nullptr : kd == 0 ? e.qn_w : (kd == 1 ? e.kn_w : nullptr);
  const bool rope = e.cs != nullptr && kd != 2;

  // a block's cos/sin rows are requested one block ahead, before the stores of
  // the block between (the memory counter is in order and counts stores too)
  float4 cs[2][4];
  auto load_cs = [&](int i, float4 (&v)[4]) {
    const int32_t p = max(tab.pos[trow + i * 16 + fr], 0);
    const float* src = e.cs + static_cast<int64_t>(p) * HD + c;
    v[0] = *reinterpret_cast<const float4*>(src);
    v[1] = *reinterpret_cast<const float4*>(src + 4);
    v[2] = *reinterpret_cast<const float4*>(src + HD / 2);
    v[3] = *reinterpret_cast<const float4*>(src + HD / 2 + 4);
  };
  if (rope) load_cs(0, cs[0]);
  float g1[8], g2[8];
  if (nw) {
    qkv_vec8(nw, e.qk_w_dtype, c, g1);
    qkv_vec8(nw, e.qk_w_dtype, HD / 2 + c, g2);
  }
  {
    float b1[8], b2[8];
    if (e.bias) {
      qkv_vec8(e.bias, e.bias_dtype, gc, b1);
      qkv_vec8(e.bias, e.bias_dtype, gc + HD / 2, b2);
    }
#pragma unroll
    for (int i = 0; i < MA; ++i) {
      const float r = e.row_scale ? tab.scale[trow + i * 16 + fr] : 1.f;
      float x1[8], x2[8];
#pragma unroll
      for (int t = 0; t < 8; ++t) {
        x1[t] = acc[i][t >> 2][t & 3];
        x2[t] = acc[i][2 + (t >> 2)][t & 3];
        if (e.row_scale) { x1[t] = x1[t] * r; x2[t] = x2[t] * r; }
        if (e.bias) { x1[t] = x1[t] + b1[t]; x2[t] = x2[t] + b2[t]; }
      }
      qkv_rnd8<D::Q>(x1, e.qkv_dt);
      qkv_rnd8<D::Q>(x2, e.qkv_dt);
#pragma unroll
      for (int t = 0; t < 8; ++t) {
        acc[i][t >> 2][t & 3] = x1[t];
        acc[i][2 + (t >> 2)][t & 3] = x2[t];
      }
      if (norm) {
        float ss = 0.f;
#pragma unroll
        for (int t = 0; t < 8; ++t) ss += x1[t] * x1[t] + x2[t] * x2[t];
        ss = lanes4_sum(ss);
        if (lane < 16) mine[i * 16 + lane] = ss;
      }
    }
  }
  if (norm) __syncthreads();
  const int dt_after = nw ? e.norm_dt : e.qkv_dt;
  const bool app = e.cache != nullptr && kd != 0;
  const bool out_ok = kd == 0 || !e.skip_kv_out;
  const int64_t hk = h - e.hq - (kd == 2 ? e.hkv : 0);
  const int64_t cbase = (kd == 2 ? e.c_skv : 0) + hk * e.c_sh + c;
  bool bad = false;
#pragma unroll
  for (int i = 0; i < MA; ++i) {
    if (rope && i + 1 < MA) load_cs(i + 1, cs[(i + 1) & 1]);
    const int64_t row = row0 + i * 16 + fr;
    float x1[8], x2[8];
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      x1[t] = acc[i][t >> 2][t & 3];
      x2[t] = acc[i][2 + (t >> 2)][t & 3];
    }
    if (nw) {
      float ss = mine[i * 16 + fr];
      if constexpr (HD == 128) ss = ss + other[i * 16 + fr];
      const float r = __builtin_amdgcn_rsqf(ss / static_cast<float>(HD) + e.qk_eps);
#pragma unroll
      for (int t = 0; t < 8; ++t) {
        x1[t] = (x1[t] * r) * g1[t];
        x2[t] = (x2[t] * r) * g2[t];
      }
      qkv_rnd8<D::N>(x1, e.norm_dt);
      qkv_rnd8<D::N>(x2, e.norm_dt);
    }
    if (rope) {
      const bool ok = tab.pos[trow + i * 16 + fr] >= 0;
      bad = bad || (!ok && row < q.m);
      const float4 (&v)[4] = cs[i & 1];
      const float co[8] = {v[0].x, v[0].y, v[0].z, v[0].w, v[1].x, v[1].y, v[1].z, v[1].w};
      const float si[8] = {v[2].x, v[2].y, v[2].z, v[2].w, v[3].x, v[3].y, v[3].z, v[3].w};
#pragma unroll
      for (int t = 0; t < 8; ++t) {
        const float u = x1[t], w = x2[t];
        x1[t] = ok ? u * co[t] - w * si[t] : 0.f;
        x2[t] = ok ? w * co[t] + u * si[t] : 0.f;
      }
      // (a rounding to the stored dtype is the store's own)
      if constexpr (D::A < 0 || D::A != D::O) {
        qkv_rnd8<D::A>(x1, dt_after);
        qkv_rnd8<D::A>(x2, dt_after);
      }
    }
    if (live && row < q.m) {
      const int64_t so = app ? tab.slot[trow + i * 16 + fr] : -1;
      if constexpr (D::O >= 0) {
        // 16-bit rows that take 16-byte stores, the cache in the output's dtype
        const u32x4_t w1 = qkv_pack8<D::O>(x1), w2 = qkv_pack8<D::O>(x2);
        if (out_ok) {
          u32x4_t* d = reinterpret_cast<u32x4_t*>(static_cast<uint16_t*>(e.out) + row * e.ldo + gc);
          if (q.stream) {
            __builtin_nontemporal_store(w1, d);
            __builtin_nontemporal_store(w2, d + HD / 16);
            asm volatile("" ::: "memory");  // else the two branches' stores are merged into plain ones
          } else {
            d[0] = w1;
            d[HD / 16] = w2;
          }
        }
        if (so >= 0) {
          u32x4_t* d = reinterpret_cast<u32x4_t*>(static_cast<uint16_t*>(e.cache) + so + cbase);
          d[0] = w1;
          d[HD / 16] = w2;
        }
      } else {
        if (out_ok) {
          qkv_store8(e.out, e.out_dt, row * e.ldo + gc, x1, q.vec_out);
          qkv_store8(e.out, e.out_dt, row * e.ldo + gc + HD / 2, x2, q.vec_out);
        }
        if (so >= 0) {
          qkv_rnd8<-1>(x1, e.out_dt);
          qkv_rnd8<-1>(x2, e.out_dt);
          qkv_store8(e.cache, e.cache_dt, so + cbase, x1, q.vec_cache);
          qkv_store8(e.cache, e.cache_dt, so + cbase + HD / 2, x2, q.vec_cache);
        }
      }
    }
  }
  if (bad && live) flag_status(e.status, BFA_STATUS_INDEX_OOB);
}

template <int MA, int RW, int CW, int NS, int DT, int HD, int EDT>
__global__ __launch_bounds__(RW * CW * 64, 2) void qkv_prefill_kernel(QkvPrefillArgs q, QkvEpi e) {
  using T = GemmTile<MA, RW, CW, NS, DT>;
  using Tab = QkvTab<T::BM, T::NW * MA * 16>;
  static_assert(sizeof(Tab) <= T::LDS_U4 * 16 && T::BM <= T::NW * 64, "the table takes the ring's place");
  __shared__ uint4 lds[T::LDS_U4];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wr = wid / CW, wc = wid % CW;
  const int b = blockIdx.x;
  const bool part = b >= q.full;
  const int rest = q.tiles_m * q.tiles_n - q.full;
  const int u = part ? gemm_band(b - q.full, rest * q.splits) : gemm_band(b, q.full);
  const int split = part ? u / rest : 0, tile = part ? q.full + (u - split * rest) : u, ns = part ? q.splits : 1;
  int tm, tn;
  gemm_tile(q.tiles_m, q.tiles_n, tile, tm, tn);
  const int64_t m0 = static_cast<int64_t>(tm) * T::BM, n0 = static_cast<int64_t>(tn) * T::BN;
  const int k0 = static_cast<int>(static_cast<int64_t>(q.kt) * split / ns);
  const int nk = static_cast<int>(static_cast<int64_t>(q.kt) * (split + 1) / ns) - k0;
  typename T::Acc acc;
  QkvTok tok{-1, 0, 1.f};
  T::run(acc, lds, q.a + static_cast<int64_t>(k0) * 64, q.w + static_cast<int64_t>(k0) * 64, q.m, q.lda, q.ldw, m0, nk,
         wid, lane, [&](int c) { return qkv_weight_row<HD>(e.n, n0, c); },
         [&] {
           if (!part && tid < T::BM) tok = qkv_token(e, min(m0 + tid, q.m - 1));
         });
  const int64_t wm0 = m0 + wr * MA * 16;
  if (part) {
    gemm_store_part<MA, 4>(q.part, static_cast<int64_t>(tile - q.full) * q.splits + split, T::NW, wid, lane,
                           static_cast<int>(cdiv(q.m - wm0, 16)), acc);
    return;
  }
  Tab& tab = *reinterpret_cast<Tab*>(lds);
  __syncthreads();  // the ring's last reads are done
  if (tid < T::BM) qkv_tab_put(tab, tid, e, tok);
  __syncthreads();
  constexpr int WPH = HD / 64;
  qkv_rows<HD, EDT, MA>(acc, e, q, wm0, wr * MA * 16, n0 / HD + wc / WPH, wc % WPH, lane, tab, tab.sum + wid * MA * 16,
                        tab.sum + (WPH == 2 ? wid ^ 1 : wid) * MA * 16);
}

// One wave per 16-token x 64-column block of a split tile, the column blocks of
// one token block next to each other, so that the two waves of a head share a
// workgroup (cw is even).
template <int HD, int EDT>
__global__ __launch_bounds__(256) void qkv_prefill_reduce_kernel(QkvPrefillArgs q, QkvEpi e, int ma, int rw, int cw,
                                                                 int items) {
  using Tab = QkvTab<32, 4 * 16>;
  __shared__ Tab tab;
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  const int per = rw * cw * ma;
  // item = (split tile, 16-token block of the tile, wave column)
  auto locate = [&](int item, int& tile, int& rb, int& wc, int64_t& row0, int& tn) {
    tile = item / per;
    const int in = item - tile * per;
    rb = in / cw;
    wc = in - rb * cw;
    int tm;
    gemm_tile(q.tiles_m, q.tiles_n, q.full + tile, tm, tn);
    row0 = (static_cast<int64_t>(tm) * rw * ma + rb) * 16;
  };
  int tile, rb, wc, tn;
  int64_t row0;
  if (tid < 32) {  // the block's two wave pairs, 16 tokens each
    locate(min(static_cast<int>(blockIdx.x) * 4 + (tid >> 4) * 2, items - 1), tile, rb, wc, row0, tn);
    qkv_tab_put(tab, tid, e, qkv_token(e, min(row0 + (tid & 15), q.m - 1)));
  }
  const int item = blockIdx.x * 4 + wid;
  locate(min(item, items - 1), tile, rb, wc, row0, tn);
  gemm_f32x4_t acc[1][4] = {};
  if (row0 < q.m) {
    const int64_t stride = static_cast<int64_t>(per) * 256;
    const int wr = rb / ma, i = rb - wr * ma;
    gemm_sum_part(reinterpret_cast<const gemm_f32x4_t*>(q.part) + static_cast<int64_t>(tile) * q.splits * stride +
                      (static_cast<int64_t>(wr * cw + wc) * ma + i) * 256 + lane,
                  stride, q.splits, acc[0]);
  }
  __syncthreads();
  constexpr int WPH = HD / 64;
  const int64_t head = item < items ? (static_cast<int64_t>(tn) * cw + wc) / WPH : e.hq + 2 * e.hkv;
  qkv_rows<HD, EDT, 1>(acc, e, q, row0, (wid >> 1) * 16, head, wc % WPH, lane, tab, tab.sum + wid * 16,
                       tab.sum + (WPH == 2 ? wid ^ 1 : wid) * 16);
}

// ------------------------------------------------------------------- host
namespace {

template <int DT, int HD, int EDT>
void launch_edt(const GemmPlan& p, const QkvPrefillArgs& q, const QkvEpi& e, hipStream_t st) {
  const int rest = q.tiles_m * q.tiles_n - q.full;
  const dim3 grid(static_cast<unsigned>(q.full + rest * q.splits));
  gemm_tile_dispatch(p.tile, [&](auto t) {
    using S = decltype(t);
    hipLaunchKernelGGL((qkv_prefill_kernel<S::MA, S::RW, S::CW, S::NS, DT, HD, EDT>), grid, dim3(S::RW * S::CW * 64), 0,
                       st, q, e);
  });
  if (rest > 0) {
    const GemmTileInfo& t = kGemmTiles[p.tile];
    const int items = rest * t.rw * t.cw * t.ma;
    hipLaunchKernelGGL((qkv_prefill_reduce_kernel<HD, EDT>), dim3(static_cast<unsigned>(cdiv(items, 4))), dim3(256), 0,
                       st, q, e, t.ma, t.rw, t.cw, items);
  }
}

template <int DT, int HD>
void launch_hd(const GemmPlan& p, const QkvPrefillArgs& q, const QkvEpi& e, int edt, hipStream_t st) {
  if constexpr (DT == BFA_DTYPE_BF16) {
    if (edt == EDT_F32_BF16) return launch_edt<DT, HD, EDT_F32_BF16>(p, q, e, st);
    if (edt == EDT_BF16) return launch_edt<DT, HD, EDT_BF16>(p, q, e, st);
  } else {
    if (edt == EDT_F32_F16) return launch_edt<DT, HD, EDT_F32_F16>(p, q, e, st);
  }
  launch_edt<DT, HD, EDT_RT>(p, q, e, st);
}

}  // namespace

// The partials stay within what the entry point without a workspace holds
// beside the operand, so that it runs the same plan.
GemmPlan qkv_prefill_plan(int64_t m, int64_t n, int64_t k, int64_t operand_bytes, bool split) {
  // (the reduction resolves positions and cache slots again before its stores: 8
  // us with its launch; TinyLlama, 214 tokens: split 19.6 us, whole 18.9)
  return gemm_plan(m, n, k, 6.0, 8.0, split ? std::max<int64_t>(0, BFA_NOALLOC_SCRATCH_BYTES - operand_bytes) : 0);
}

void launch_qkv_prefill(const GemmPlan& p, QkvPrefillArgs q, const QkvEpi& e, int dt, int edt, hipStream_t st) {
  q.tiles_m = p.tiles_m;
  q.tiles_n = p.tiles_n;
  q.full = p.full;
  q.splits = p.splits;
  q.kt = static_cast<int>(q.k / 64);
  q.vec_out = e.out_dt == BFA_DTYPE_F32 || e.ldo % 8 == 0;
  q.vec_cache = e.cache_dt == BFA_DTYPE_F32 ||
                (e.c_skv % 8 == 0 && e.c_sh % 8 == 0 && e.app.c_sp % 8 == 0 && e.app.c_ss % 8 == 0);
  // Large outputs are stored past the caches (stream_output): at 8192 tokens the
  // Llama-3-8B projection's 100 MB then leave the operand and weight panels in
  // L2 and the Infinity Cache, 366 -> 353 us.
  q.stream = stream_output(q.m * e.n * dtype_size(e.out_dt));
  // the fixed forms store 16 bytes at a time and a cache of the output's dtype
  if (!q.vec_out || (e.cache && (!q.vec_cache || e.cache_dt != e.out_dt))) edt = EDT_RT;
  if (dt == BFA_DTYPE_BF16) {
    if (e.hd == 128) launch_hd<BFA_DTYPE_BF16, 128>(p, q, e, edt, st);
    else launch_hd<BFA_DTYPE_BF16, 64>(p, q, e, edt, st);
  } else {
    if (e.hd == 128) launch_hd<BFA_DTYPE_F16, 128>(p, q, e, edt, st);
    else launch_hd<BFA_DTYPE_F16, 64>(p, q, e, edt, st);
  }
}

}  // namespace bfa
