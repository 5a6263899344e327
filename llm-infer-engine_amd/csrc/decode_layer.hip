// Fused W8A16 kernels of one decode step (M <= 16 token rows).
//
// A decode step of the W8A16 Llama block (src/model_quantized.py:42-93 with
// src/model.py:39-127) is a chain of small matrix-vector products; run one
// launch per reference op, the step is dominated by launch gaps and by
// kernels too small to reach HBM bandwidth.  These kernels fold every
// elementwise neighbour of a projection into it:
//
//   rmsnorm -> wq | wk | wv -> RoPE(q), RoPE(k) + KV-cache append, v append
//   wo -> + residual
//   rmsnorm -> w1 | w3 -> silu(w1 x) * (w3 x)
//   w2 -> + residual
//
// Arithmetic follows the reference op by op: RMSNorm in fp32 rounded once to
// the activation dtype (src/rms_norm.py:32-38); each projection accumulates
// x.f32 * q.f32 in fp32 and applies the row scale after the sum
// (src/quant_linear.py:37-57), rounded to the activation dtype; RoPE,
// residual adds and silu/mul then act on those rounded values exactly as the
// reference's separate ops do (src/rope.py:85-86, src/model.py:23, :113-127).
//
// GEMV design (MI355X): the int8 weights are the only large operand and are
// read once.  A workgroup owns a few tiles of 8 (up to 8 token rows, or where
// larger tiles would leave half the CUs idle) or 16 output rows of one (or, for
// SwiGLU, two) weight matrices and its waves split K.  The products run on
// v_mfma_f32_16x16x32_{bf16,f16}: weight rows are the A operand (int8 converted
// exactly in registers), x^T the B operand with the columns beyond M zero.  A
// wave issues every load of its K slice before its first MFMA, so the whole
// matrix is in flight at once (these GEMVs are latency-bound: a few MB each).
// With the RMSNorm prologue each wave normalises its own slice of x in
// registers.
#include <math.h>
#include <type_traits>

#include "common.hpp"

namespace mi {

enum : int32_t {
  kEpiStore = 0,     // y = round(acc * s)
  kEpiResidual = 1,  // y = round(res + round(acc * s))
  kEpiSwiglu = 2,    // y = round(round(silu(a)) * b), a/b = rounded w1/w3 outputs
  kEpiQkvRope = 3,   // q -> RoPE -> q_out; k -> RoPE -> cache_k[pos]; v -> cache_v[pos]
};

struct LayerGemvArgs {
  const void* x;        // [M, K], unit k stride, row stride x_sm
  const void* norm_w;   // [K] RMSNorm weight (prologue) or null
  float eps;
  const int8_t* w0;     // first matrix [N0, K] (QKV: wq; SwiGLU: w1)
  const int8_t* w1;     // second matrix (QKV: wk; SwiGLU: w3) or null
  const int8_t* w2;     // third matrix (QKV: wv) or null
  const void* s0;       // row scales of w0 / w1 / w2
  const void* s1;
  const void* s2;
  int64_t w_sn0, w_sn1, w_sn2;  // weight row strides (bytes)
  void* y;              // output [M, N] (store / residual / swiglu) or q_out
  const void* res;      // residual [M, N]
  int64_t x_sm, y_sm, res_sm;
  int32_t M, K, N;      // N: output rows (QKV: Hq*D)
  int32_t n_tiles0;     // QKV: tiles of wq (the rest are wk then wv)
  int32_t n_tiles1;
  int32_t pair_kv;      // QKV with two tiles per block: wk / wv tiles paired too
  // QKV + RoPE + append
  const void* cos;      // [rows, D/2] tables, row stride c_ss (elements); position
  const void* sin;      //   p uses row p - rope_row0
  int64_t c_ss, rope_row0, rope_rows;
  const int64_t* pos;   // device position (one for all rows)
  void* ck;             // cache views of this layer: element (m, h, p, d) at
  void* cv;             //   m*c_sb + h*c_sh + p*c_st + d
  int64_t c_sb, c_sh, c_st;
  int64_t capacity;     // T
  int32_t Hq, Hkv, D;
};

template <typename T> struct LMfma;
template <> struct LMfma<bf16_t> {
  typedef __bf16 v8 __attribute__((ext_vector_type(8)));
  __device__ static inline f32x4 mma(const v8& a, const v8& b, const f32x4& c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
  }
};
template <> struct LMfma<f16_t> {
  typedef _Float16 v8 __attribute__((ext_vector_type(8)));
  __device__ static inline f32x4 mma(const v8& a, const v8& b, const f32x4& c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
  }
};

// 8 signed bytes (two words) -> 8 activation-dtype values (exact).
template <typename T, typename V8>
__device__ inline V8 i8x8_cvt(uint32_t lo, uint32_t hi) {
  if constexpr (std::is_same<T, bf16_t>::value) {
    // integers of magnitude <= 128 have 8 significant bits: the fp32 upper
    // halves are the bf16 values, so pair them with one byte permute
    auto hi2 = [](float a, float b) {
      return __builtin_amdgcn_perm(__float_as_uint(b), __float_as_uint(a), 0x07060302u);
    };
    u32x4 r;
    r.x = hi2((float)(int8_t)lo, (float)(int8_t)(lo >> 8));
    r.y = hi2((float)(int8_t)(lo >> 16), (float)(int8_t)(lo >> 24));
    r.z = hi2((float)(int8_t)hi, (float)(int8_t)(hi >> 8));
    r.w = hi2((float)(int8_t)(hi >> 16), (float)(int8_t)(hi >> 24));
    return __builtin_bit_cast(V8, r);
  } else {
    V8 r;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      r[i] = (T)(float)(int8_t)(lo >> (8 * i));
      r[4 + i] = (T)(float)(int8_t)(hi >> (8 * i));
    }
    return r;
  }
}


// x from lane (lane ^ OFF) without LDS traffic: a DPP row rotate for 8 (a
// 16-lane row rotated by 8 is the xor), the gfx950 permlane swaps for 16 and 32.
template <int OFF>
__device__ inline float dl_lane_xor(float x, int lane) {
  if constexpr (OFF == 8) {
    return __int_as_float(
        __builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x128, 0xF, 0xF, true));
  } else if constexpr (OFF == 16) {
    auto sw = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false,
                                               false);
    return __uint_as_float((lane & 16) ? sw[0] : sw[1]);
  } else {
    static_assert(OFF == 32, "lane stride");
    auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false,
                                               false);
    return __uint_as_float((lane & 32) ? sw[0] : sw[1]);
  }
}

// ---------------------------------------------------------------------------
// Diagonal-packed GEMV for M <= 8 token rows.
//
// One v_mfma_f32_16x16x32 multiplies a 16 x 32 A tile by a 32 x 16 B tile.
// With at most 8 token rows half of B's columns would be padding, and an
// 8-row weight tile half of A's rows; padding lanes still cost the CU's
// vector-memory issue (about 64 bytes per clock per CU, the limit of these
// small GEMVs once the weight stream is in flight).  Here both halves carry
// data: A lanes of rows r < 8 hold weight row n(r) over the first 64 k of a
// 128-k superchunk, rows r >= 8 the same weight rows over the second 64 k; B
// columns c < 8 hold token row c over the first 64 k, columns c >= 8 token row
// c - 8 over the second.  C[r][c] + C[r + 8][c + 8] (r, c < 8) is then the
// 128-k dot product and the off-diagonal quadrants are discarded: every byte
// loaded is used.
//
// A block has NW waves splitting K (SC consecutive superchunks each, K =
// 128 * NW * SC) and owns TPB 8-row tiles of each of its NMAT matrices.  With
// the RMSNorm prologue each wave normalises its own x slice in registers (the
// row statistics meet once in LDS).  Each wave folds its diagonal quadrants
// in registers, the waves' sums meet in LDS, and one thread per (token row,
// output row) sums them and runs the epilogue.
template <typename T, int NW, int SC, bool NORM, int EPI, int TPB>
__global__ __launch_bounds__(64 * NW) void dgemv_kernel(LayerGemvArgs a) {
  using MM = LMfma<T>;
  typedef typename MM::v8 v8;
  constexpr int NMAT = EPI == kEpiSwiglu ? 2 : 1;
  constexpr int NT = NMAT * TPB;                       // 8-row A tiles per block
  constexpr int RB = 8 * TPB;                          // output rows per block (per matrix)
  constexpr int NOUT = EPI == kEpiQkvRope ? 64 * TPB : 8 * RB;  // epilogue threads
  static_assert(NOUT <= 64 * NW, "too few threads for the epilogue");
  __shared__ __align__(16) float red[NT][8][8][NW];    // [tile][row][token][wave]
  __shared__ float ssq[NORM ? NW : 1][8];              // per-wave sums of squares

  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r16 = lane & 15, g = lane >> 4;
  const int rr = r16 & 7;                // A: tile row / B: token row
  const int kofs = (r16 >> 3) * 64 + 16 * g;
  const bool m_ok = rr < a.M;
  // K slice of this wave, rotated by block so that concurrent blocks do not all
  // read the same x lines at the same time
  const int ks = (w + (int)blockIdx.x) % NW;
  const int kw = ks * SC * 128;

  // ---- which matrix / tiles this block owns.  QKV: one tile per block, or
  //      (TPB = 2) tiles 2b and 2b + 1 of wq for the first ceil(n_tiles0 / 2)
  //      blocks, then the wk and the wv tiles one per block (or in pairs with
  //      pair_kv).  A CU that runs two blocks streams x twice and sets the
  //      launch's time, so grids with more tiles than CUs pair them (ntv: the
  //      tiles this block really has; a missing second tile loads zeros)
  int mat0 = 0, tile0 = blockIdx.x * TPB, ntv = TPB;
  if constexpr (EPI == kEpiQkvRope) {
    int b = blockIdx.x;
    const int per0 = TPB == 2 ? (a.n_tiles0 + 1) >> 1 : a.n_tiles0;
    const bool pkv = TPB == 2 && a.pair_kv != 0;
    const int per1 = pkv ? (a.n_tiles1 + 1) >> 1 : a.n_tiles1;
    int nt = a.n_tiles0;
    if (b >= per0) {
      b -= per0;
      mat0 = 1;
      if (b >= per1) { b -= per1; mat0 = 2; }
      nt = a.n_tiles1;
    }
    const bool paired = TPB == 2 && (mat0 == 0 || pkv);
    tile0 = paired ? 2 * b : b;
    ntv = paired ? min(2, nt - tile0) : 1;
  }
  const int half = a.D >> 1, tph = EPI == kEpiQkvRope ? half >> 2 : 1;
  // weight row of tile row `row` of tile `tim` of the matrix: the QKV tiles hold
  // 4 rotation pairs (rows 0..3 dims d, rows 4..7 dims d + D/2)
  auto w_row = [&](int tim, int row) -> int {
    if constexpr (EPI == kEpiQkvRope) {
      const int head = tim / tph, j = tim - head * tph;
      return head * a.D + 4 * j + (row & 3) + ((row >> 2) ? half : 0);
    } else {
      return tim * 8 + row;
    }
  };
  const int8_t* wm0 = mat0 == 0 ? a.w0 : (mat0 == 1 ? a.w1 : a.w2);
  const int64_t wsn0 = mat0 == 0 ? a.w_sn0 : (mat0 == 1 ? a.w_sn1 : a.w_sn2);
  const int nvalid = EPI == kEpiQkvRope ? (mat0 == 0 ? a.Hq : a.Hkv) * a.D : a.N;
  // weight rows through buffer resources (host-checked: each matrix spans
  // < 2^31 bytes); rows past N get an out-of-range offset and load zeros
  buf_rsrc wr[NMAT];
  wr[0] = make_rsrc(wm0, (uint32_t)((int64_t)(nvalid - 1) * wsn0 + a.K));
  if constexpr (NMAT == 2) wr[1] = make_rsrc(a.w1, (uint32_t)((int64_t)(a.N - 1) * a.w_sn1 + a.K));
  uint32_t woff[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const int n = w_row(tile0 + (t % TPB), rr);
    const int64_t sn = t / TPB == 0 ? wsn0 : a.w_sn1;
    woff[t] = (n < nvalid && (t % TPB) < ntv) ? (uint32_t)((int64_t)n * sn) : kOobOffset;
  }

  // ---- B operand (token rows through a buffer resource: rows >= M read zeros
  //      without a memory access), then the norm weights, then every weight
  //      load of this wave; all issued before the first wait
  const buf_rsrc xrs =
      make_rsrc(a.x, (uint32_t)(((int64_t)(a.M - 1) * a.x_sm + a.K) * sizeof(T)));
  const uint32_t xo = m_ok ? (uint32_t)((int64_t)rr * a.x_sm * sizeof(T)) : kOobOffset;
  u32x4 xr[SC][2];
#pragma unroll
  for (int s = 0; s < SC; ++s) {
    const int k0 = kw + s * 128 + kofs;
    xr[s][0] = buf_load16(xrs, xo + (uint32_t)(k0 * sizeof(T)));
    xr[s][1] = buf_load16(xrs, xo + (uint32_t)((k0 + 8) * sizeof(T)));
  }
  u32x4 nr[NORM ? SC : 1][2];
  if constexpr (NORM) {
#pragma unroll
    for (int s = 0; s < SC; ++s) {
      const T* np = reinterpret_cast<const T*>(a.norm_w) + kw + s * 128 + kofs;
      nr[s][0] = load16(np);
      nr[s][1] = load16(np + 8);
    }
  }
  u32x4 wq[NT][SC];
#pragma unroll
  for (int s = 0; s < SC; ++s)
#pragma unroll
    for (int t = 0; t < NT; ++t)
      wq[t][s] = buf_load16_nt(wr[t / TPB], woff[t] + (uint32_t)(kw + s * 128 + kofs));

  // ---- epilogue operands, behind the weights (every thread loads from
  //      clamped indices; only threads < NOUT use them)
  const int et = tid % NOUT;
  T e_s0, e_s1, e_res, e_cos, e_sin;
  int64_t pos = 0;
  if constexpr (EPI == kEpiQkvRope) {
    pos = *a.pos;
    const T* sc = reinterpret_cast<const T*>(mat0 == 0 ? a.s0 : (mat0 == 1 ? a.s1 : a.s2));
    const int tt = tile0 + min(et >> 6, ntv - 1);   // this epilogue thread's tile
    const int row = et & 7, j = tt % tph;
    e_s0 = sc[w_row(tt, row)];
    e_s1 = sc[w_row(tt, row ^ 4)];
    const int64_t crow = min(max(pos - a.rope_row0, (int64_t)0), a.rope_rows - 1);
    const int ii = 4 * j + (row & 3);
    e_cos = reinterpret_cast<const T*>(a.cos)[crow * a.c_ss + ii];
    e_sin = reinterpret_cast<const T*>(a.sin)[crow * a.c_ss + ii];
  } else {
    const int em = min(et / RB, a.M - 1);
    const int en = min(blockIdx.x * RB + et % RB, a.N - 1);
    e_s0 = reinterpret_cast<const T*>(a.s0)[en];
    if constexpr (EPI == kEpiSwiglu) e_s1 = reinterpret_cast<const T*>(a.s1)[en];
    if constexpr (EPI == kEpiResidual)
      e_res = reinterpret_cast<const T*>(a.res)[(int64_t)em * a.res_sm + en];
  }
  __builtin_amdgcn_sched_barrier(0);

  // ---- RMSNorm: per-token-row sum of squares over this lane's k (lanes c,
  //      c ^ 8 and every k group share a token row), over waves in LDS; then
  //      x * rstd * w rounded once to T, in place
  if constexpr (NORM) {
    float ss = 0.f;
#pragma unroll
    for (int s = 0; s < SC; ++s)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        float v[8];
        Chunk<T>::unpack(xr[s][h], v);
#pragma unroll
        for (int e = 0; e < 8; ++e) ss = fmaf(v[e], v[e], ss);
      }
    ss += dl_lane_xor<8>(ss, lane);
    ss += dl_lane_xor<16>(ss, lane);
    ss += dl_lane_xor<32>(ss, lane);
    if (lane < 8) ssq[w][lane] = ss;
    __syncthreads();
    float tot = 0.f;
#pragma unroll
    for (int ww = 0; ww < NW; ++ww) tot += ssq[ww][rr];
    const float rstd = 1.0f / sqrtf(tot / (float)a.K + a.eps);
#pragma unroll
    for (int s = 0; s < SC; ++s)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        float v[8], wn[8];
        Chunk<T>::unpack(xr[s][h], v);
        Chunk<T>::unpack(nr[s][h], wn);
        typedef T t8 __attribute__((ext_vector_type(8)));
        t8 o;
#pragma unroll
        for (int e = 0; e < 8; ++e) o[e] = Elem<T>::from_f32(v[e] * rstd * wn[e]);
        xr[s][h] = __builtin_bit_cast(u32x4, o);
      }
  }

  // ---- MFMAs over the wave's superchunks
  f32x4 acc[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < SC; ++s) {
    const v8 xb0 = __builtin_bit_cast(v8, xr[s][0]);
    const v8 xb1 = __builtin_bit_cast(v8, xr[s][1]);
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      acc[t] = MM::mma(i8x8_cvt<T, v8>(wq[t][s].x, wq[t][s].y), xb0, acc[t]);
      acc[t] = MM::mma(i8x8_cvt<T, v8>(wq[t][s].z, wq[t][s].w), xb1, acc[t]);
    }
  }

  // ---- fold the diagonal quadrants: lane c + 16 g (g < 2, c < 8) holds
  //      C[4g + i][c], lane + 40 holds C[4g + i + 8][c + 8]
#pragma unroll
  for (int t = 0; t < NT; ++t) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float v = acc[t][i] + dl_lane_xor<8>(dl_lane_xor<32>(acc[t][i], lane), lane);
      if (g < 2 && r16 < 8) red[t][4 * g + i][r16][w] = v;
    }
  }
  __syncthreads();
  if (tid >= NOUT) return;

  // sum over waves of tile t, row `row`, token row `mm`
  auto wsum = [&](int t, int row, int mm) -> float {
    const f32x4* p = reinterpret_cast<const f32x4*>(&red[t][row][mm][0]);
    float acc_s = 0.f;
#pragma unroll
    for (int q = 0; q < NW / 4; ++q) {
      const f32x4 v = p[q];
      acc_s += v[0] + v[1] + v[2] + v[3];
    }
    return acc_s;
  };
  auto f32_of = [](T v) { return Elem<T>::to_f32(v); };
  auto rnd = [](float v) { return Elem<T>::to_f32(Elem<T>::from_f32(v)); };

  if constexpr (EPI == kEpiQkvRope) {
    const int te = tid >> 6, mm = (tid >> 3) & 7, row = tid & 7;
    if (mm >= a.M || te >= ntv) return;
    const int tt = tile0 + te;
    const float yv = rnd(wsum(te, row, mm) * f32_of(e_s0));
    const float yp = rnd(wsum(te, row ^ 4, mm) * f32_of(e_s1));
    const bool hi = row >= 4;
    const int head = tt / tph;
    const int d = w_row(tt, row) - head * a.D;
    T out;
    if (mat0 == 2) {
      out = Elem<T>::from_f32(yv);                  // v: appended unrotated (bitwise)
    } else {
      const float cs = f32_of(e_cos), sn = f32_of(e_sin);
      const float x1 = hi ? yp : yv, x2 = hi ? yv : yp;
      T y1, y2;
      {
#pragma clang fp contract(off)
        const float x1c = x1 * cs, x2s = x2 * sn, x2c = x2 * cs, x1s = x1 * sn;
        y1 = Elem<T>::from_f32(x1c - x2s);
        y2 = Elem<T>::from_f32(x2c + x1s);
      }
      out = hi ? y2 : y1;
    }
    if (mat0 == 0) {
      reinterpret_cast<T*>(a.y)[((int64_t)mm * a.Hq + head) * a.D + d] = out;
    } else if (pos >= 0 && pos < a.capacity) {
      T* c = reinterpret_cast<T*>(mat0 == 1 ? a.ck : a.cv);
      c[(int64_t)mm * a.c_sb + (int64_t)head * a.c_sh + pos * a.c_st + d] = out;
    }
  } else {
    const int mm = tid / RB, j = tid - mm * RB;
    const int n = blockIdx.x * RB + j;
    if (mm >= a.M || n >= a.N) return;
    float v = rnd(wsum(j >> 3, j & 7, mm) * f32_of(e_s0));
    if constexpr (EPI == kEpiResidual) {
      v = rnd(f32_of(e_res) + v);
    } else if constexpr (EPI == kEpiSwiglu) {
      const float b = rnd(wsum(TPB + (j >> 3), j & 7, mm) * f32_of(e_s1));
      v = rnd(silu_f32(v)) * b;
    }
    reinterpret_cast<T*>(a.y)[(int64_t)mm * a.y_sm + n] = Elem<T>::from_f32(v);
  }
}

// A lane's 16 bytes of weight row r for the first / second 64 k of a 128-k pair
// of chunks, from the two loads of the pair: a holds rows 0..7 and b rows 8..15,
// lanes r < 8 the first 64 k and lanes r >= 8 the second (each load reads whole
// 128-byte lines of 8 rows).  One DPP row rotate by 8 per word.
__device__ inline u32x4 rows_lo(const u32x4& a, const u32x4& b) {
  u32x4 o;
#pragma unroll
  for (int i = 0; i < 4; ++i)   // lanes 8..15 take b of lane r - 8
    o[i] = (uint32_t)__builtin_amdgcn_update_dpp((int)a[i], (int)b[i], 0x128, 0xF, 0xC, false);
  return o;
}
__device__ inline u32x4 rows_hi(const u32x4& a, const u32x4& b) {
  u32x4 o;
#pragma unroll
  for (int i = 0; i < 4; ++i)   // lanes 0..7 take a of lane r + 8
    o[i] = (uint32_t)__builtin_amdgcn_update_dpp((int)b[i], (int)a[i], 0x128, 0xF, 0x3, false);
  return o;
}

// ---------------------------------------------------------------------------
// GEMV for 9..16 token rows.
//
// With more than 8 token rows the B operand of v_mfma_f32_16x16x32 is full, so
// an A tile is 16 weight rows: lane (r, g) feeds 16 consecutive k of weight row
// r and of token row r for each 64-k chunk (two MFMAs); the weights of a pair of
// chunks are loaded as whole 128-byte lines of 8 rows (rows_lo / rows_hi).  A block has NW waves
// that split K (SC consecutive chunks each, K = 64 * NW * SC) and owns TPB
// tiles of RT rows (16, or 8 with the other A rows unused) of each of its NMAT
// matrices: every wave reads its slice of x
// once, straight into the B registers, for all of the block's tiles.  x is what
// bounds these calls, not the weights: a block with one tile reads twice as
// many bytes of x (16 rows of 2 bytes) as of int8 weights, so tiles are grouped
// until the grid is about one block per CU, and all weight loads are issued
// before the first wait.  With the RMSNorm prologue each wave normalises its
// own x slice in registers.  The waves' sums meet in LDS.
// MI355X, M = 16, per call in a graph over rotating weights, against one tile per
// block with 64-byte pieces of 16 rows per load (8-row tiles for N < 3840):
// [3072, 3072] 10.8 -> 6.3 us, [3072, 8192] 25.2 -> 14.6, SwiGLU 2 x [8192, 3072]
// 17.9 -> 13.0 (3.9 TB/s), SwiGLU 2 x [8192, 2048] 11.7 -> 9.5, [3072, 2048] 6.9 -> 4.9.
// What is left is x: the same calls with all 16 rows at one address take 1 to 3 us less.
template <typename T, int NW, int SC, bool NORM, int EPI, int TPB, int RT>
__global__ __launch_bounds__(64 * NW) void rows_gemv_kernel(LayerGemvArgs a) {
  using MM = LMfma<T>;
  typedef typename MM::v8 v8;
  constexpr int NMAT = EPI == kEpiSwiglu ? 2 : 1;
  constexpr int NT = NMAT * TPB;                       // A tiles (RT rows) per block
  constexpr int NOUT = 16 * RT * TPB;                  // outputs of a block
  constexpr int NO = (NOUT + 64 * NW - 1) / (64 * NW); // outputs of a thread
  __shared__ __align__(16) float red[NW][NT][16][16];  // [wave][tile][token][row]
  __shared__ float ssq[NORM ? NW : 1][16];             // per-wave sums of squares

  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, g = lane >> 4;   // A: tile row / B: token row; k group
  // K slice of this wave, rotated by block (concurrent blocks read different x lines)
  const int kw = ((w + (int)blockIdx.x) % NW) * SC * 64;
  const int kx = kw + 16 * g;

  // ---- the block's tiles.  QKV: tiles of wq, then wk, then wv in one list,
  //      each 8 rotation pairs of a head (rows 0..7 dims d, rows 8..15 d + D/2)
  const int half = a.D >> 1, tph = EPI == kEpiQkvRope ? half >> 3 : 1;
  const int n_tiles = EPI == kEpiQkvRope ? a.n_tiles0 + 2 * a.n_tiles1 : (a.N + RT - 1) / RT;
  auto mat_of = [&](int tile) -> int {
    if constexpr (EPI != kEpiQkvRope) return 0;
    return tile < a.n_tiles0 ? 0 : tile < a.n_tiles0 + a.n_tiles1 ? 1 : 2;
  };
  auto w_row = [&](int tile, int mat, int row) -> int {
    if constexpr (EPI == kEpiQkvRope) {
      const int tim = mat == 0 ? tile : tile - a.n_tiles0 - (mat == 2 ? a.n_tiles1 : 0);
      const int head = tim / tph, j = tim - head * tph;
      return head * a.D + 8 * j + (row & 7) + ((row >> 3) ? half : 0);
    } else {
      return tile * RT + row;
    }
  };
  // weight rows through buffer resources (host-checked: each matrix spans < 2^31
  // bytes); rows past N and tiles past the list load zeros without an access
  buf_rsrc wr[NT];
  uint32_t woff[NT][2];
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const int tile = blockIdx.x * TPB + t % TPB, mat = mat_of(tile);
    const bool b3 = t >= TPB;                          // SwiGLU's second matrix
    const int8_t* wm = b3 || mat == 1 ? a.w1 : mat == 2 ? a.w2 : a.w0;
    const int64_t sn = b3 || mat == 1 ? a.w_sn1 : mat == 2 ? a.w_sn2 : a.w_sn0;
    const int rows = EPI == kEpiQkvRope && mat != 0 ? a.Hkv * a.D : a.N;
    wr[t] = make_rsrc(wm, (uint32_t)((int64_t)(rows - 1) * sn + a.K));
#pragma unroll
    for (int h = 0; h < RT / 8; ++h) {
      const int n = w_row(tile, mat, 8 * h + (r & 7));
      woff[t][h] = (tile < n_tiles && n < rows ? (uint32_t)((int64_t)n * sn) : kOobOffset) +
                   (r >> 3) * 64 + 16 * g;
    }
  }

  // ---- x (rows >= M read zeros), norm weights, then every weight load
  const buf_rsrc xrs =
      make_rsrc(a.x, (uint32_t)(((int64_t)(a.M - 1) * a.x_sm + a.K) * sizeof(T)));
  const uint32_t xo = r < a.M ? (uint32_t)((int64_t)r * a.x_sm * sizeof(T)) : kOobOffset;
  u32x4 xr[SC][2];
#pragma unroll
  for (int s = 0; s < SC; ++s) {
    xr[s][0] = buf_load16(xrs, xo + (uint32_t)((kx + s * 64) * sizeof(T)));
    xr[s][1] = buf_load16(xrs, xo + (uint32_t)((kx + s * 64 + 8) * sizeof(T)));
  }
  u32x4 nr[NORM ? SC : 1][2];
  if constexpr (NORM) {
#pragma unroll
    for (int s = 0; s < SC; ++s) {
      const T* np = reinterpret_cast<const T*>(a.norm_w) + kx + s * 64;
      nr[s][0] = load16(np);
      nr[s][1] = load16(np + 8);
    }
  }
  u32x4 wq[NT][SC];
#pragma unroll
  for (int s = 0; s < SC; ++s)
#pragma unroll
    for (int t = 0; t < NT; ++t)
      if (RT == 16 || s % 2 == 0)
        wq[t][s] = buf_load16_nt(wr[t], woff[t][s & 1] + (uint32_t)(kw + (s >> 1) * 128));

  // ---- epilogue operands behind the weights, from clamped indices
  T e_s0[NO], e_s1[NO], e_res[NO], e_cos[NO], e_sin[NO];
  const int64_t pos = EPI == kEpiQkvRope ? *a.pos : 0;
#pragma unroll
  for (int o = 0; o < NO; ++o) {
    const int i = min(tid + o * 64 * NW, NOUT - 1);
    const int tile = min((int)blockIdx.x * TPB + i / (16 * RT), n_tiles - 1);
    const int row = i % RT, m = min(i / RT % 16, a.M - 1);
    if constexpr (EPI == kEpiQkvRope) {
      const int mat = mat_of(tile), n = w_row(tile, mat, row);
      const T* sc = reinterpret_cast<const T*>(mat == 0 ? a.s0 : mat == 1 ? a.s1 : a.s2);
      e_s0[o] = sc[n];
      e_s1[o] = sc[w_row(tile, mat, row ^ 8)];
      const int64_t crow = min(max(pos - a.rope_row0, (int64_t)0), a.rope_rows - 1);
      const int ii = (n % a.D) % half;
      e_cos[o] = reinterpret_cast<const T*>(a.cos)[crow * a.c_ss + ii];
      e_sin[o] = reinterpret_cast<const T*>(a.sin)[crow * a.c_ss + ii];
    } else {
      const int n = min(tile * RT + row, a.N - 1);
      e_s0[o] = reinterpret_cast<const T*>(a.s0)[n];
      if constexpr (EPI == kEpiSwiglu) e_s1[o] = reinterpret_cast<const T*>(a.s1)[n];
      if constexpr (EPI == kEpiResidual)
        e_res[o] = reinterpret_cast<const T*>(a.res)[(int64_t)m * a.res_sm + n];
    }
  }
  __builtin_amdgcn_sched_barrier(0);

  // ---- RMSNorm: a token row's sum of squares over this lane's k, the k groups
  //      and the waves; then x * rstd * w rounded once to T, in place
  if constexpr (NORM) {
    float ss = 0.f;
#pragma unroll
    for (int s = 0; s < SC; ++s)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        float v[8];
        Chunk<T>::unpack(xr[s][h], v);
#pragma unroll
        for (int e = 0; e < 8; ++e) ss = fmaf(v[e], v[e], ss);
      }
    ss += dl_lane_xor<16>(ss, lane);
    ss += dl_lane_xor<32>(ss, lane);
    if (lane < 16) ssq[w][lane] = ss;
    __syncthreads();
    float tot = 0.f;
#pragma unroll
    for (int ww = 0; ww < NW; ++ww) tot += ssq[ww][r];
    const float rstd = 1.0f / sqrtf(tot / (float)a.K + a.eps);
#pragma unroll
    for (int s = 0; s < SC; ++s)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        float v[8], wn[8];
        Chunk<T>::unpack(xr[s][h], v);
        Chunk<T>::unpack(nr[s][h], wn);
        typedef T t8 __attribute__((ext_vector_type(8)));
        t8 o;
#pragma unroll
        for (int e = 0; e < 8; ++e) o[e] = Elem<T>::from_f32(v[e] * rstd * wn[e]);
        xr[s][h] = __builtin_bit_cast(u32x4, o);
      }
  }

  // ---- MFMAs over the wave's chunks; acc[i] = C[tile row 4g + i][token r]
  f32x4 acc[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < SC; ++s) {
    const v8 xb0 = __builtin_bit_cast(v8, xr[s][0]);
    const v8 xb1 = __builtin_bit_cast(v8, xr[s][1]);
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      // (8-row tiles: A rows 8..15 are left as they come, nobody reads their sums)
      u32x4 wv;
      if constexpr (RT == 16)
        wv = s & 1 ? rows_hi(wq[t][s - 1], wq[t][s]) : rows_lo(wq[t][s], wq[t][s + 1]);
      else
        wv = s & 1 ? rows_hi(wq[t][s - 1], wq[t][s - 1]) : wq[t][s];
      acc[t] = MM::mma(i8x8_cvt<T, v8>(wv.x, wv.y), xb0, acc[t]);
      acc[t] = MM::mma(i8x8_cvt<T, v8>(wv.z, wv.w), xb1, acc[t]);
    }
  }
#pragma unroll
  for (int t = 0; t < NT; ++t) *reinterpret_cast<f32x4*>(&red[w][t][r][4 * g]) = acc[t];
  __syncthreads();

  auto wsum = [&](int t, int m, int row) -> float {
    float v = 0.f;
#pragma unroll
    for (int ww = 0; ww < NW; ++ww) v += red[ww][t][m][row];
    return v;
  };
  auto f32_of = [](T v) { return Elem<T>::to_f32(v); };
  auto rnd = [](float v) { return Elem<T>::to_f32(Elem<T>::from_f32(v)); };
#pragma unroll
  for (int o = 0; o < NO; ++o) {
    const int i = tid + o * 64 * NW;
    const int t = i / (16 * RT), tile = blockIdx.x * TPB + t, row = i % RT, m = i / RT % 16;
    if (i >= NOUT || tile >= n_tiles || m >= a.M) continue;
    if constexpr (EPI == kEpiQkvRope) {
      const int mat = mat_of(tile), n = w_row(tile, mat, row);
      const float yv = rnd(wsum(t, m, row) * f32_of(e_s0[o]));
      const float yp = rnd(wsum(t, m, row ^ 8) * f32_of(e_s1[o]));
      const int head = n / a.D, d = n - head * a.D;
      T out;
      if (mat == 2) {
        out = Elem<T>::from_f32(yv);                  // v: appended unrotated (bitwise)
      } else {
        const bool hi = row >= 8;
        T y1, y2;
        rope_rotate<T, T>(hi ? yp : yv, hi ? yv : yp, e_cos[o], e_sin[o], y1, y2);
        out = hi ? y2 : y1;
      }
      if (mat == 0) {
        reinterpret_cast<T*>(a.y)[((int64_t)m * a.Hq + head) * a.D + d] = out;
      } else if (pos >= 0 && pos < a.capacity) {
        T* c = reinterpret_cast<T*>(mat == 1 ? a.ck : a.cv);
        c[(int64_t)m * a.c_sb + (int64_t)head * a.c_sh + pos * a.c_st + d] = out;
      }
    } else {
      const int n = tile * RT + row;
      if (n >= a.N) continue;
      float v = rnd(wsum(t, m, row) * f32_of(e_s0[o]));
      if constexpr (EPI == kEpiResidual) {
        v = f32_of(e_res[o]) + v;
      } else if constexpr (EPI == kEpiSwiglu) {
        const float b = rnd(wsum(TPB + t, m, row) * f32_of(e_s1[o]));
        v = rnd(silu_f32(v)) * b;
      }
      reinterpret_cast<T*>(a.y)[(int64_t)m * a.y_sm + n] = Elem<T>::from_f32(v);
    }
  }
}

namespace {

template <typename T, bool NORM, int EPI, int TPB, int NW, int SC, int RT>
hipError_t launch_rows(const LayerGemvArgs& a, int n_tiles, hipStream_t st) {
  hipLaunchKernelGGL((rows_gemv_kernel<T, NW, SC, NORM, EPI, TPB, RT>),
                     dim3((unsigned)((n_tiles + TPB - 1) / TPB)), dim3(64 * NW), 0, st, a);
  return hipGetLastError();
}

// Waves and chunks per wave from K = 64 * NW * SC, at most 16 waves.
template <typename T, bool NORM, int EPI, int TPB, int RT>
hipError_t dispatch_rows_k(const LayerGemvArgs& a, int n_tiles, hipStream_t st) {
  switch (a.K) {
    case 512: return launch_rows<T, NORM, EPI, TPB, 4, 2, RT>(a, n_tiles, st);
    case 1024: return launch_rows<T, NORM, EPI, TPB, 8, 2, RT>(a, n_tiles, st);
    case 1536: return launch_rows<T, NORM, EPI, TPB, 12, 2, RT>(a, n_tiles, st);
    case 2048: return launch_rows<T, NORM, EPI, TPB, 8, 4, RT>(a, n_tiles, st);
    default: break;
  }
  if constexpr (!NORM) {   // the prologue serves K <= 2048 (host-checked)
    switch (a.K) {
      case 3072: return launch_rows<T, NORM, EPI, TPB, 12, 4, RT>(a, n_tiles, st);
      // 16 waves have 128 registers each: one tile of two matrices at a time
      case 4096:
        return launch_rows<T, NORM, EPI, EPI == kEpiSwiglu ? 1 : TPB, 16, 4, RT>(a, n_tiles, st);
      default: break;
    }
    if constexpr (EPI != kEpiSwiglu) {  // two weight streams: K <= 4096 (host-checked)
      switch (a.K) {
        case 6144: return launch_rows<T, NORM, EPI, 1, 16, 6, RT>(a, n_tiles, st);
        case 8192: return launch_rows<T, NORM, EPI, 1, 16, 8, RT>(a, n_tiles, st);
        default: break;
      }
    }
  }
  return hipErrorInvalidValue;
}

template <typename T, int EPI, int TPB, int RT>
hipError_t dispatch_rows_norm(const LayerGemvArgs& a, int n_tiles, hipStream_t st) {
  return a.norm_w != nullptr ? dispatch_rows_k<T, true, EPI, TPB, RT>(a, n_tiles, st)
                             : dispatch_rows_k<T, false, EPI, TPB, RT>(a, n_tiles, st);
}

// 9..16 rows: two tiles per block when one per block is more than a block per CU, and
// tiles of 8 rows where tiles of 16 leave half the CUs without a block (twice the
// blocks and twice the reads of x, but half the weights and sums per block).  MI355X,
// 16 rows, 16- against 8-row tiles, per call in a graph: [2048, 8192] 12.9 -> 11.5 us,
// [1024, 6144] 10.1 -> 8.9, [512, 2048] 4.7 -> 4.4, [2048, 512] 3.0 -> 2.8; [2080, 8192],
// the first N past the line, 12.9 with 16-row tiles.
template <typename T, int EPI>
hipError_t dispatch_rows(const LayerGemvArgs& a, int n_tiles, hipStream_t st) {
  const int cus = device_cu_count();
  if constexpr (EPI != kEpiQkvRope)
    if (2 * n_tiles <= cus) return dispatch_rows_norm<T, EPI, 1, 8>(a, (a.N + 7) / 8, st);
  return n_tiles > cus ? dispatch_rows_norm<T, EPI, 2, 16>(a, n_tiles, st)
                       : dispatch_rows_norm<T, EPI, 1, 16>(a, n_tiles, st);
}

// Diagonal-packed kernel (M <= 8): waves and superchunks per wave from K =
// 128 * NW * SC, at most 16 waves.
template <typename T, bool NORM, int EPI, int TPB, int NW, int SC>
hipError_t launch_dg(const LayerGemvArgs& a, int n_blocks, hipStream_t st) {
  hipLaunchKernelGGL((dgemv_kernel<T, NW, SC, NORM, EPI, TPB>), dim3((unsigned)n_blocks),
                     dim3(64 * NW), 0, st, a);
  return hipGetLastError();
}

template <typename T, bool NORM, int EPI, int TPB>
hipError_t dispatch_dg_k(const LayerGemvArgs& a, int n_blocks, hipStream_t st) {
  switch (a.K) {
    case 512: return launch_dg<T, NORM, EPI, TPB, 4, 1>(a, n_blocks, st);
    case 1024: return launch_dg<T, NORM, EPI, TPB, 8, 1>(a, n_blocks, st);
    case 1536: return launch_dg<T, NORM, EPI, TPB, 12, 1>(a, n_blocks, st);
    // K = 2048 (the 1B model's projections from the residual stream): fewer,
    // longer waves pay the per-wave set-up, RMSNorm statistics and cross-wave
    // reduction less often.  One MI355X, M = 8, per call in a 16-layer graph:
    // wo + residual 4.03 -> 3.75 us (16 x 1 -> 4 x 4), w1|w3 + SwiGLU 11.2 ->
    // 9.9 us (8 x 2), RMSNorm + QKV + RoPE + append about 0.85 us less (4 x 4).
    case 2048:
      if constexpr (EPI == kEpiSwiglu) return launch_dg<T, NORM, EPI, TPB, 8, 2>(a, n_blocks, st);
      else return launch_dg<T, NORM, EPI, TPB, 4, 4>(a, n_blocks, st);
    case 3072: return launch_dg<T, NORM, EPI, TPB, 12, 2>(a, n_blocks, st);
    case 4096: return launch_dg<T, NORM, EPI, TPB, 16, 2>(a, n_blocks, st);
    default: break;
  }
  if constexpr (EPI != kEpiSwiglu) {  // two weight streams: K <= 4096 (host-checked)
    switch (a.K) {
      case 6144: return launch_dg<T, NORM, EPI, TPB, 16, 3>(a, n_blocks, st);
      case 8192: return launch_dg<T, NORM, EPI, TPB, 16, 4>(a, n_blocks, st);
      default: break;
    }
  }
  return hipErrorInvalidValue;
}

template <typename T, int EPI, int TPB>
hipError_t dispatch_dg(const LayerGemvArgs& a, int n_blocks, hipStream_t st) {
  return a.norm_w != nullptr ? dispatch_dg_k<T, true, EPI, TPB>(a, n_blocks, st)
                             : dispatch_dg_k<T, false, EPI, TPB>(a, n_blocks, st);
}

// Store / residual / SwiGLU projections: the diagonal-packed kernel for M <= 8
// (one 8-row tile per block; SwiGLU two tiles of each matrix), else the 16-row
// kernel.
template <typename T, int EPI>
hipError_t dispatch_linear(const LayerGemvArgs& a, hipStream_t st) {
  if (a.M <= 8) {
    constexpr int TPB = EPI == kEpiSwiglu ? 2 : 1;
    return dispatch_dg<T, EPI, TPB>(a, (a.N + 8 * TPB - 1) / (8 * TPB), st);
  }
  return dispatch_rows<T, EPI>(a, (a.N + 15) / 16, st);
}

bool k_supported(int64_t K) {
  return K == 512 || K == 1024 || K == 1536 || K == 2048 || K == 3072 || K == 4096 ||
         K == 6144 || K == 8192;
}

int32_t check_x(const void* x, int64_t M, int64_t K, int64_t x_sm, const void* norm_w,
                int32_t dtype, const char* what) {
  if (x == nullptr) {
    set_last_error("%s: null x", what);
    return MI_ERR_INVALID;
  }
  if (dtype != MI_DTYPE_BF16 && dtype != MI_DTYPE_F16) {
    set_last_error("%s: activations must be bf16 or fp16 (dtype %d)", what, (int)dtype);
    return MI_ERR_UNSUPPORTED;
  }
  if (M < 1 || M > 16 || !k_supported(K)) {
    set_last_error("%s: need 1 <= M <= 16 and K in {512, 1024, 1536, 2048, 3072, 4096, 6144, "
                   "8192} (M=%lld K=%lld)", what, (long long)M, (long long)K);
    return MI_ERR_UNSUPPORTED;
  }
  if ((uintptr_t)x % 16 != 0 || (x_sm * 2) % 16 != 0) {
    set_last_error("%s: x rows must be 16-byte aligned", what);
    return MI_ERR_INVALID;
  }
  if (x_sm < 0 || ((M - 1) * x_sm + K) * 2 >= ((int64_t)1 << 31)) {
    set_last_error("%s: x row stride %lld out of range (x must span < 2 GB)", what,
                   (long long)x_sm);
    return MI_ERR_UNSUPPORTED;
  }
  if (norm_w != nullptr && ((uintptr_t)norm_w % 16 != 0 || M * K * 2 > 64 * 1024 ||
                            (M > 8 && K > 2048))) {
    set_last_error("%s: RMSNorm prologue needs a 16-byte aligned weight, M*K*2 <= 64 KB and "
                   "K <= 2048 for M > 8", what);
    return MI_ERR_UNSUPPORTED;
  }
  return MI_OK;
}

int32_t check_w(const int8_t* w, const void* s, int64_t w_sn, int64_t rows, int64_t K,
                const char* what) {
  if (w == nullptr || s == nullptr) {
    set_last_error("%s: null weight or scales", what);
    return MI_ERR_INVALID;
  }
  if ((uintptr_t)w % 16 != 0 || w_sn % 16 != 0) {
    set_last_error("%s: weight rows must be 16-byte aligned", what);
    return MI_ERR_UNSUPPORTED;
  }
  // weight loads use 32-bit byte offsets into the matrix
  if (w_sn < 0 || (rows - 1) * w_sn + K >= ((int64_t)1 << 31)) {
    set_last_error("%s: weight matrix out of range (%lld rows x %lld-byte stride must span "
                   "< 2 GB)", what, (long long)rows, (long long)w_sn);
    return MI_ERR_UNSUPPORTED;
  }
  return MI_OK;
}

}  // namespace
}  // namespace mi

using namespace mi;

extern "C" int32_t mi_w8a16_linear_fused(
    const void* x, int64_t x_sm, const void* norm_w, float eps, const int8_t* w_a,
    const void* s_a, int64_t w_sn_a, const int8_t* w_b, const void* s_b, int64_t w_sn_b,
    const void* res, int64_t res_sm, void* y, int64_t y_sm, int64_t M, int64_t N, int64_t K,
    int32_t epilogue, int32_t dtype, void* stream) {
  const char* what = "w8a16_linear_fused";
  int32_t st = check_x(x, M, K, x_sm, norm_w, dtype, what);
  if (st != MI_OK) return st;
  if ((st = check_w(w_a, s_a, w_sn_a, N, K, what)) != MI_OK) return st;
  if (y == nullptr || N < 1 || N > INT32_MAX - 16) {
    set_last_error("%s: null output or bad N (%lld)", what, (long long)N);
    return MI_ERR_INVALID;
  }
  if (epilogue == kEpiResidual && res == nullptr) {
    set_last_error("%s: residual epilogue needs res", what);
    return MI_ERR_INVALID;
  }
  if (epilogue == kEpiSwiglu && (st = check_w(w_b, s_b, w_sn_b, N, K, what)) != MI_OK) return st;
  if (epilogue == kEpiSwiglu && K > 4096) {
    set_last_error("%s: the SwiGLU epilogue supports K <= 4096 (K=%lld)", what,
                   (long long)K);
    return MI_ERR_UNSUPPORTED;
  }
  if (epilogue != kEpiStore && epilogue != kEpiResidual && epilogue != kEpiSwiglu) {
    set_last_error("%s: unknown epilogue %d", what, (int)epilogue);
    return MI_ERR_INVALID;
  }
  LayerGemvArgs a{};
  a.x = x; a.norm_w = norm_w; a.eps = eps;
  a.w0 = w_a; a.s0 = s_a; a.w_sn0 = w_sn_a;
  a.w1 = w_b; a.s1 = s_b; a.w_sn1 = w_sn_b;
  a.y = y; a.res = res; a.x_sm = x_sm; a.y_sm = y_sm; a.res_sm = res_sm;
  a.M = (int32_t)M; a.K = (int32_t)K; a.N = (int32_t)N;
  hipStream_t s = (hipStream_t)stream;
  hipError_t e;
  if (dtype == MI_DTYPE_BF16) {
    e = epilogue == kEpiStore ? dispatch_linear<bf16_t, kEpiStore>(a, s)
        : epilogue == kEpiResidual ? dispatch_linear<bf16_t, kEpiResidual>(a, s)
                                   : dispatch_linear<bf16_t, kEpiSwiglu>(a, s);
  } else {
    e = epilogue == kEpiStore ? dispatch_linear<f16_t, kEpiStore>(a, s)
        : epilogue == kEpiResidual ? dispatch_linear<f16_t, kEpiResidual>(a, s)
                                   : dispatch_linear<f16_t, kEpiSwiglu>(a, s);
  }
  if (e != hipSuccess) {
    set_last_error("%s: launch failed: %s", what, hipGetErrorString(e));
    return (int32_t)e;
  }
  return MI_OK;
}

extern "C" int32_t mi_w8a16_qkv_rope_append(
    const void* x, int64_t x_sm, const void* norm_w, float eps, const int8_t* wq,
    const void* sq, int64_t wq_sn, const int8_t* wk, const void* sk, int64_t wk_sn,
    const int8_t* wv, const void* sv, int64_t wv_sn, const void* cos, const void* sin,
    int64_t c_ss, int64_t rope_row0, int64_t rope_rows, const int64_t* pos, void* q_out,
    void* cache_k, void* cache_v,
    int64_t c_sb, int64_t c_sh, int64_t c_st, int64_t capacity, int64_t M, int64_t K,
    int64_t n_heads, int64_t n_kv_heads, int64_t head_dim, int32_t dtype, void* stream) {
  const char* what = "w8a16_qkv_rope_append";
  int32_t st = check_x(x, M, K, x_sm, norm_w, dtype, what);
  if (st != MI_OK) return st;
  if ((st = check_w(wq, sq, wq_sn, n_heads * head_dim, K, what)) != MI_OK) return st;
  if ((st = check_w(wk, sk, wk_sn, n_kv_heads * head_dim, K, what)) != MI_OK) return st;
  if ((st = check_w(wv, sv, wv_sn, n_kv_heads * head_dim, K, what)) != MI_OK) return st;
  if (cos == nullptr || sin == nullptr || pos == nullptr || q_out == nullptr ||
      cache_k == nullptr || cache_v == nullptr || rope_rows < 1 || c_ss < head_dim / 2) {
    set_last_error("%s: null rope table, position, output or cache pointer", what);
    return MI_ERR_INVALID;
  }
  if (head_dim < 16 || head_dim % 16 != 0 || n_heads < 1 || n_kv_heads < 1 ||
      n_heads % n_kv_heads != 0 || capacity < 1 || n_heads * head_dim > INT32_MAX / 2) {
    set_last_error("%s: unsupported heads (%lld/%lld) or head_dim %lld", what,
                   (long long)n_heads, (long long)n_kv_heads, (long long)head_dim);
    return MI_ERR_UNSUPPORTED;
  }
  LayerGemvArgs a{};
  a.x = x; a.norm_w = norm_w; a.eps = eps;
  a.w0 = wq; a.s0 = sq; a.w_sn0 = wq_sn;
  a.w1 = wk; a.s1 = sk; a.w_sn1 = wk_sn;
  a.w2 = wv; a.s2 = sv; a.w_sn2 = wv_sn;
  a.y = q_out; a.x_sm = x_sm;
  a.M = (int32_t)M; a.K = (int32_t)K; a.N = (int32_t)(n_heads * head_dim);
  a.cos = cos; a.sin = sin; a.c_ss = c_ss; a.rope_row0 = rope_row0; a.rope_rows = rope_rows;
  a.pos = pos;
  a.ck = cache_k; a.cv = cache_v; a.c_sb = c_sb; a.c_sh = c_sh; a.c_st = c_st;
  a.capacity = capacity;
  a.Hq = (int32_t)n_heads; a.Hkv = (int32_t)n_kv_heads; a.D = (int32_t)head_dim;
  hipStream_t s = (hipStream_t)stream;
  hipError_t e;
  if (M <= 8) {
    // diagonal-packed kernel: 8-row tiles of 4 rotation pairs
    const int tph = (int)(head_dim / 8);
    a.n_tiles0 = (int32_t)(n_heads * tph);
    a.n_tiles1 = (int32_t)(n_kv_heads * tph);
    const int n_tiles = a.n_tiles0 + 2 * a.n_tiles1, cus = device_cu_count();
    if (n_tiles > cus) {
      // tiles in pairs (see dgemv_kernel): wq's first, and wk's / wv's as well
      // when that alone leaves more blocks than CUs.  One MI355X, M = 8, K =
      // 2048, 16-call graph: Llama-3.2-1B (384 tiles -> 256 blocks) 6.34 ->
      // 5.29 us per call
      const int per0 = (a.n_tiles0 + 1) / 2;
      a.pair_kv = per0 + 2 * a.n_tiles1 > cus ? 1 : 0;
      const int n_blocks = per0 + 2 * (a.pair_kv ? (a.n_tiles1 + 1) / 2 : a.n_tiles1);
      e = dtype == MI_DTYPE_BF16 ? dispatch_dg<bf16_t, kEpiQkvRope, 2>(a, n_blocks, s)
                                 : dispatch_dg<f16_t, kEpiQkvRope, 2>(a, n_blocks, s);
    } else {
      e = dtype == MI_DTYPE_BF16 ? dispatch_dg<bf16_t, kEpiQkvRope, 1>(a, n_tiles, s)
                                 : dispatch_dg<f16_t, kEpiQkvRope, 1>(a, n_tiles, s);
    }
  } else {
    const int tph = (int)(head_dim / 16);   // tiles (8 rotation pairs each) per head
    a.n_tiles0 = (int32_t)(n_heads * tph);
    a.n_tiles1 = (int32_t)(n_kv_heads * tph);
    const int n_tiles = a.n_tiles0 + 2 * a.n_tiles1;
    e = dtype == MI_DTYPE_BF16 ? dispatch_rows<bf16_t, kEpiQkvRope>(a, n_tiles, s)
                               : dispatch_rows<f16_t, kEpiQkvRope>(a, n_tiles, s);
  }
  if (e != hipSuccess) {
    set_last_error("%s: launch failed: %s", what, hipGetErrorString(e));
    return (int32_t)e;
  }
  return MI_OK;
}
