// W8A16 GEMM for prefill: y[m, n] = (sum_k x[m, k] * q[n, k]) * s[n], any M.
//
// Math of the reference's GEMM kernel (src/quant_linear.py:123-188): the int8
// weight is converted to the activation dtype (exact, |q| <= 128), products are
// accumulated in fp32, the per-row scale is applied once to the finished sum
// (:180-183) and the result is rounded to x's dtype.  The reference dispatches
// to it when the flattened input has more than 8 rows (:273).
//
// MI355X design.  At prefill sizes (M in the thousands) the product is
// MFMA-bound: a 128 x 256 (m x n) output tile per workgroup of 4 waves, 64-deep
// k stages, v_mfma_f32_32x32x16_{bf16,f16} with fp32 accumulators, two
// workgroups per CU (two waves per SIMD, so one wave's VALU and LDS work issues
// under the other's MFMAs).
//  * Each wave owns 64 output columns (n) and all 128 rows (m).  The activation
//    tile is shared by the 4 waves and copied global->LDS by DMA
//    (global_load_lds_dwordx4: no VGPRs, no VALU); the int8 weight fragments
//    are private to a wave and go straight from global memory to registers
//    (a wave's 64 rows x 64 k = 4 KB per stage).  Both are fetched one stage
//    ahead.
//  * The weight is widened to the activation dtype in registers right before
//    the MFMAs; every widened fragment feeds 4 MFMAs: 1.5 VALU ops per element
//    = 3 per 32x32x16 MFMA.
//  * The weight rows are the MFMA A operand and the activation rows the B
//    operand, so each lane's accumulators hold 4 consecutive output columns
//    of one row (8-byte stores).
//  * The k order inside a 64-deep stage is permuted identically for both
//    operands: the lane of half h feeds k = 32h + 8j .. 32h + 8j + 7 to MFMA
//    step j, so it reads 32 contiguous k of a row (two 16-byte loads of the
//    weight row, four 16-byte LDS reads of the activation row).  The sum is
//    over the same k.
//  * Activation rows are XOR-swizzled by 16-byte chunk in LDS so those reads
//    are free of bank conflicts; the DMA realises the swizzle by choosing which
//    chunk each lane fetches (a DMA wave instruction writes 1 KB contiguously).
//  * The 256 column scales are staged in LDS at the start, so the epilogue has
//    no dependent global loads.
//  * Tiles are ordered so that concurrently resident workgroups of one XCD
//    (blocks are dealt to the 8 XCDs round-robin) cover a patch of 8 m-tiles
//    and share their operand rows in that XCD's L2.
#include <type_traits>

#include "common.hpp"

namespace mi {

struct GemmArgs {
  const unsigned char* x;  // [M, K] activations (unit k stride), rows x_sm elements apart
  const unsigned char* w;  // [N, K] int8, rows w_sn bytes apart
  const void* scales;      // [N] (element stride s_sn)
  void* y;                 // [M, N] (unit n stride), rows y_sm elements apart
  int64_t x_sm, w_sn, s_sn, y_sm;
  int32_t M, N, K;
  int32_t tiles_m, tiles_n;
  int32_t y_vec;           // rows of y allow 8-byte stores of 4 columns
  // split-K: workgroup (tile, split) sums stages [split * split_stages, +split_stages)
  // into part[split][m][n] (fp32, rows of N); one split = the whole K
  float* part;
  int32_t split_stages;
  int32_t part_vec;        // part rows allow 16-byte stores of 4 columns
  int32_t y_line;          // y and its rows are 16-byte aligned (whole-line epilogue)
  // SwiGLU form: y = silu(x w^T * s) * (x w3^T * s3), each product rounded to
  // the activation dtype first (w3 / scales3 / strides as w / scales)
  const unsigned char* w3;
  const void* scales3;
  int64_t w3_sn, s3_sn;
  // residual form (res != nullptr): y = round(res + round(x w^T * s)), res [M, N]
  // in the activation dtype with unit column stride, rows res_sm elements apart
  const void* res;
  int64_t res_sm;
  int32_t res_line;        // res and its rows are 16-byte aligned
};

// 8 activation-dtype values a and b (16 bytes each): round(a + b) per element
template <typename T>
__device__ inline u32x4 add8(const u32x4& a, const u32x4& b) {
  float fa[8], fb[8];
  Chunk<T>::unpack(a, fa);
  Chunk<T>::unpack(b, fb);
  typedef T t8 __attribute__((ext_vector_type(8)));
  t8 o;
#pragma unroll
  for (int e = 0; e < 8; ++e) o[e] = Elem<T>::from_f32(fa[e] + fb[e]);
  return __builtin_bit_cast(u32x4, o);
}

constexpr int kGmBM = 128;                      // output rows (m) per workgroup
constexpr int kGmBN = 256;                      // output columns (n) per workgroup
constexpr int kGmBK = 64;                       // k per stage
constexpr int kGmXBytes = kGmBM * kGmBK * 2;    // activation tile per stage, 16 KB
constexpr int kGmXDma = kGmXBytes / 1024 / 4;   // 1 KB DMA instructions per wave and stage
constexpr int kGmGroupM = 8;                    // m-tiles per tile group
// LDS: two activation stages, then the workgroup's column scales (fp32)
constexpr size_t kGmLdsBytes = 2 * kGmXBytes + kGmBN * sizeof(float);

// silu(x) = x / (1 + e^-x) with the hardware exp2 and reciprocal (a few ulp
// of fp32; the SwiGLU epilogue rounds it to the activation dtype right after)
__device__ inline float silu_fast(float x) {
  return x * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-x * 1.44269504f));
}

// chunk swizzle of activation row r (8 chunks of 16 bytes per row)
__device__ inline int gm_xswz(int r) { return ((r >> 1) ^ (r << 2)) & 7; }

template <typename T> struct GemmOps;
template <> struct GemmOps<bf16_t> {
  typedef __bf16 v8 __attribute__((ext_vector_type(8)));
  __device__ static inline f32x16 mma(const v8& a, const v8& b, const f32x16& c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
  }
  // upper halves of two fp32 values whose low 16 bits are zero
  __device__ static inline uint32_t hi2(float lo, float hi) {
    return __builtin_amdgcn_perm(__float_as_uint(hi), __float_as_uint(lo), 0x07060302u);
  }
  // 8 int8 (two words) -> 8 bf16, exact: each byte is sign-extended and
  // converted to fp32 (one SDWA op); integers of magnitude <= 128 have 8
  // significant bits, so the fp32 upper halves are the bf16 values.
  __device__ static inline v8 widen(uint32_t lo, uint32_t hi) {
    u32x4 r;
    r.x = hi2((float)(int8_t)lo, (float)(int8_t)(lo >> 8));
    r.y = hi2((float)(int8_t)(lo >> 16), (float)(int8_t)(lo >> 24));
    r.z = hi2((float)(int8_t)hi, (float)(int8_t)(hi >> 8));
    r.w = hi2((float)(int8_t)(hi >> 16), (float)(int8_t)(hi >> 24));
    return __builtin_bit_cast(v8, r);
  }
};
template <> struct GemmOps<f16_t> {
  typedef _Float16 v8 __attribute__((ext_vector_type(8)));
  typedef _Float16 h2 __attribute__((ext_vector_type(2)));
  __device__ static inline f32x16 mma(const v8& a, const v8& b, const f32x16& c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
  }
  // two bytes of u (= q ^ 0x80 = q + 128) -> fp16 pair 1024 + u (bit pattern
  // 0x6400 | u), minus 1152 -> q exactly (fp16 spacing is 1 in [1024, 2048)).
  __device__ static inline uint32_t pair(uint32_t u, uint32_t sel) {
    const h2 v = __builtin_bit_cast(h2, __builtin_amdgcn_perm(0x64646464u, u, sel));
    return __builtin_bit_cast(uint32_t, v - h2{(_Float16)1152.f, (_Float16)1152.f});
  }
  __device__ static inline v8 widen(uint32_t lo, uint32_t hi) {
    lo ^= 0x80808080u;
    hi ^= 0x80808080u;
    u32x4 r;
    r.x = pair(lo, 0x04010400u);
    r.y = pair(lo, 0x04030402u);
    r.z = pair(hi, 0x04010400u);
    r.w = pair(hi, 0x04030402u);
    return __builtin_bit_cast(v8, r);
  }
};

// Tile of a linear workgroup id: ids dealt round-robin to the 8 XCDs are first
// regrouped so that each XCD's ids are consecutive, then consecutive ids walk
// groups of kGmGroupM m-tiles, m fastest.
__device__ inline void gm_tile(int tiles_m, int tiles_n, int b, int& tm, int& tn) {
  const int G = tiles_m * tiles_n;
  if ((G & 7) == 0) b = (b & 7) * (G >> 3) + (b >> 3);
  const int group = kGmGroupM * tiles_n;
  const int g = b / group, first = g * kGmGroupM;
  const int gm = min(tiles_m - first, kGmGroupM);
  const int in = b - g * group;
  tm = first + in % gm;
  tn = in / gm;
}

// One workgroup's 128 x 256 output tile (tm, tn) of the GEMM described by a
// (split-K: the k stages of `split`).  SWIGLU: the tile is 128 columns of the
// gated product, its 256 weight rows the 128 matching rows of w and of w3
// (each wave: 32 rows of each), combined in the epilogue.
template <typename T, typename ST, bool PARTIAL, bool SWIGLU = false>
__device__ __forceinline__ void gemm_tile_body(const GemmArgs& a, int tm, int tn, int split) {
  static_assert(!(PARTIAL && SWIGLU), "the SwiGLU epilogue needs the whole K");
  using OP = GemmOps<T>;
  typedef typename OP::v8 v8;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // the wave's 64 columns
  const int r = lane & 31, h = lane >> 5;
  const int m0 = tm * kGmBM, n0 = tn * (SWIGLU ? kGmBN / 2 : kGmBN);

  // the workgroup's 256 column scales as fp32, staged in LDS after the first
  // stage's copies are issued (read by the epilogue; published by the main
  // loop's first barrier)
  ST sc_raw;
  if constexpr (SWIGLU) {   // [0, 128): w's scales, [128, 256): w3's
    const bool hi = threadIdx.x >= kGmBN / 2;
    const int c = min(n0 + (int)(threadIdx.x & (kGmBN / 2 - 1)), a.N - 1);
    sc_raw = hi ? reinterpret_cast<const ST*>(a.scales3)[(int64_t)c * a.s3_sn]
                : reinterpret_cast<const ST*>(a.scales)[(int64_t)c * a.s_sn];
  } else {
    sc_raw = reinterpret_cast<const ST*>(a.scales)[(int64_t)min(n0 + (int)threadIdx.x, a.N - 1) * a.s_sn];
  }
  float* const sc_lds = reinterpret_cast<float*>(smem_raw + 2 * kGmXBytes);

  // ---- activation DMA: instruction i of wave wv copies tile rows
  // 8 (4 wv + i) .. + 8; lane t fetches logical chunk (t % 8) ^ swz(row) of
  // row t / 8 (byte offsets relative to the stage's first column).
  uint32_t x_off[kGmXDma];
#pragma unroll
  for (int i = 0; i < kGmXDma; ++i) {
    const int row = 8 * (kGmXDma * wv + i) + (lane >> 3);
    const int c = (lane & 7) ^ gm_xswz(row);
    const int gm = min(m0 + row, a.M - 1);                 // rows past M: clamped, never stored
    x_off[i] = (uint32_t)((int64_t)(gm - m0) * a.x_sm * 2 + c * 16);
  }
  const unsigned char* x_base = a.x + (int64_t)m0 * a.x_sm * 2;
  const uint32_t lds0 = lds_addr(smem_raw);
  const int s_begin = PARTIAL ? split * a.split_stages : 0;
  const int nk = PARTIAL ? min(s_begin + a.split_stages, a.K / kGmBK) : a.K / kGmBK;
  auto issue_x = [&](int s) {
    const uint32_t xl = lds0 + (s & 1) * kGmXBytes;
    const unsigned char* xb = x_base + (int64_t)s * kGmBK * 2;
#pragma unroll
    for (int i = 0; i < kGmXDma; ++i) lds_dma16(xb, x_off[i], xl + (kGmXDma * wv + i) * 1024);
  };

  // ---- weight fragments: lane (r, h) of fragment nf loads the 32 k
  // 32h .. 32h + 31 of the stage from weight row n0 + 64 wv + 32 nf + r (rows
  // past N clamped, never stored).
  const unsigned char* w_row[2];
#pragma unroll
  for (int nf = 0; nf < 2; ++nf) {
    if constexpr (SWIGLU)   // fragment 0 from w, 1 from w3: the same 32 output columns
      w_row[nf] = (nf ? a.w3 : a.w) + (int64_t)min(n0 + 32 * wv + r, a.N - 1) * (nf ? a.w3_sn : a.w_sn) + 32 * h;
    else
      w_row[nf] = a.w + (int64_t)min(n0 + 64 * wv + 32 * nf + r, a.N - 1) * a.w_sn + 32 * h;
  }
  auto load_w = [&](int s, u32x4 (&q)[2][2]) {
#pragma unroll
    for (int nf = 0; nf < 2; ++nf)
#pragma unroll
      for (int e = 0; e < 2; ++e) q[nf][e] = load16(w_row[nf] + (int64_t)s * kGmBK + 16 * e);
  };

  // ---- activation fragment mf: LDS row 32 mf + r, chunks 4h + j (j = MFMA k step)
  int x_rd[4][4];
#pragma unroll
  for (int mf = 0; mf < 4; ++mf) {
    const int row = 32 * mf + r;
#pragma unroll
    for (int j = 0; j < 4; ++j) x_rd[mf][j] = row * 128 + 16 * ((4 * h + j) ^ gm_xswz(row));
  }

  f32x16 acc[4][2];
#pragma unroll
  for (int mf = 0; mf < 4; ++mf)
#pragma unroll
    for (int nf = 0; nf < 2; ++nf)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[mf][nf][i] = 0.f;

  // One stage: stage s's activation tile is in LDS slot s % 2 and its weight
  // fragments in wc; the copies of stage s + 1 (activation DMA, weight loads
  // into wn) are issued before its MFMAs so that they land under them.
  auto step = [&](int s, u32x4 (&wc)[2][2], u32x4 (&wn)[2][2]) {
    dma_wait_all();                          // this wave's copies of stage s landed
    // wc is read here, after the wait, so the compiler's own wait for the
    // weight loads also falls here and not after the next stage's copies
    __asm__ volatile("" ::"v"(wc[0][0]), "v"(wc[0][1]), "v"(wc[1][0]), "v"(wc[1][1]));
    // every wave's part of stage s is in LDS, and every wave is done reading
    // the slot that the next copy overwrites (stage s - 1's)
    block_sync_lds();
    if (s + 1 < nk) {
      issue_x(s + 1);
      load_w(s + 1, wn);
    }
    // keep the next stage's loads ahead of this stage's MFMAs
    __builtin_amdgcn_sched_barrier(0);
    const unsigned char* st = smem_raw + (s & 1) * kGmXBytes;
    v8 xa[4][4];
#pragma unroll
    for (int mf = 0; mf < 4; ++mf)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        xa[mf][j] = __builtin_bit_cast(v8, *reinterpret_cast<const u32x4*>(st + x_rd[mf][j]));
#pragma unroll
    for (int j = 0; j < 4; ++j) {
#pragma unroll
      for (int nf = 0; nf < 2; ++nf) {
        const u32x4& q = wc[nf][j >> 1];
        const v8 wb = (j & 1) ? OP::widen(q.z, q.w) : OP::widen(q.x, q.y);
#pragma unroll
        for (int mf = 0; mf < 4; ++mf) acc[mf][nf] = OP::mma(wb, xa[mf][j], acc[mf][nf]);
      }
    }
  };

  // two register sets for the weight fragments, alternating by stage
  u32x4 wa[2][2], wb[2][2];
  issue_x(s_begin);
  load_w(s_begin, wa);
  sc_lds[threadIdx.x] = Elem<ST>::to_f32(sc_raw);
  int s = s_begin;
  for (; s + 1 < nk; s += 2) {
    step(s, wa, wb);
    step(s + 1, wb, wa);
  }
  if (s < nk) step(s, wa, wb);

  // ---- epilogue: acc[mf][nf][4 g + i] = C[n][m] with
  // n = n0 + 64 wv + 32 nf + 8 g + 4 h + i, m = m0 + 32 mf + r
  if constexpr (PARTIAL) {
    // unscaled fp32 sums of this split's k range
    float* pp = a.part + (int64_t)split * a.M * a.N;
#pragma unroll
    for (int nf = 0; nf < 2; ++nf)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int nb = n0 + 64 * wv + 32 * nf + 8 * g + 4 * h;
#pragma unroll
        for (int mf = 0; mf < 4; ++mf) {
          const int m = m0 + 32 * mf + r;
          if (m >= a.M) continue;
          float* q = pp + (int64_t)m * a.N + nb;
          if (a.part_vec && nb + 3 < a.N) {
            *reinterpret_cast<f32x4*>(q) = f32x4{acc[mf][nf][4 * g], acc[mf][nf][4 * g + 1],
                                                 acc[mf][nf][4 * g + 2], acc[mf][nf][4 * g + 3]};
          } else {
#pragma unroll
            for (int i = 0; i < 4; ++i)
              if (nb + i < a.N) q[i] = acc[mf][nf][4 * g + i];
          }
        }
      }
    return;
  }
  T* y = reinterpret_cast<T*>(a.y);
  if constexpr (SWIGLU) {
    // acc[mf][0] / acc[mf][1]: w / w3 products of the same 4 columns per g,
    // rounded where the unfused chain rounds: y1, y3, silu(y1), the product
    // (silu with the hardware exp2 and reciprocal: within an ulp of the
    // chain's bits)
    auto rnd = [](float v) { return Elem<T>::to_f32(Elem<T>::from_f32(v)); };
    typedef T t4 __attribute__((ext_vector_type(4)));
    auto gate4 = [&](int mf, int g, const f32x4& s1, const f32x4& s3) {
      t4 v;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float y1 = rnd(acc[mf][0][4 * g + i] * s1[i]);
        const float y3 = rnd(acc[mf][1][4 * g + i] * s3[i]);
        v[i] = Elem<T>::from_f32(rnd(silu_fast(y1)) * y3);
      }
      return v;
    };
    if (a.y_line && n0 + kGmBN / 2 <= a.N) {
      // whole-line stores as below: each wave stages its 32 columns of 32
      // rows at a time and writes a row's 64 bytes with 4 lanes x 16 bytes
      constexpr int RS = 80;                 // staged row stride (bytes, padded)
      block_sync_lds();
      unsigned char* const stg = smem_raw + wv * 32 * RS;
      f32x4 s1[4], s3[4];
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        s1[g] = *reinterpret_cast<const f32x4*>(sc_lds + 32 * wv + 8 * g + 4 * h);
        s3[g] = *reinterpret_cast<const f32x4*>(sc_lds + kGmBN / 2 + 32 * wv + 8 * g + 4 * h);
      }
#pragma unroll
      for (int mf = 0; mf < 4; ++mf) {
#pragma unroll
        for (int g = 0; g < 4; ++g)
          *reinterpret_cast<t4*>(stg + r * RS + (8 * g + 4 * h) * 2) = gate4(mf, g, s1[g], s3[g]);
        __asm__ volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // the wave's own rows are staged
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const int rr = 16 * i + (lane >> 2), cc = lane & 3;
          const u32x4 v = *reinterpret_cast<const u32x4*>(stg + rr * RS + cc * 16);
          const int m = m0 + 32 * mf + rr;
          if (m < a.M)
            *reinterpret_cast<u32x4*>(y + (int64_t)m * a.y_sm + n0 + 32 * wv + 8 * cc) = v;
        }
      }
      return;
    }
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int nl = 32 * wv + 8 * g + 4 * h, nb = n0 + nl;
      const f32x4 s1 = *reinterpret_cast<const f32x4*>(sc_lds + nl);
      const f32x4 s3 = *reinterpret_cast<const f32x4*>(sc_lds + kGmBN / 2 + nl);
#pragma unroll
      for (int mf = 0; mf < 4; ++mf) {
        const int m = m0 + 32 * mf + r;
        if (m >= a.M) continue;
        const t4 v = gate4(mf, g, s1, s3);
        T* yp = y + (int64_t)m * a.y_sm + nb;
        if (a.y_vec && nb + 3 < a.N) {
          *reinterpret_cast<t4*>(yp) = v;
        } else {
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (nb + i < a.N) yp[i] = v[i];
        }
      }
    }
    return;
  }
  if (a.y_line && (a.res == nullptr || a.res_line) && n0 + kGmBN <= a.N) {
    // Whole-line stores: each wave stages its 64 columns of 32 rows at a time
    // in LDS (the activation stages, free once every wave has read the last
    // one) and writes each row's 128 bytes with 8 lanes x 16 bytes of one
    // instruction, instead of 16-byte pieces of 32 rows from 8 instructions.
    constexpr int RS = 136;                  // staged row stride (bytes, padded)
    block_sync_lds();
    unsigned char* const stg = smem_raw + wv * 32 * RS;
    typedef T t4 __attribute__((ext_vector_type(4)));
    f32x4 s4[2][4];
#pragma unroll
    for (int nf = 0; nf < 2; ++nf)
#pragma unroll
      for (int g = 0; g < 4; ++g)
        s4[nf][g] = *reinterpret_cast<const f32x4*>(sc_lds + 64 * wv + 32 * nf + 8 * g + 4 * h);
#pragma unroll
    for (int mf = 0; mf < 4; ++mf) {
#pragma unroll
      for (int nf = 0; nf < 2; ++nf)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          t4 v;
#pragma unroll
          for (int i = 0; i < 4; ++i) v[i] = Elem<T>::from_f32(acc[mf][nf][4 * g + i] * s4[nf][g][i]);
          *reinterpret_cast<t4*>(stg + r * RS + (32 * nf + 8 * g + 4 * h) * 2) = v;
        }
      __asm__ volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // the wave's own rows are staged
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int rr = 8 * i + (lane >> 3), cc = lane & 7;
        u32x4 v = *reinterpret_cast<const u32x4*>(stg + rr * RS + cc * 16);
        const int m = m0 + 32 * mf + rr;
        if (m < a.M) {
          const int64_t col = n0 + 64 * wv + 8 * cc;
          if (a.res != nullptr)
            v = add8<T>(v, load16(reinterpret_cast<const T*>(a.res) + (int64_t)m * a.res_sm + col));
          *reinterpret_cast<u32x4*>(y + (int64_t)m * a.y_sm + col) = v;
        }
      }
    }
    return;
  }
#pragma unroll
  for (int nf = 0; nf < 2; ++nf) {
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int nl = 64 * wv + 32 * nf + 8 * g + 4 * h, nb = n0 + nl;
      const f32x4 s4 = *reinterpret_cast<const f32x4*>(sc_lds + nl);
#pragma unroll
      for (int mf = 0; mf < 4; ++mf) {
        const int m = m0 + 32 * mf + r;
        if (m >= a.M) continue;
        T* yp = y + (int64_t)m * a.y_sm + nb;
        const T* rp = a.res != nullptr
                          ? reinterpret_cast<const T*>(a.res) + (int64_t)m * a.res_sm + nb
                          : nullptr;
        auto outv = [&](int i) {
          const T v = Elem<T>::from_f32(acc[mf][nf][4 * g + i] * s4[i]);
          return a.res != nullptr ? Elem<T>::from_f32(Elem<T>::to_f32(rp[i]) + Elem<T>::to_f32(v)) : v;
        };
        if (a.y_vec && nb + 3 < a.N) {
          typedef T t4 __attribute__((ext_vector_type(4)));
          t4 v;
#pragma unroll
          for (int i = 0; i < 4; ++i) v[i] = outv(i);
          *reinterpret_cast<t4*>(yp) = v;
        } else {
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (nb + i < a.N) yp[i] = outv(i);
        }
      }
    }
  }
}

template <typename T, typename ST, bool PARTIAL>
__global__ __launch_bounds__(256, 2) void w8a16_gemm_kernel(GemmArgs a) {
  // split-K: workgroup ids run over all tiles of split 0, then of split 1, ...
  const int n_tiles = a.tiles_m * a.tiles_n;
  const int split = PARTIAL ? (int)blockIdx.x / n_tiles : 0;
  int tm, tn;
  gm_tile(a.tiles_m, a.tiles_n, (int)blockIdx.x - split * n_tiles, tm, tn);
  gemm_tile_body<T, ST, PARTIAL>(a, tm, tn, split);
}

// The gated feed-forward input projection silu(x w1^T) * (x w3^T) in one
// GEMM: 128-column tiles of the product, each reading the matching rows of w1
// and w3, so neither projection is written out.
template <typename T, typename ST>
__global__ __launch_bounds__(256, 2) void w8a16_gemm_swiglu_kernel(GemmArgs a) {
  int tm, tn;
  gm_tile(a.tiles_m, a.tiles_n, (int)blockIdx.x, tm, tn);
  gemm_tile_body<T, ST, false, true>(a, tm, tn, 0);
}

// Several GEMMs of one activation x (e.g. the q, k and v projections) in one
// launch: the 128 x 256 tiles of all matrices form one grid, matrix i owning
// tile columns [col0[i], col0[i + 1]); the grid is walked in the single-GEMM
// order (XCD regrouping, groups of m-tiles), so each XCD's resident tiles
// share activation rows across the matrices.  Each tile is computed exactly
// as by w8a16_gemm_kernel on its own matrix.
constexpr int kGmMaxMats = 4;
struct GemmMultiArgs {
  GemmArgs mat[kGmMaxMats];
  int32_t col0[kGmMaxMats + 1];
  int32_t n_mats, tiles_m;
};

template <typename T, typename ST>
__global__ __launch_bounds__(256, 2) void w8a16_gemm_multi_kernel(GemmMultiArgs ma) {
  int tm, tn;
  gm_tile(ma.tiles_m, ma.col0[ma.n_mats], (int)blockIdx.x, tm, tn);
  int i = 0;
#pragma unroll
  for (int j = 1; j < kGmMaxMats; ++j)
    if (j < ma.n_mats && tn >= ma.col0[j]) i = j;
  gemm_tile_body<T, ST, false>(ma.mat[i], tm, tn - ma.col0[i], 0);
}

// Split-K finish: y[m, n] = round((sum over splits, in split order, of
// part[s][m][n]) * scale[n]); one thread per 4 consecutive columns of a row.
template <typename T, typename ST>
__global__ __launch_bounds__(256) void w8a16_splitk_reduce_kernel(GemmArgs a, int32_t splits) {
  const int64_t q4 = (a.N + 3) / 4;
  const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= (int64_t)a.M * q4) return;
  const int m = (int)(idx / q4), nb = (int)(idx - (int64_t)m * q4) * 4;
  const ST* sc = reinterpret_cast<const ST*>(a.scales);
  const int64_t plane = (int64_t)a.M * a.N;
  const float* pp = a.part + (int64_t)m * a.N + nb;
  T* yp = reinterpret_cast<T*>(a.y) + (int64_t)m * a.y_sm + nb;
  if (a.part_vec && nb + 3 < a.N) {
    f32x4 t = *reinterpret_cast<const f32x4*>(pp);
    for (int sp = 1; sp < splits; ++sp) t += *reinterpret_cast<const f32x4*>(pp + sp * plane);
    typedef T t4 __attribute__((ext_vector_type(4)));
    t4 v;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      v[i] = Elem<T>::from_f32(t[i] * Elem<ST>::to_f32(sc[(int64_t)(nb + i) * a.s_sn]));
      if (a.res != nullptr)
        v[i] = Elem<T>::from_f32(
            Elem<T>::to_f32(reinterpret_cast<const T*>(a.res)[(int64_t)m * a.res_sm + nb + i]) +
            Elem<T>::to_f32(v[i]));
    }
    if (a.y_vec) {
      *reinterpret_cast<t4*>(yp) = v;
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) yp[i] = v[i];
    }
  } else {
    for (int i = 0; i < 4 && nb + i < a.N; ++i) {
      float t = pp[i];
      for (int sp = 1; sp < splits; ++sp) t += pp[i + sp * plane];
      T v = Elem<T>::from_f32(t * Elem<ST>::to_f32(sc[(int64_t)(nb + i) * a.s_sn]));
      if (a.res != nullptr)
        v = Elem<T>::from_f32(
            Elem<T>::to_f32(reinterpret_cast<const T*>(a.res)[(int64_t)m * a.res_sm + nb + i]) +
            Elem<T>::to_f32(v));
      yp[i] = v;
    }
  }
}

// ---------------------------------------------------------------------------
// Small-M GEMM: 17 rows up to a few hundred (a chat prompt, a large decode batch).
//
// Here the weights (and the re-reads of x) decide: a 128 x 256 tile grid leaves
// CUs idle, and gemm_tile_body's one stage of prefetch exposes a memory round
// trip per 64 k when a CU has one workgroup.  So:
//  * 8 waves per workgroup, NG = 8 / KG of them side by side in n (32 columns
//    each) and KG behind each other in k (64 k of every stage), all on the same
//    BM = 32 MB rows; the tile is 32 MB x 32 NG and its k groups meet in LDS at
//    the end, in k-group order.
//  * x and the int8 weights both come by LDS DMA into a ring of S stages of
//    64 KG k (120 to 144 KB, one workgroup per CU), S - 1 of them in flight; the
//    wait counts this wave's own copies (vmcnt), one barrier per stage publishes
//    them and frees the slot that the next copy overwrites.
//  * the two operands use the widening of the large GEMM; their 16-byte chunks are
//    XOR-swizzled by the row so that an LDS read of 8 rows covers all banks.
//  * a stage's operands are read from LDS one step ahead of their MFMAs.
// What bounds it: per 128 k a CU spends about 0.4 us (widening, 12 VALU ops of a wave
// per 16 k of 32 columns, and the barrier) plus 0.17 us per 32-row block (its MFMAs and LDS
// reads).  MI355X, per call in a graph over rotating weights, against split K and
// separate silu and product launches: 300 rows SwiGLU 2 x [8192, 2048] 73.3 -> 30.7 us
// (655 TFLOP/s), [2048, 8192] + residual 31.9 -> 25.6, [2048, 2048] 21.4 -> 10.6; 48
// rows SwiGLU 2 x [8192, 3072] 44.7 -> 16.3 (3.1 TB/s), [3072, 8192] 27.7 -> 15.1.
constexpr int kMidMats = 3;
struct MidMat {
  const unsigned char* w;   // [N, K] int8, rows w_sn bytes apart
  const void* scales;       // [N], element stride s_sn
  void* y;                  // [M, N] (SwiGLU: of matrix 0 only)
  int64_t w_sn, s_sn, y_sm;
  int32_t N, col0;          // columns; first tile column of the matrix in the grid
  int32_t y_vec;            // rows of y take 8-byte stores of 4 columns
};
struct MidArgs {
  MidMat mat[kMidMats];
  const unsigned char* x;   // [M, K], rows x_sm elements apart
  const void* res;          // residual [M, N], rows res_sm elements apart, or null
  float* part;              // split-K sums [split][M][N] or null
  int64_t x_sm, res_sm;
  int32_t M, K, n_mats, tiles_m, tiles_n, split_stages, res_vec, part_vec;
};
enum : int { kMidStore = 0, kMidPartial = 1, kMidSwiglu = 2 };

template <int MB, int KG> struct MidShape {
  // k of a k group in a stage: 32 where 64 would leave two stages in the ring and
  // no registers for the operands read ahead
  static constexpr int kKP = MB > 3 ? 32 : 64;
  static constexpr int kNG = 8 / KG, kBM = 32 * MB, kBN = 32 * kNG, kBK = kKP * KG;
  static constexpr int kXBytes = kBM * kBK * 2, kWBytes = kBN * kBK;   // per stage
  static constexpr int kStage = kXBytes + kWBytes;
  static constexpr int kS = 147456 / kStage > 8 ? 8 : 147456 / kStage;
  // 1 KB copies per stage; of x a wave makes kXDma, or one less (waves 4..7 where
  // MB is odd and the x copies do not divide by 8)
  static constexpr int kXAll = kXBytes / 1024, kXDma = (kXAll + 7) / 8, kWDma = kWBytes / 1024 / 8;
  static constexpr bool kXEven = kXAll % 8 == 0;
  static constexpr size_t kLds = (size_t)kS * kStage + kBN * sizeof(float);   // + column scales
  static_assert(kS >= 2, "ring of two stages at least");
};

template <int N>
__device__ __forceinline__ void vm_wait() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

template <typename T, typename ST, int MB, int KG, int EPI>
__global__ __launch_bounds__(512) void w8a16_mid_kernel(MidArgs a) {
  using OP = GemmOps<T>;
  using SH = MidShape<MB, KG>;
  typedef typename OP::v8 v8;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const int lane = threadIdx.x & 63, r = lane & 31, h = lane >> 5;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int ng = wv % SH::kNG, kg = wv / SH::kNG;

  // ---- tile: ids dealt round-robin to the 8 XCDs become consecutive per XCD,
  //      m fastest, so that an XCD's tiles share weight rows in its L2
  const int G = a.tiles_m * a.tiles_n;
  const int split = EPI == kMidPartial ? (int)blockIdx.x / G : 0;
  int b = (int)blockIdx.x - split * G;
  {
    const int xcd = b & 7, q = G >> 3, rem = G & 7;
    b = xcd * q + min(xcd, rem) + (b >> 3);
  }
  const int tm = b % a.tiles_m, tn = b / a.tiles_m;
  int mi = 0;
  if constexpr (EPI == kMidStore) {
#pragma unroll
    for (int j = 1; j < kMidMats; ++j)
      if (j < a.n_mats && tn >= a.mat[j].col0) mi = j;
  }
  const MidMat& mt = a.mat[mi];
  constexpr int kCols = EPI == kMidSwiglu ? SH::kBN / 2 : SH::kBN;   // output columns
  const int m0 = tm * SH::kBM, n0 = (tn - (EPI == kMidStore ? mt.col0 : 0)) * kCols;

  // ---- copies of this wave: 1 KB of consecutive LDS each, lane t the 16 bytes
  //      at 16 t; the swizzle chooses which chunk of the row that is.  Rows past
  //      M or N are clamped and never stored.
  constexpr int XC = SH::kBK / 8, WC = SH::kBK / 16;   // 16-byte chunks of a row
  // chunk swizzle of a row: 8 consecutive rows' equal chunks fall in 8 different
  // 16-byte columns of the 128 bytes that LDS serves at once
  auto swz = [](int row, int chunks) { return chunks >= 8 ? row & 7 : (row >> 1) & 3; };
  uint32_t x_off[SH::kXDma], w_off[SH::kWDma];
  const unsigned char* w_base[SH::kWDma];
#pragma unroll
  for (int i = 0; i < SH::kXDma; ++i) {
    const int row = (8 * i + wv) * (64 / XC) + lane / XC;
    const int c = (lane % XC) ^ swz(row, XC);
    x_off[i] = (uint32_t)((int64_t)(min(m0 + row, a.M - 1) - m0) * a.x_sm * 2 + c * 16);
  }
#pragma unroll
  for (int i = 0; i < SH::kWDma; ++i) {
    const int row0 = (SH::kWDma * wv + i) * (64 / WC);       // wave-uniform first row
    const int row = row0 + lane / WC;
    const int c = (lane % WC) ^ swz(row, WC);
    if constexpr (EPI == kMidSwiglu) {
      // 32 rows of a wave: 16 of w1, then the same 16 output columns' rows of w3
      const MidMat& ms = a.mat[(row0 >> 4) & 1];
      const int n = min(n0 + 16 * (row >> 5) + (row & 15), mt.N - 1) - n0;
      w_base[i] = ms.w + (int64_t)n0 * ms.w_sn;
      w_off[i] = (uint32_t)((int64_t)n * ms.w_sn + c * 16);
    } else {
      w_base[i] = mt.w + (int64_t)n0 * mt.w_sn;
      w_off[i] = (uint32_t)((int64_t)(min(n0 + row, mt.N - 1) - n0) * mt.w_sn + c * 16);
    }
  }
  const unsigned char* x_base = a.x + (int64_t)m0 * a.x_sm * 2;
  const uint32_t lds0 = lds_addr(smem_raw);
  const int nk_all = a.K / SH::kBK;
  const int s0 = EPI == kMidPartial ? split * a.split_stages : 0;
  const int nk = EPI == kMidPartial ? min(s0 + a.split_stages, nk_all) : nk_all;
  auto issue = [&](int s, int slot) {
    const uint32_t l = lds0 + (uint32_t)slot * SH::kStage;
#pragma unroll
    for (int i = 0; i < SH::kWDma; ++i)
      lds_dma16(w_base[i] + (int64_t)s * SH::kBK, w_off[i],
                l + SH::kXBytes + (SH::kWDma * wv + i) * 1024);
#pragma unroll
    for (int i = 0; i < SH::kXDma; ++i)
      if (SH::kXEven || i + 1 < SH::kXDma || wv < 4)
        lds_dma16(x_base + (int64_t)s * SH::kBK * 2, x_off[i], l + (8 * i + wv) * 1024);
  };

  // ---- operand reads: weight row 32 ng + r and activation row 32 mb + r, the
  //      k of the k group: lane half h the h-th half of them
  constexpr int KJ = SH::kKP / 16, WE = SH::kKP / 32;   // MFMA k steps; weight chunks of a lane
  int w_rd[WE], x_rd[KJ];
  {
    const int row = 32 * ng + r;
#pragma unroll
    for (int e = 0; e < WE; ++e)
      w_rd[e] = SH::kXBytes + row * SH::kBK + 16 * ((2 * WE * kg + WE * h + e) ^ swz(row, WC));
#pragma unroll
    for (int j = 0; j < KJ; ++j)
      x_rd[j] = r * SH::kBK * 2 + 16 * ((2 * KJ * kg + KJ * h + j) ^ swz(r, XC));
  }

  // the tile's column scales (SwiGLU: w1's, then w3's): loaded ahead of the copies,
  // put in LDS for the epilogue after the main loop
  float* const sc_lds = reinterpret_cast<float*>(smem_raw + SH::kS * SH::kStage);
  ST sc_raw = (ST)0.f;
  if (EPI != kMidPartial && threadIdx.x < SH::kBN) {
    const MidMat& ms = a.mat[EPI == kMidSwiglu ? (threadIdx.x >= kCols) : mi];
    const int n = min(n0 + (int)(threadIdx.x % kCols), ms.N - 1);
    sc_raw = reinterpret_cast<const ST*>(ms.scales)[(int64_t)n * ms.s_sn];
  }

  f32x16 acc[MB];
#pragma unroll
  for (int mb = 0; mb < MB; ++mb)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[mb][i] = 0.f;

  // Stage s's operands are read from LDS one step before its MFMAs, so that the
  // reads (and the copies behind them) run under the MFMAs of stage s - 1: with
  // the waves in step at the barrier, reads and MFMAs would otherwise take turns.
  struct Ops { u32x4 q[WE]; v8 xa[KJ][MB]; };
  // this wave's copies landed, but for the last `later` stages' worth (a constant:
  // a chain of branches over run-time counts cost 200 cycles per stage)
  auto wait = [&](auto later) {
    constexpr int L = decltype(later)::value;
    if (SH::kXEven || wv < 4) vm_wait<L * (SH::kXDma + SH::kWDma)>();
    else vm_wait<L * (SH::kXDma + SH::kWDma - 1)>();
  };
  auto read = [&](int slot, Ops& o) {
    const unsigned char* st = smem_raw + slot * SH::kStage;
#pragma unroll
    for (int e = 0; e < WE; ++e) o.q[e] = *reinterpret_cast<const u32x4*>(st + w_rd[e]);
#pragma unroll
    for (int j = 0; j < KJ; ++j)
#pragma unroll
      for (int mb = 0; mb < MB; ++mb)
        o.xa[j][mb] = __builtin_bit_cast(
            v8, *reinterpret_cast<const u32x4*>(st + x_rd[j] + mb * 32 * SH::kBK * 2));
  };
  auto mul = [&](const Ops& o) {
#pragma unroll
    for (int j = 0; j < KJ; ++j) {
      const u32x4& q = o.q[j >> 1];
      const v8 wb = (j & 1) ? OP::widen(q.z, q.w) : OP::widen(q.x, q.y);
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) acc[mb] = OP::mma(wb, o.xa[j][mb], acc[mb]);
    }
  };
  int slot = 0;   // of stage s
  constexpr int S = SH::kS, kHalf = (S - 1) / 2;
  auto step = [&](auto steady, int s, const Ops& cur, Ops& next) {
    const int old = slot;
    slot = slot + 1 == S ? 0 : slot + 1;
    if (decltype(steady)::value || s + 1 < nk) {
      if (decltype(steady)::value) wait(std::integral_constant<int, S - 2>());
      else if (nk - 2 - s >= kHalf) wait(std::integral_constant<int, kHalf>());
      else wait(std::integral_constant<int, 0>());
      // stage s + 1 is published, and every wave has read stage s: its slot is free
      block_sync_lds();
      read(slot, next);
      if (decltype(steady)::value) issue(s + S, old);
    }
    __builtin_amdgcn_sched_barrier(0);
    mul(cur);
  };
#pragma unroll
  for (int p = 0; p < S; ++p)
    if (s0 + p < nk) issue(s0 + p, p);
  if (nk - s0 >= S) wait(std::integral_constant<int, S - 1>());
  else wait(std::integral_constant<int, 0>());
  block_sync_lds();
  Ops oa, ob;
  read(0, oa);
  int s = s0;
  for (; s + S + 1 < nk; s += 2) {   // stages s and s + 1 each have an (s + S)-th to fetch
    step(std::true_type(), s, oa, ob);
    step(std::true_type(), s + 1, ob, oa);
  }
  if (s + S < nk) {                  // one more
    step(std::true_type(), s, oa, ob);
    ++s;
    oa = ob;
  }
  for (; s + 1 < nk; s += 2) {
    step(std::false_type(), s, oa, ob);
    step(std::false_type(), s + 1, ob, oa);
  }
  if (s < nk) step(std::false_type(), s, oa, ob);

  // ---- the k groups' sums: unit (mb, g) = columns 8 g + 4 h .. + 3 of rows 32 mb + r
  //      is finished by one owner wave of the n group, which adds the KG sums in
  //      k-group order; the others hand theirs over in LDS (the ring, once every
  //      wave has read its last stage)
  auto owner = [](int mb, int g) { return KG == 2 ? (g & 1) : ((2 * mb + (g & 1)) & (KG - 1)); };
  constexpr int UPO = KG == 2 ? 2 * MB : 2;    // units of an owner
  auto unit_at = [&](int mb, int g, int src) -> f32x4* {
    const int own = owner(mb, g), local = KG == 2 ? 2 * mb + (g >> 1) : (g >> 1);
    const int k = src < own ? src : src - 1;
    return reinterpret_cast<f32x4*>(smem_raw) +
           ((((ng * KG + own) * UPO + local) * (KG - 1) + k) * 64 + lane);
  };
  block_sync_lds();
  if (EPI != kMidPartial && threadIdx.x < SH::kBN) sc_lds[threadIdx.x] = Elem<ST>::to_f32(sc_raw);
#pragma unroll
  for (int mb = 0; mb < MB; ++mb)
#pragma unroll
    for (int g = 0; g < 4; ++g)
      if (owner(mb, g) != kg)
        *unit_at(mb, g, kg) = f32x4{acc[mb][4 * g], acc[mb][4 * g + 1], acc[mb][4 * g + 2],
                                    acc[mb][4 * g + 3]};
  block_sync_lds();
  auto unit = [&](int mb, int g) -> f32x4 {
    const f32x4 own = f32x4{acc[mb][4 * g], acc[mb][4 * g + 1], acc[mb][4 * g + 2], acc[mb][4 * g + 3]};
    f32x4 t = kg == 0 ? own : *unit_at(mb, g, 0);
#pragma unroll
    for (int src = 1; src < KG; ++src) t += src == kg ? own : *unit_at(mb, g, src);
    return t;
  };

  if constexpr (EPI == kMidPartial) {
    float* pp = a.part + (int64_t)split * a.M * mt.N;
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        if (owner(mb, g) != kg) continue;
        const f32x4 t = unit(mb, g);
        const int nb = n0 + 32 * ng + 8 * g + 4 * h, m = m0 + 32 * mb + r;
        if (m >= a.M) continue;
        float* q = pp + (int64_t)m * mt.N + nb;
        if (a.part_vec && nb + 3 < mt.N) {
          *reinterpret_cast<f32x4*>(q) = t;
        } else {
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (nb + i < mt.N) q[i] = t[i];
        }
      }
    return;
  }
  typedef T t4 __attribute__((ext_vector_type(4)));
  auto rnd = [](float v) { return Elem<T>::to_f32(Elem<T>::from_f32(v)); };
  T* const y = reinterpret_cast<T*>(mt.y);
  constexpr int GO = EPI == kMidSwiglu ? 2 : 4;   // column groups of the output
#pragma unroll
  for (int g = 0; g < GO; ++g) {
    const int nb = n0 + (EPI == kMidSwiglu ? 16 : 32) * ng + 8 * g + 4 * h;
    const f32x4 s1 = *reinterpret_cast<const f32x4*>(sc_lds + nb - n0);
    f32x4 s3 = s1;
    if constexpr (EPI == kMidSwiglu) s3 = *reinterpret_cast<const f32x4*>(sc_lds + kCols + nb - n0);
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
      if (owner(mb, g) != kg) continue;
      const f32x4 t = unit(mb, g);
      t4 v;
      if constexpr (EPI == kMidSwiglu) {
        const f32x4 u = unit(mb, g + 2);   // same owner: owner() looks at g's low bit
#pragma unroll
        for (int i = 0; i < 4; ++i)
          v[i] = Elem<T>::from_f32(rnd(silu_f32(rnd(t[i] * s1[i]))) * rnd(u[i] * s3[i]));
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = Elem<T>::from_f32(t[i] * s1[i]);
      }
      const int m = m0 + 32 * mb + r;
      if (m >= a.M) continue;
      T* yp = y + (int64_t)m * mt.y_sm + nb;
      const T* rp = reinterpret_cast<const T*>(a.res) + (int64_t)m * a.res_sm + nb;
      if (mt.y_vec && nb + 3 < mt.N && (a.res == nullptr || a.res_vec)) {
        if (a.res != nullptr) {
          const t4 rv = *reinterpret_cast<const t4*>(rp);
#pragma unroll
          for (int i = 0; i < 4; ++i)
            v[i] = Elem<T>::from_f32(Elem<T>::to_f32(rv[i]) + Elem<T>::to_f32(v[i]));
        }
        *reinterpret_cast<t4*>(yp) = v;
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (nb + i < mt.N)
            yp[i] = a.res == nullptr
                        ? v[i] : Elem<T>::from_f32(Elem<T>::to_f32(rp[i]) + Elem<T>::to_f32(v[i]));
      }
    }
  }
}

}  // namespace mi

using namespace mi;

namespace {

// Argument checks shared by both entry points; fills `a` (no split).
int32_t gemm_setup(const char* what, const void* x, const int8_t* w, const void* scales,
                   void* y, int64_t m, int64_t n, int64_t k, int64_t x_sm, int64_t w_sn,
                   int64_t s_sn, int64_t y_sm, GemmArgs& a) {
  if (x == nullptr || w == nullptr || scales == nullptr || y == nullptr) {
    set_last_error("%s: null pointer", what);
    return MI_ERR_INVALID;
  }
  if (m <= 0 || n <= 0 || k <= 0 || m > INT32_MAX || n > INT32_MAX || k > INT32_MAX) {
    set_last_error("%s: need positive M, N, K below 2^31 (M=%lld N=%lld K=%lld)", what,
                   (long long)m, (long long)n, (long long)k);
    return MI_ERR_INVALID;
  }
  if (k % kGmBK != 0) {
    set_last_error("%s: K must be a multiple of %d (K=%lld)", what, kGmBK, (long long)k);
    return MI_ERR_UNSUPPORTED;
  }
  // tile-relative DMA offsets are 32-bit: 128 activation rows of x_sm elements
  if (x_sm < k || w_sn < k || y_sm < n || x_sm > (1LL << 23) || w_sn > (1LL << 23)) {
    set_last_error("%s: row strides must cover a row and be below 2^23 elements", what);
    return MI_ERR_INVALID;
  }
  if ((uintptr_t)x % 16 != 0 || (x_sm * 2) % 16 != 0 || (uintptr_t)w % 16 != 0 || w_sn % 16 != 0) {
    set_last_error("%s: x and weight rows must be 16-byte aligned", what);
    return MI_ERR_INVALID;
  }
  const int64_t tiles_m = (m + kGmBM - 1) / kGmBM, tiles_n = (n + kGmBN - 1) / kGmBN;
  if (tiles_m * tiles_n > INT32_MAX / 64) {
    set_last_error("%s: too many tiles", what);
    return MI_ERR_INVALID;
  }
  a = GemmArgs{static_cast<const unsigned char*>(x), reinterpret_cast<const unsigned char*>(w),
               scales, y, x_sm, w_sn, s_sn, y_sm, (int32_t)m, (int32_t)n, (int32_t)k,
               (int32_t)tiles_m, (int32_t)tiles_n,
               ((uintptr_t)y % 8 == 0 && y_sm % 4 == 0) ? 1 : 0,
               nullptr, (int32_t)(k / kGmBK), 0,
               ((uintptr_t)y % 16 == 0 && y_sm % 8 == 0) ? 1 : 0};
  return MI_OK;
}

bool dtypes_ok(int32_t dtype, int32_t sdtype) {
  return (dtype == MI_DTYPE_BF16 || dtype == MI_DTYPE_F16) &&
         (sdtype == MI_DTYPE_BF16 || sdtype == MI_DTYPE_F16 || sdtype == MI_DTYPE_F32);
}

template <bool PARTIAL>
void launch_gemm(const GemmArgs& a, int32_t splits, int32_t dtype, int32_t sdtype, hipStream_t st) {
  dim3 grid((unsigned)((int64_t)a.tiles_m * a.tiles_n * splits)), block(256);
#define MI_GEMM(T, ST) \
  hipLaunchKernelGGL((w8a16_gemm_kernel<T, ST, PARTIAL>), grid, block, kGmLdsBytes, st, a)
  if (dtype == MI_DTYPE_BF16 && sdtype == MI_DTYPE_BF16) MI_GEMM(bf16_t, bf16_t);
  else if (dtype == MI_DTYPE_BF16 && sdtype == MI_DTYPE_F32) MI_GEMM(bf16_t, float);
  else if (dtype == MI_DTYPE_BF16 && sdtype == MI_DTYPE_F16) MI_GEMM(bf16_t, f16_t);
  else if (dtype == MI_DTYPE_F16 && sdtype == MI_DTYPE_F16) MI_GEMM(f16_t, f16_t);
  else if (dtype == MI_DTYPE_F16 && sdtype == MI_DTYPE_F32) MI_GEMM(f16_t, float);
  else MI_GEMM(f16_t, bf16_t);
#undef MI_GEMM
}

void launch_multi(const GemmMultiArgs& ma, int32_t dtype, int32_t sdtype, hipStream_t st) {
  dim3 grid((unsigned)((int64_t)ma.tiles_m * ma.col0[ma.n_mats])), block(256);
#define MI_GEMM(T, ST) \
  hipLaunchKernelGGL((w8a16_gemm_multi_kernel<T, ST>), grid, block, kGmLdsBytes, st, ma)
  if (dtype == MI_DTYPE_BF16 && sdtype == MI_DTYPE_BF16) MI_GEMM(bf16_t, bf16_t);
  else if (dtype == MI_DTYPE_BF16 && sdtype == MI_DTYPE_F32) MI_GEMM(bf16_t, float);
  else if (dtype == MI_DTYPE_BF16 && sdtype == MI_DTYPE_F16) MI_GEMM(bf16_t, f16_t);
  else if (dtype == MI_DTYPE_F16 && sdtype == MI_DTYPE_F16) MI_GEMM(f16_t, f16_t);
  else if (dtype == MI_DTYPE_F16 && sdtype == MI_DTYPE_F32) MI_GEMM(f16_t, float);
  else MI_GEMM(f16_t, bf16_t);
#undef MI_GEMM
}

void launch_swiglu(const GemmArgs& a, int32_t dtype, int32_t sdtype, hipStream_t st) {
  dim3 grid((unsigned)((int64_t)a.tiles_m * a.tiles_n)), block(256);
#define MI_GEMM(T, ST) \
  hipLaunchKernelGGL((w8a16_gemm_swiglu_kernel<T, ST>), grid, block, kGmLdsBytes, st, a)
  if (dtype == MI_DTYPE_BF16 && sdtype == MI_DTYPE_BF16) MI_GEMM(bf16_t, bf16_t);
  else if (dtype == MI_DTYPE_BF16 && sdtype == MI_DTYPE_F32) MI_GEMM(bf16_t, float);
  else if (dtype == MI_DTYPE_BF16 && sdtype == MI_DTYPE_F16) MI_GEMM(bf16_t, f16_t);
  else if (dtype == MI_DTYPE_F16 && sdtype == MI_DTYPE_F16) MI_GEMM(f16_t, f16_t);
  else if (dtype == MI_DTYPE_F16 && sdtype == MI_DTYPE_F32) MI_GEMM(f16_t, float);
  else MI_GEMM(f16_t, bf16_t);
#undef MI_GEMM
}

void launch_reduce(const GemmArgs& a, int32_t splits, int32_t dtype, int32_t sdtype,
                   hipStream_t st) {
  const int64_t threads = (int64_t)a.M * ((a.N + 3) / 4);
  dim3 grid((unsigned)((threads + 255) / 256)), block(256);
#define MI_RED(T, ST) \
  hipLaunchKernelGGL((w8a16_splitk_reduce_kernel<T, ST>), grid, block, 0, st, a, splits)
  if (dtype == MI_DTYPE_BF16 && sdtype == MI_DTYPE_BF16) MI_RED(bf16_t, bf16_t);
  else if (dtype == MI_DTYPE_BF16 && sdtype == MI_DTYPE_F32) MI_RED(bf16_t, float);
  else if (dtype == MI_DTYPE_BF16 && sdtype == MI_DTYPE_F16) MI_RED(bf16_t, f16_t);
  else if (dtype == MI_DTYPE_F16 && sdtype == MI_DTYPE_F16) MI_RED(f16_t, f16_t);
  else if (dtype == MI_DTYPE_F16 && sdtype == MI_DTYPE_F32) MI_RED(f16_t, float);
  else MI_RED(f16_t, bf16_t);
#undef MI_RED
}

int32_t launch_status(const char* what) {
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) {
    set_last_error("%s: launch failed: %s", what, hipGetErrorString(e));
    return (int32_t)e;
  }
  return MI_OK;
}

}  // namespace

extern "C" int32_t mi_w8a16_gemm(const void* x, const int8_t* w, const void* scales, void* y,
                                 int64_t m, int64_t n, int64_t k, int64_t x_sm, int64_t w_sn,
                                 int64_t s_sn, int64_t y_sm, int32_t dtype, int32_t sdtype,
                                 void* stream) {
  GemmArgs a;
  int32_t rc = gemm_setup("w8a16_gemm", x, w, scales, y, m, n, k, x_sm, w_sn, s_sn, y_sm, a);
  if (rc != MI_OK) return rc;
  if (!dtypes_ok(dtype, sdtype)) {
    set_last_error("w8a16_gemm: activations must be bf16 or fp16 (dtype %d, scales %d)",
                   (int)dtype, (int)sdtype);
    return MI_ERR_UNSUPPORTED;
  }
  launch_gemm<false>(a, 1, dtype, sdtype, (hipStream_t)stream);
  return launch_status("w8a16_gemm");
}

// Split count for mi_w8a16_gemm_splitk (measured on MI355X): 1 (no split) once
// the 128 x 256 tiles give every CU a workgroup; otherwise about one workgroup
// per CU (at one tile per two CUs the split still gains a little: wk / wv at
// M = 8192, 37.0 -> 36.1 us), each split at least 8 stages (512 k)
// deep, at most 8 splits, and the fp32 partials (written and read once) at
// most 64 MiB.
extern "C" int64_t mi_w8a16_gemm_splits(int64_t m, int64_t n, int64_t k) {
  if (m <= 0 || n <= 0 || k <= 0 || k % kGmBK != 0) return 1;
  const int64_t tiles = ((m + kGmBM - 1) / kGmBM) * ((n + kGmBN - 1) / kGmBN);
  const int64_t cus = device_cu_count();
  if (tiles >= cus) return 1;
  int64_t s = cus / tiles;
  const int64_t nk = k / kGmBK;
  if (s > nk / 8) s = nk / 8;
  if (s > 8) s = 8;
  while (s > 1 && s * m * n * 4 > (64LL << 20)) --s;
  // splits actually used: every split gets ceil(nk / s) stages
  if (s > 1) {
    const int64_t per = (nk + s - 1) / s;
    s = (nk + per - 1) / per;
  }
  return s < 1 ? 1 : s;
}

extern "C" int32_t mi_w8a16_gemm_splitk(const void* x, const int8_t* w, const void* scales,
                                        void* y, int64_t m, int64_t n, int64_t k,
                                        int64_t x_sm, int64_t w_sn, int64_t s_sn, int64_t y_sm,
                                        float* part, int64_t part_elems, int64_t splits,
                                        int32_t dtype, int32_t sdtype, void* stream) {
  GemmArgs a;
  int32_t rc = gemm_setup("w8a16_gemm_splitk", x, w, scales, y, m, n, k, x_sm, w_sn, s_sn, y_sm, a);
  if (rc != MI_OK) return rc;
  if (!dtypes_ok(dtype, sdtype)) {
    set_last_error("w8a16_gemm_splitk: activations must be bf16 or fp16 (dtype %d, scales %d)",
                   (int)dtype, (int)sdtype);
    return MI_ERR_UNSUPPORTED;
  }
  const int64_t nk = k / kGmBK;
  if (splits < 2 || splits > nk || splits > 64) {
    set_last_error("w8a16_gemm_splitk: need 2 <= splits <= min(K / %d, 64) (splits=%lld)", kGmBK,
                   (long long)splits);
    return MI_ERR_INVALID;
  }
  const int64_t per = (nk + splits - 1) / splits;
  const int64_t used = (nk + per - 1) / per;   // splits that own at least one stage
  if (part == nullptr || part_elems < used * m * n) {
    set_last_error("w8a16_gemm_splitk: workspace needs %lld fp32 elements (given %lld)",
                   (long long)(used * m * n), (long long)part_elems);
    return MI_ERR_INVALID;
  }
  a.part = part;
  a.split_stages = (int32_t)per;
  a.part_vec = ((uintptr_t)part % 16 == 0 && n % 4 == 0) ? 1 : 0;
  hipStream_t st = (hipStream_t)stream;
  launch_gemm<true>(a, (int32_t)used, dtype, sdtype, st);
  rc = launch_status("w8a16_gemm_splitk");
  if (rc != MI_OK) return rc;
  launch_reduce(a, (int32_t)used, dtype, sdtype, st);
  return launch_status("w8a16_gemm_splitk");
}

extern "C" int32_t mi_w8a16_gemm_multi(const void* x, int64_t m, int64_t k, int64_t x_sm,
                                       int32_t n_mats, const int8_t* const* w,
                                       const void* const* scales, void* const* y,
                                       const int64_t* n, const int64_t* w_sn,
                                       const int64_t* s_sn, const int64_t* y_sm,
                                       int32_t dtype, int32_t sdtype, void* stream) {
  const char* what = "w8a16_gemm_multi";
  if (n_mats < 1 || n_mats > kGmMaxMats || w == nullptr || scales == nullptr || y == nullptr ||
      n == nullptr || w_sn == nullptr || s_sn == nullptr || y_sm == nullptr) {
    set_last_error("%s: need 1..%d matrices and non-null argument arrays (n_mats=%d)", what,
                   kGmMaxMats, (int)n_mats);
    return MI_ERR_INVALID;
  }
  if (!dtypes_ok(dtype, sdtype)) {
    set_last_error("%s: activations must be bf16 or fp16 (dtype %d, scales %d)", what,
                   (int)dtype, (int)sdtype);
    return MI_ERR_UNSUPPORTED;
  }
  GemmMultiArgs ma{};
  int64_t cols = 0;
  for (int i = 0; i < n_mats; ++i) {
    int32_t rc = gemm_setup(what, x, w[i], scales[i], y[i], m, n[i], k, x_sm, w_sn[i], s_sn[i],
                            y_sm[i], ma.mat[i]);
    if (rc != MI_OK) return rc;
    ma.col0[i] = (int32_t)cols;
    cols += ma.mat[i].tiles_n;
  }
  ma.tiles_m = ma.mat[0].tiles_m;
  if (ma.tiles_m * cols > INT32_MAX / 64) {
    set_last_error("%s: too many tiles", what);
    return MI_ERR_INVALID;
  }
  ma.col0[n_mats] = (int32_t)cols;
  ma.n_mats = n_mats;
  launch_multi(ma, dtype, sdtype, (hipStream_t)stream);
  return launch_status(what);
}

extern "C" int32_t mi_w8a16_gemm_swiglu(const void* x, const int8_t* w1, const void* scales1,
                                        const int8_t* w3, const void* scales3, void* y,
                                        int64_t m, int64_t n, int64_t k, int64_t x_sm,
                                        int64_t w1_sn, int64_t s1_sn, int64_t w3_sn,
                                        int64_t s3_sn, int64_t y_sm, int32_t dtype,
                                        int32_t sdtype, void* stream) {
  const char* what = "w8a16_gemm_swiglu";
  GemmArgs a;
  int32_t rc = gemm_setup(what, x, w1, scales1, y, m, n, k, x_sm, w1_sn, s1_sn, y_sm, a);
  if (rc != MI_OK) return rc;
  if (w3 == nullptr || scales3 == nullptr) {
    set_last_error("%s: null pointer", what);
    return MI_ERR_INVALID;
  }
  if (w3_sn < k || w3_sn > (1LL << 23) || (uintptr_t)w3 % 16 != 0 || w3_sn % 16 != 0) {
    set_last_error("%s: w3 rows must cover K, be 16-byte aligned and below 2^23 bytes apart",
                   what);
    return MI_ERR_INVALID;
  }
  if (!dtypes_ok(dtype, sdtype)) {
    set_last_error("%s: activations must be bf16 or fp16 (dtype %d, scales %d)", what,
                   (int)dtype, (int)sdtype);
    return MI_ERR_UNSUPPORTED;
  }
  a.tiles_n = (int32_t)((n + kGmBN / 2 - 1) / (kGmBN / 2));
  if ((int64_t)a.tiles_m * a.tiles_n > INT32_MAX / 64) {
    set_last_error("%s: too many tiles", what);
    return MI_ERR_INVALID;
  }
  a.w3 = reinterpret_cast<const unsigned char*>(w3);
  a.scales3 = scales3;
  a.w3_sn = w3_sn;
  a.s3_sn = s3_sn;
  launch_swiglu(a, dtype, sdtype, (hipStream_t)stream);
  return launch_status(what);
}

extern "C" int32_t mi_w8a16_gemm_residual(const void* x, const int8_t* w, const void* scales,
                                          const void* res, void* y, int64_t m, int64_t n,
                                          int64_t k, int64_t x_sm, int64_t w_sn, int64_t s_sn,
                                          int64_t res_sm, int64_t y_sm, float* part,
                                          int64_t part_elems, int64_t splits, int32_t dtype,
                                          int32_t sdtype, void* stream) {
  const char* what = "w8a16_gemm_residual";
  GemmArgs a;
  int32_t rc = gemm_setup(what, x, w, scales, y, m, n, k, x_sm, w_sn, s_sn, y_sm, a);
  if (rc != MI_OK) return rc;
  if (res == nullptr || res_sm < n) {
    set_last_error("%s: null residual or residual rows shorter than N", what);
    return MI_ERR_INVALID;
  }
  if (!dtypes_ok(dtype, sdtype)) {
    set_last_error("%s: activations must be bf16 or fp16 (dtype %d, scales %d)", what,
                   (int)dtype, (int)sdtype);
    return MI_ERR_UNSUPPORTED;
  }
  a.res = res;
  a.res_sm = res_sm;
  a.res_line = ((uintptr_t)res % 16 == 0 && res_sm % 8 == 0) ? 1 : 0;
  hipStream_t st = (hipStream_t)stream;
  if (splits <= 1) {
    launch_gemm<false>(a, 1, dtype, sdtype, st);
    return launch_status(what);
  }
  const int64_t nk = k / kGmBK;
  if (splits > nk || splits > 64) {
    set_last_error("%s: need splits <= min(K / %d, 64) (splits=%lld)", what, kGmBK,
                   (long long)splits);
    return MI_ERR_INVALID;
  }
  const int64_t per = (nk + splits - 1) / splits;
  const int64_t used = (nk + per - 1) / per;
  if (part == nullptr || part_elems < used * m * n) {
    set_last_error("%s: workspace needs %lld fp32 elements (given %lld)", what,
                   (long long)(used * m * n), (long long)part_elems);
    return MI_ERR_INVALID;
  }
  a.part = part;
  a.split_stages = (int32_t)per;
  a.part_vec = ((uintptr_t)part % 16 == 0 && n % 4 == 0) ? 1 : 0;
  launch_gemm<true>(a, (int32_t)used, dtype, sdtype, st);
  rc = launch_status(what);
  if (rc != MI_OK) return rc;
  launch_reduce(a, (int32_t)used, dtype, sdtype, st);
  return launch_status(what);
}

// ---- small-M GEMM: shape rules and launch ---------------------------------

namespace {

// k groups per workgroup: 4 (64-column tiles) up to 64 rows, where x is cheap
// to re-read and every CU should stream weights; 2 (128 columns) above.
int mid_kg(int64_t m) { return m <= 64 ? 4 : 2; }

// K granularity: a stage of the tallest-stage kernels
int mid_bk(int kg) { return 64 * kg; }

// K splits of one matrix: 2048 k per split at least, about one workgroup per CU.
int64_t mid_splits(int64_t m, int64_t n, int64_t k) {
  const int kg = mid_kg(m);
  const int64_t bn = 256 / kg, mmax = kg == 4 ? 64 : 160;
  const int64_t tiles = ((m + mmax - 1) / mmax) * ((n + bn - 1) / bn);
  int64_t s = device_cu_count() / (tiles > 0 ? tiles : 1);
  if (s > k / 2048) s = k / 2048;
  if (s > 8) s = 8;
  while (s > 1 && s * m * n * 4 > (64LL << 20)) --s;
  if (s <= 1) return 1;
  const int64_t nk = k / mid_bk(kg), per = (nk + s - 1) / s;
  return (nk + per - 1) / per;
}

// 32-row blocks per tile: the least rounds of the grid times the bytes that a
// workgroup copies per stage, over the sizes that are built.
int mid_mb(int64_t m, int64_t tiles_n, int kg) {
  const int cus = device_cu_count(), top = kg == 4 ? 2 : 5;
  int best = 1;
  int64_t cost = INT64_MAX;
  for (int mb = 1; mb <= top; ++mb) {
    const int64_t tiles = (m + 32 * mb - 1) / (32 * mb) * tiles_n;
    // a stage of 64 kg k: 4 kg KB of x for each row block, 16 KB of weights; the
    // measured stage times follow (300 rows: 0.59 us for one block, 1.28 for five)
    const int64_t c = (tiles + cus - 1) / cus * (4 * kg * mb + 16);
    if (c < cost) { cost = c; best = mb; }
  }
  return best;
}

// Tile columns of a call: of all its matrices, or of the gated product (SwiGLU).
int64_t mid_tiles_n(int kg, int32_t n_mats, const int64_t* n, int32_t epilogue) {
  const int64_t cols = epilogue == 2 ? 128 / kg : 256 / kg;
  int64_t t = 0;
  for (int i = 0; i < (epilogue == 2 ? 1 : n_mats); ++i) t += (n[i] + cols - 1) / cols;
  return t;
}

template <typename T, typename ST, int MB, int KG, int EPI>
hipError_t mid_launch(const MidArgs& a, int64_t splits, hipStream_t st) {
  using SH = MidShape<MB, KG>;
  static const hipError_t attr = hipFuncSetAttribute(
      reinterpret_cast<const void*>(w8a16_mid_kernel<T, ST, MB, KG, EPI>),
      hipFuncAttributeMaxDynamicSharedMemorySize, (int)SH::kLds);
  if (attr != hipSuccess) return attr;
  const unsigned grid = (unsigned)((int64_t)a.tiles_m * a.tiles_n * splits);
  hipLaunchKernelGGL((w8a16_mid_kernel<T, ST, MB, KG, EPI>), dim3(grid), dim3(512), SH::kLds, st, a);
  return hipGetLastError();
}

template <typename T, typename ST, int EPI>
hipError_t mid_dispatch(const MidArgs& a, int kg, int mb, int64_t splits, hipStream_t st) {
  if (kg == 4)
    return mb == 1 ? mid_launch<T, ST, 1, 4, EPI>(a, splits, st)
                   : mid_launch<T, ST, 2, 4, EPI>(a, splits, st);
  switch (mb) {
    case 1: return mid_launch<T, ST, 1, 2, EPI>(a, splits, st);
    case 2: return mid_launch<T, ST, 2, 2, EPI>(a, splits, st);
    case 3: return mid_launch<T, ST, 3, 2, EPI>(a, splits, st);
    case 4: return mid_launch<T, ST, 4, 2, EPI>(a, splits, st);
    default: return mid_launch<T, ST, 5, 2, EPI>(a, splits, st);
  }
}

template <int EPI>
hipError_t mid_dtypes(const MidArgs& a, int kg, int mb, int64_t splits, int32_t dtype,
                      int32_t sdtype, hipStream_t st) {
  if (dtype == MI_DTYPE_BF16) {
    if (sdtype == MI_DTYPE_BF16) return mid_dispatch<bf16_t, bf16_t, EPI>(a, kg, mb, splits, st);
    if (sdtype == MI_DTYPE_F16) return mid_dispatch<bf16_t, f16_t, EPI>(a, kg, mb, splits, st);
    return mid_dispatch<bf16_t, float, EPI>(a, kg, mb, splits, st);
  }
  if (sdtype == MI_DTYPE_BF16) return mid_dispatch<f16_t, bf16_t, EPI>(a, kg, mb, splits, st);
  if (sdtype == MI_DTYPE_F16) return mid_dispatch<f16_t, f16_t, EPI>(a, kg, mb, splits, st);
  return mid_dispatch<f16_t, float, EPI>(a, kg, mb, splits, st);
}

}  // namespace

extern "C" int64_t mi_w8a16_small_gemm_splits(int64_t m, int64_t n, int64_t k) {
  if (m <= 0 || n <= 0 || k <= 0) return 1;
  return mid_splits(m, n, k);
}

extern "C" int64_t mi_w8a16_small_gemm_tile_rows(int64_t m, int32_t n_mats, const int64_t* n,
                                                 int64_t k, int32_t epilogue) {
  if (m <= 0 || n_mats < 1 || n_mats > kMidMats || n == nullptr || k <= 0) return 0;
  const int kg = mid_kg(m);
  const int64_t splits = n_mats == 1 ? mid_splits(m, n[0], k) : 1;
  return 32 * mid_mb(m, mid_tiles_n(kg, n_mats, n, epilogue) * splits, kg);
}

extern "C" int32_t mi_w8a16_small_gemm(const void* x, int64_t m, int64_t k, int64_t x_sm,
                                       int32_t n_mats, const int8_t* const* w,
                                       const void* const* scales, void* const* y,
                                       const int64_t* n, const int64_t* w_sn,
                                       const int64_t* s_sn, const int64_t* y_sm,
                                       int32_t epilogue, const void* res, int64_t res_sm,
                                       float* part, int64_t part_elems, int32_t dtype,
                                       int32_t sdtype, void* stream) {
  const char* what = "w8a16_small_gemm";
  if (n_mats < 1 || n_mats > kMidMats || w == nullptr || scales == nullptr || y == nullptr ||
      n == nullptr || w_sn == nullptr || s_sn == nullptr || y_sm == nullptr) {
    set_last_error("%s: need 1..%d matrices and non-null argument arrays (n_mats=%d)", what,
                   kMidMats, (int)n_mats);
    return MI_ERR_INVALID;
  }
  if (!dtypes_ok(dtype, sdtype)) {
    set_last_error("%s: activations must be bf16 or fp16 (dtype %d, scales %d)", what,
                   (int)dtype, (int)sdtype);
    return MI_ERR_UNSUPPORTED;
  }
  // epilogue 0: y_i = x w_i^T * s_i;  1: y = res + that (one matrix);
  // 2: y_0 = silu(x w_0^T * s_0) * (x w_1^T * s_1) (two matrices of one shape)
  if (epilogue < 0 || epilogue > 2 || (epilogue == 1 && (n_mats != 1 || res == nullptr)) ||
      (epilogue == 2 && (n_mats != 2 || n[0] != n[1])) || (epilogue != 1 && res != nullptr)) {
    set_last_error("%s: epilogue %d does not fit %d matrices", what, (int)epilogue, (int)n_mats);
    return MI_ERR_INVALID;
  }
  if (m < 1 || m > 65535) {
    set_last_error("%s: need 1 <= M <= 65535 (M=%lld)", what, (long long)m);
    return MI_ERR_INVALID;
  }
  const int kg = mid_kg(m);
  if (k % mid_bk(kg) != 0) {
    set_last_error("%s: K must be a multiple of %d (K=%lld)", what, mid_bk(kg), (long long)k);
    return MI_ERR_UNSUPPORTED;
  }
  MidArgs a{};
  const int64_t tiles_n = mid_tiles_n(kg, n_mats, n, epilogue);
  for (int i = 0; i < n_mats; ++i) {
    GemmArgs g;
    void* yi = epilogue == 2 ? y[0] : y[i];
    int32_t rc = gemm_setup(what, x, w[i], scales[i], yi, m, n[i], k, x_sm, w_sn[i], s_sn[i],
                            epilogue == 2 ? y_sm[0] : y_sm[i], g);
    if (rc != MI_OK) return rc;
    a.mat[i] = MidMat{g.w, g.scales, yi, g.w_sn, g.s_sn, g.y_sm, g.N,
                      (int32_t)mid_tiles_n(kg, i, n, 0), g.y_vec};
  }
  if (epilogue == 1 && res_sm < n[0]) {
    set_last_error("%s: residual rows shorter than N", what);
    return MI_ERR_INVALID;
  }
  a.x = static_cast<const unsigned char*>(x);
  a.res = res;
  a.x_sm = x_sm;
  a.res_sm = res_sm;
  a.res_vec = res != nullptr && (uintptr_t)res % 8 == 0 && res_sm % 4 == 0 ? 1 : 0;
  a.M = (int32_t)m;
  a.K = (int32_t)k;
  a.n_mats = n_mats;
  const int64_t splits = n_mats == 1 ? mid_splits(m, n[0], k) : 1;
  if (n_mats > 1) {
    for (int i = 0; i < n_mats; ++i)
      if (mid_splits(m, n[i], k) != 1) {
        set_last_error("%s: a matrix that splits K has no fused form (N=%lld K=%lld)", what,
                       (long long)n[i], (long long)k);
        return MI_ERR_UNSUPPORTED;
      }
  }
  const int mb = (int)(mi_w8a16_small_gemm_tile_rows(m, n_mats, n, k, epilogue) / 32);
  a.tiles_m = (int32_t)((m + 32 * mb - 1) / (32 * mb));
  a.tiles_n = (int32_t)tiles_n;
  if (tiles_n * a.tiles_m * splits > INT32_MAX / 64) {
    set_last_error("%s: too many tiles", what);
    return MI_ERR_INVALID;
  }
  hipStream_t st = (hipStream_t)stream;
  hipError_t e;
  if (splits > 1) {
    if (part == nullptr || part_elems < splits * m * n[0]) {
      set_last_error("%s: workspace needs %lld fp32 elements (given %lld)", what,
                     (long long)(splits * m * n[0]), (long long)part_elems);
      return MI_ERR_INVALID;
    }
    const int64_t nk = k / mid_bk(kg);
    a.part = part;
    // in stages of the kernel that runs (half as deep above three row blocks)
    a.split_stages = (int32_t)((nk + splits - 1) / splits) * (mb > 3 ? 2 : 1);
    a.part_vec = (uintptr_t)part % 16 == 0 && n[0] % 4 == 0 ? 1 : 0;
    e = mid_dtypes<kMidPartial>(a, kg, mb, splits, dtype, sdtype, st);
    if (e == hipSuccess) {
      GemmArgs g;
      gemm_setup(what, x, w[0], scales[0], y[0], m, n[0], k, x_sm, w_sn[0], s_sn[0], y_sm[0], g);
      g.part = part;
      g.part_vec = a.part_vec;
      g.res = res;
      g.res_sm = res_sm;
      launch_reduce(g, (int32_t)splits, dtype, sdtype, st);
      e = hipGetLastError();
    }
  } else {
    e = epilogue == 2 ? mid_dtypes<kMidSwiglu>(a, kg, mb, 1, dtype, sdtype, st)
                      : mid_dtypes<kMidStore>(a, kg, mb, 1, dtype, sdtype, st);
  }
  if (e != hipSuccess) {
    set_last_error("%s: launch failed: %s", what, hipGetErrorString(e));
    return (int32_t)e;
  }
  return MI_OK;
}
