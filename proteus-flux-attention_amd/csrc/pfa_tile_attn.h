// Packed attention on tiles: implicit causal and additively masked branches,
// 16 query rows per wave on the matrix cores.
//
// The rows of one head that lie together in the packed order share every key,
// so a workgroup takes 16 * RG consecutive packed rows and streams the keys
// 0..kmax of their head once, in tiles of TK keys through a two-stage LDS
// ring.  Each wave computes S^T = K Q^T and O^T += V^T P^T, so a lane owns
// one query row (lane mod 16) and, of every 16-key block, the keys
// 4 (lane/16) ..+3.  The row kernel (pfa_attn.hip) reads every key from cache
// again for each row and multiplies on the vector unit.  At 16 heads x 4,096
// tokens x 64 dims, half the rows active, f16 causal: 815 -> 81 us (213
// TFLOP/s; bound by the softmax's vector work, three P.V products beside it).
// 16 heads x 1,500 tokens, f32 masked: 377 -> 98 us (47 TFLOP/s of the 154
// that a large f32 product reaches; 188 blocks of rows do not fill the chip).
//
// Scores, softmax and sums are f32, and P keeps all 24 bits of its f32 value:
//   f32  : v_mfma_f32_16x16x4_f32 (four fma in turn) for both products, in
//     short sums (products_f32).
//   16-bit inputs: QK^T products are exact in f32; P is split into three parts
//     of the input type (split_p), three products per tile.
//   int8 : values are exact in bf16 (converted on the way into LDS), P as for
//     bf16; the per-head scales ride on the score scale and the output.
// Two things are below the row kernel: f16 inputs hold P to 2^-39 absolutely
// where it is under 2^-16 (an f16 result, whose last bit is 2^-24 at least, has
// room for what that leaves out only with values over 2^14), and with 16-bit and
// int8 inputs a P under 2^-126 counts as zero.  Distance from the 64-bit result over lengths of 16 to 400
// (24 draws each), of the row kernel's: f32 0.85-0.99, int8 0.57-0.76; with P
// in two 16-bit parts and longer sums int8 was at 1.4-1.6 and f32 at 1.1-1.4,
// for 4-19% less time.
//
// KS = 4/RG key splits: with few rows the four waves of a workgroup share
// fewer row groups and take every KS-th tile each; their partial states meet
// in LDS at the end.
//
// A row whose result is not finite is recomputed by the row loop
// (attend_row): the tiles multiply zero probabilities with keys past the row's
// own, and 0 * inf must not reach it.
#pragma once

#include "pfa_attn.h"

namespace pfa {
namespace tile {

typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2_t __attribute__((ext_vector_type(2)));

template <int IDT, int D, int KS>
struct Cfg {
  static constexpr bool kF32 = IDT == PFA_F32;
  static constexpr int RG = 4 / KS;            // 16-row groups per workgroup
  static constexpr int NH = D > 64 ? 2 : 1;    // 64-dim halves of a 16-bit tile row
  // keys per tile: two stages of KS K and V tiles within 64 KB
  static constexpr int kFit = kF32 ? 4096 / (KS * D) : 128 / (KS * NH);
  static constexpr int TK = kFit > 64 ? 64 : kFit;
  static constexpr int NKB = TK / 16;
  static constexpr int NDC = D > 32 ? D / 32 : 1;  // 32-dim score products (16-bit)
  static constexpr int NDB = D / 16;               // 16-dim output blocks
  static constexpr int kHalfBytes = kF32 ? TK * D * 4 : TK * 128 * NH;  // K (or V) of one tile
  static constexpr int kTileBytes = 2 * kHalfBytes;
  static constexpr int kStageBytes = KS * kTileBytes;
  static constexpr int kWaves = (IDT == PFA_F16 || IDT == PFA_BF16) && D <= 64 && KS == 1 ? 4 : 2;
  static_assert(NKB >= 1 && (kF32 || NKB >= 2), "tile too small");
};

// Kernel modes: implicit causal, or a mask of f32 or of 16-bit entries.
enum TileMode { kTileCausal = 0, kTileMask32 = 1, kTileMask16 = 2 };

// f32 tile rows of D/4 16-byte chunks: chunk c of row r sits at slot
// c ^ f32_swz(r), so that the sixteen rows of a K fragment read and the
// sixteen chunks of a V fragment read fall in different bank groups.
template <int D>
__device__ __forceinline__ int f32_swz(int r) {
  if constexpr (D >= 64) return r & 15;
  else if constexpr (D == 32) return (r >> 1) & 7;
  else return (r >> 2) & 3;
}

// f16 products for f16 inputs, bf16 products for bf16 and int8 (whose values
// are exact in bf16).
template <int IDT>
__device__ __forceinline__ f32x4_t mfma16(bf16x8_t a, bf16x8_t b, f32x4_t c) {
  if constexpr (IDT != PFA_F16) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
  } else {
    f16x8_t x, y;
    __builtin_memcpy(&x, &a, 16);
    __builtin_memcpy(&y, &b, 16);
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(x, y, c, 0, 0, 0);
  }
}

// P (8 values) as kParts parts of the product type, each cut off from what
// the parts before it leave: all 24 bits of P.  bf16 parts carry 8 bits each
// at any size; f16 parts 11, of kPScale P (and the row sum with it), so that P
// has its 24 bits down to 2^-16 and 2^-39 absolutely below.  The scale is
// multiplied on: in the exponent it would cost the exponent's own last bits.
constexpr int kParts = 3;
template <int IDT>
constexpr float kPScale = IDT == PFA_F16 ? 32768.f : 1.f;
template <int IDT>
__device__ __forceinline__ void split_p(const float (&p)[8], bf16x8_t (&part)[kParts]) {
  float r[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) r[i] = p[i];
#pragma unroll
  for (int n = 0; n < kParts; ++n) {
    if constexpr (IDT == PFA_F16) {
      f16x2_t h[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const auto w = __builtin_amdgcn_cvt_pkrtz(r[2 * i], r[2 * i + 1]);
        __builtin_memcpy(&h[i], &w, 4);
        r[2 * i] -= (float)h[i][0];
        r[2 * i + 1] -= (float)h[i][1];
      }
      __builtin_memcpy(&part[n], h, 16);
    } else {
      uint32_t h[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const uint32_t a = __float_as_uint(r[2 * i]), b = __float_as_uint(r[2 * i + 1]);
        h[i] = __builtin_amdgcn_perm(b, a, 0x07060302u);  // their upper halves
        r[2 * i] -= __uint_as_float(a & 0xffff0000u);
        r[2 * i + 1] -= __uint_as_float(b & 0xffff0000u);
      }
      __builtin_memcpy(&part[n], h, 16);
    }
  }
}

// 2^x of a probability or a factor of one.  f32 results keep the row kernel's
// denormals.
template <int IDT>
__device__ __forceinline__ float exp2_p(float x) {
  if constexpr (IDT == PFA_F32) return exp2f(x);
  else return __builtin_amdgcn_exp2f(x);
}

// Whether a score is scaled in the step that takes it off its maximum.  The
// maximum is a rounded product and the score then is not: at large scores it
// can come out above it, P above 1, where f16 parts end (at 2^17 of 2^15 P).
template <int IDT>
constexpr bool kFused = IDT != PFA_F16;

// int8 values as bf16
__device__ __forceinline__ bf16x8_t i8_bf16(uint32_t x, uint32_t y) {
  const uint32_t w[2] = {x, y};
  uint32_t o[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t v = w[i >> 1] >> (16 * (i & 1));
    o[i] = __builtin_amdgcn_perm(__float_as_uint((float)(int8_t)(v >> 8)), __float_as_uint((float)(int8_t)v), 0x07060302u);
  }
  bf16x8_t b;
  __builtin_memcpy(&b, o, 16);
  return b;
}

template <bool FIRST, typename V>
__device__ __forceinline__ V& pick(V& a, V& b) {
  if constexpr (FIRST) return a;
  else return b;
}

// A result from its sum: divided where it may be stored as f32, by the
// reciprocal where 16 bits of it are.
template <int IDT>
__device__ __forceinline__ float normalise(float x, float l, float inv, float vs) {
  if constexpr (IDT == PFA_F32) return x / l;
  else if constexpr (IDT == PFA_I8) return x / l * vs;
  else return x * inv;
}

// The query of a row, negated.
template <bool F32, int NX, int NF>
__device__ __forceinline__ void negate_q(f32x4_t (&qx)[NX], bf16x8_t (&qf)[NF]) {
  if constexpr (F32) {
#pragma unroll
    for (int j = 0; j < NX; ++j) qx[j] = -qx[j];
  } else {
#pragma unroll
    for (int dc = 0; dc < NF; ++dc) {
      uint32_t w[4];
      __builtin_memcpy(w, &qf[dc], 16);
#pragma unroll
      for (int i = 0; i < 4; ++i) w[i] ^= 0x80008000u;
      __builtin_memcpy(&qf[dc], w, 16);
    }
  }
}

// Sum of N (a power of two) values in a tree.
template <int N, typename V>
__device__ __forceinline__ V tree_sum(V (&x)[N]) {
#pragma unroll
  for (int w = 1; w < N; w *= 2)
#pragma unroll
    for (int i = 0; i + w < N; i += 2 * w) x[i] = x[i] + x[i + w];
  return x[0];
}

// The f32 product over 4 N k-steps of four terms, a(n) b(n): sums of eight
// terms, then a tree, so that no sum is longer than the row kernel's lanes
// keep it.  (Sums of sixteen leave results of 32-dim heads 9% further from the
// 64-bit ones than the row kernel's, and take 3% less time.)
template <int N, typename A, typename B>
__device__ __forceinline__ f32x4_t products_f32(A a, B b) {
  f32x4_t part[2 * N];
#pragma unroll
  for (int n = 0; n < 2 * N; ++n) {
    part[n] = __builtin_amdgcn_mfma_f32_16x16x4f32(a(2 * n), b(2 * n), f32x4_t{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    part[n] = __builtin_amdgcn_mfma_f32_16x16x4f32(a(2 * n + 1), b(2 * n + 1), part[n], 0, 0, 0);
  }
  return tree_sum(part);
}

// Store n consecutive output values (aligned to n elements).
template <int N>
__device__ __forceinline__ void store_n(void* row, int odt, int d, const float* v) {
  if (odt == PFA_F32) {
    __builtin_memcpy(__builtin_assume_aligned((float*)row + d, 4 * N), v, 4 * N);
  } else {
    uint16_t w[N];
#pragma unroll
    for (int i = 0; i < N; ++i) w[i] = odt == PFA_BF16 ? f32_to_bf16(v[i]) : f32_to_f16(v[i]);
    __builtin_memcpy(__builtin_assume_aligned((uint16_t*)row + d, 2 * N), w, 2 * N);
  }
}

template <int IDT, int D, int KS, int MODE>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(MODE == kTileCausal ? Cfg<IDT, D, KS>::kWaves : 2, 8)))
tile_attn_kernel(AttnArgs a, int odt) {
  using C = Cfg<IDT, D, KS>;
  using IT = typename Elem<IDT>::T;
  constexpr bool MASKED = MODE != kTileCausal;
  constexpr int RG = C::RG, TK = C::TK, NKB = C::NKB, NDB = C::NDB, NH = C::NH;
  constexpr int kRows = 16 * RG;
  __shared__ __align__(16) uint8_t ring[2 * C::kStageBytes];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r16 = lane & 15, g = lane >> 4;
  const int rg = wid % RG, ks = wid / RG;
  // Each XCD walks one contiguous slice of the packed rows; every second run
  // of 32 workgroups (one per CU of the XCD) goes backwards.
  const int64_t per = gridDim.x / 8;
  int64_t j = blockIdx.x / 8;
  if ((j >> 5) & 1) {
    const int64_t b0 = j & ~(int64_t)31, e0 = min<int64_t>(b0 + 32, per);
    j = b0 + (e0 - 1 - j);
  }
  const int64_t lb = (blockIdx.x % 8) * per + (per - 1 - j);
  const int64_t r0 = lb * kRows;
  const int64_t nrow = attn_rows(a);
  if (r0 >= nrow) return;

  // lane l (< kRows) of every wave holds row l's token and head
  int t_l = -1, h_l = -1;
  if (lane < kRows && r0 + lane < nrow) {
    t_l = a.token_idx[r0 + lane];
    h_l = t_l >= 0 ? a.row_head[r0 + lane] : -1;
  }
  const uint32_t ring_lds = __builtin_amdgcn_readfirstlane(lds_addr(ring));
  SwzLane L;
  if constexpr (!C::kF32) L.init();
  // every K/V byte offset of a head fits in 32 bits
  const bool off32 = a.k.s_t > 0 && a.v.s_t > 0 && (a.T + 1) * max(a.k.s_t, a.v.s_t) * (int64_t)sizeof(IT) < (1ll << 32);

  for (int s0 = 0; s0 < kRows;) {
    const int hp = __builtin_amdgcn_readlane(h_l, s0);
    const uint64_t other = __ballot(lane > s0 && (h_l != hp || lane >= kRows));
    const int s1 = other ? __builtin_ctzll(other) : kRows;
    if (hp < 0) {
      s0 = s1;
      continue;
    }
    const int bh = a.head_map ? a.head_map[hp] : hp;
    const int64_t bb = bh / a.H, hh = bh % a.H;
    const int qs = 16 * rg + r16;  // this lane's row of the workgroup
    const int tq = __shfl(t_l, qs, 64);
    const bool qv = qs >= s0 && qs < s1;
    // token range of the segment and of this wave's rows in it
    int smax = (lane >= s0 && lane < s1) ? t_l : -1;
    int wmax = qv ? tq : -1, wmin = qv ? tq : INT32_MAX;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) smax = max(smax, __shfl_xor(smax, o, 64));
#pragma unroll
    for (int o = 1; o < 16; o <<= 1) {
      wmax = max(wmax, __shfl_xor(wmax, o, 64));
      wmin = min(wmin, __shfl_xor(wmin, o, 64));
    }
    // the last key, of those there are: below 0 no key at all (no score, NaN
    // rows, as in the row kernel), and the loads stay at key 0
    const int kmax = min(__builtin_amdgcn_readfirstlane(MASKED ? a.head_max[hp] : smax), (int)a.T - 1);
    const int kload = max(kmax, 0);
    wmax = __builtin_amdgcn_readfirstlane(wmax);
    wmin = __builtin_amdgcn_readfirstlane(wmin);
    const int nstep = kmax / (TK * KS) + 1;

    const IT* kb = (const IT*)a.k.ptr + bb * a.k.s_b + hh * a.k.s_h;
    const IT* vb = (const IT*)a.v.ptr + bb * a.v.s_b + hh * a.v.s_h;
    const IT* qp = (const IT*)a.q.ptr + bb * a.q.s_b + hh * a.q.s_h + (int64_t)(qv ? tq : 0) * a.q.s_t;

    // ---- tiles into LDS: step st brings the tiles st*KS .. st*KS+KS-1 ----
    // f32 and 16-bit tiles go by LDS DMA (1 KB per wave and transfer); int8
    // tiles through registers, converted to bf16 on the way.
    // Thread tid moves the 16-byte slots tid + 256 j of each K or V tile; the
    // rows of j > 0 lie a multiple of 16 further (8 for f32 rows of 128), so
    // the chunk that belongs in the slot is the same for every j (but for the
    // swizzle's bit 3).
    constexpr int CPR = C::kF32 ? D / 4 : 8;                // chunks per row (of one half)
    constexpr int kRowStep = 256 / CPR;                     // rows between j and j + 1
    constexpr int kJ = C::kHalfBytes / 4096;                // slots per thread
    static_assert(C::kHalfBytes % 4096 == 0 && kRowStep % 8 == 0, "slot layout");
    constexpr int kFlip = kRowStep % 16 ? 32 : 0;           // elements of the swizzle's bit 3
    const int row0 = tid / CPR;
    const int elem0 = C::kF32 ? 4 * ((tid % CPR) ^ f32_swz<D>(row0))
                              : 8 * (((tid & 7) ^ tile_swz(row0)) & (D >= 64 ? 7 : D / 8 - 1));
    auto request = [&](int st) {
      const uint32_t stage = ring_lds + (uint32_t)(st & 1) * C::kStageBytes + 1024u * (uint32_t)wid;
#pragma unroll
      for (int sub = 0; sub < KS; ++sub)
#pragma unroll
        for (int j = 0; j < kJ; ++j) {
          // 16-bit tiles of D = 128: the second 64-dim half after the first
          const int row = row0 + kRowStep * j % TK, elem = (elem0 ^ (kFlip * (j & 1))) + 64 * (kRowStep * j / TK);
          const int key = min((st * KS + sub) * TK + row, kload);
          const uint32_t dst = stage + sub * C::kTileBytes + 4096 * j;
          if (off32) {
            lds_dma16_s(kb, ((uint32_t)key * (uint32_t)a.k.s_t + elem) * (uint32_t)sizeof(IT), dst);
            lds_dma16_s(vb, ((uint32_t)key * (uint32_t)a.v.s_t + elem) * (uint32_t)sizeof(IT), dst + C::kHalfBytes);
          } else {
            lds_dma16(kb + (int64_t)key * a.k.s_t + elem, dst);
            lds_dma16(vb + (int64_t)key * a.v.s_t + elem, dst + C::kHalfBytes);
          }
        }
    };
    constexpr int CW = D >= 32 ? D / 8 : 4;                 // 8-value chunks staged per int8 row
    constexpr int kReg = IDT == PFA_I8 ? 2 * KS * TK * CW / 256 : 1;  // chunks per thread and step
    uint2 regs[kReg];
    auto fetch8 = [&](int st) {
#pragma unroll
      for (int j = 0; j < kReg; ++j) {
        const int n = tid + 256 * j;
        const int c = n % CW, row = (n / CW) % TK, sub = (n / (CW * TK)) % KS;
        const int key = min((st * KS + sub) * TK + row, kload);
        const int e = 8 * (c & (D / 8 - 1));
        const IT* src = n / (CW * TK * KS) ? vb + (int64_t)key * a.v.s_t + e : kb + (int64_t)key * a.k.s_t + e;
        regs[j] = *reinterpret_cast<const uint2*>(src);
      }
    };
    auto stash8 = [&](int st) {
      uint8_t* stage = ring + (st & 1) * C::kStageBytes;
#pragma unroll
      for (int j = 0; j < kReg; ++j) {
        const int n = tid + 256 * j;
        const int c = n % CW, row = (n / CW) % TK, sub = (n / (CW * TK)) % KS;
        const int isv = n / (CW * TK * KS);
        const bf16x8_t h = i8_bf16(regs[j].x, regs[j].y);
        uint8_t* dst = stage + sub * C::kTileBytes + isv * C::kHalfBytes + (c >> 3) * TK * 128 + row * 128 +
                       16 * ((c & 7) ^ tile_swz(row));
        __builtin_memcpy(__builtin_assume_aligned(dst, 16), &h, 16);
      }
    };
    if constexpr (IDT == PFA_I8) fetch8(0);
    else request(0);

    // ---- this lane's query row ----
    // 16-bit: the chunks 4dc + g (8 dims each); f32: the chunks 4j + g (4 dims)
    bf16x8_t qf[C::NDC];
    f32x4_t qx[D / 16];
    if constexpr (C::kF32) {
#pragma unroll
      for (int j = 0; j < D / 16; ++j) qx[j] = *reinterpret_cast<const f32x4_t*>(qp + 16 * j + 4 * g);
#pragma unroll
      for (int j = 0; j < D / 16; ++j) asm volatile("" : "+v"(qx[j]));  // settled before the tile loop
    } else {
#pragma unroll
      for (int dc = 0; dc < C::NDC; ++dc) {
        qf[dc] = bf16x8_t{};
        if (D >= 32 || g < 2) {
          if constexpr (IDT == PFA_I8) {
            const uint2 w = *reinterpret_cast<const uint2*>(qp + 32 * dc + 8 * g);
            qf[dc] = i8_bf16(w.x, w.y);
          } else {
            qf[dc] = *reinterpret_cast<const bf16x8_t*>(qp + 32 * dc + 8 * g);
          }
        }
        asm volatile("" : "+v"(qf[dc]));
      }
    }
    float sl2 = a.scale * kLog2e;
    if constexpr (IDT == PFA_I8) sl2 *= a.q_scale[bh] * a.k_scale[bh];
    if (sl2 < 0.f) {
      // the maximum may be taken over unscaled scores (kFused): negate q
      // instead
      sl2 = -sl2;
      negate_q<C::kF32>(qx, qf);
    }

    float m = -INFINITY, l = 0.f;
    f32x4_t acc[NDB];
#pragma unroll
    for (int db = 0; db < NDB; ++db) acc[db] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    const int64_t mrow = MASKED ? (int64_t)(qv ? tq : 0) * a.T : 0;
    // mask entries of the next tile, loaded a step ahead (a load waited for
    // inside the step would wait for the step's tile transfers too)
    // (at most the row's last four entries, so that the loads take no branch)
    constexpr int MW = MODE == kTileMask32 ? 4 : 2;  // words of four entries
    uint32_t mk[MASKED ? NKB : 1][MW];
    auto fetch_mask = [&](int st) {
      const int kt = (st * KS + ks) * TK + 4 * g;
#pragma unroll
      for (int b = 0; b < NKB; ++b)
        __builtin_memcpy(mk[b], (const uint8_t*)a.mask + (mrow + min(kt + 16 * b, (int)a.T - 4)) * MW, 4 * MW);
    };
    if constexpr (MASKED) fetch_mask(0);

    if constexpr (IDT == PFA_I8) stash8(0);
    for (int st = 0; st < nstep; ++st) {
      dma_wait_barrier<0>();
      const int k0 = (st * KS + ks) * TK;
      float mc[MASKED ? NKB : 1][4];
      if constexpr (MASKED) {
#pragma unroll
        for (int b = 0; b < NKB; ++b)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            if constexpr (MODE == kTileMask32) {
              mc[b][i] = __uint_as_float(mk[b][i]);
            } else {
              const uint16_t h = (uint16_t)(mk[b][i >> 1] >> (16 * (i & 1)));
              mc[b][i] = a.mask_dtype == PFA_BF16 ? bf16_to_f32(h) : f16_to_f32(h);
            }
          }
        if (k0 + TK > (int)a.T) {  // the row's end: entries loaded before their place move down
#pragma unroll
          for (int b = 0; b < NKB; ++b) {
            const int past = k0 + 16 * b + 4 * g - ((int)a.T - 4);
#pragma unroll
            for (int sft = 0; sft < 3; ++sft)
              if (past > sft) {
                mc[b][0] = mc[b][1];
                mc[b][1] = mc[b][2];
                mc[b][2] = mc[b][3];
              }
          }
        }
        if (st + 1 < nstep) fetch_mask(st + 1);
      }
      if (st + 1 < nstep) {
        if constexpr (IDT == PFA_I8) fetch8(st + 1);
        else request(st + 1);
      }
      // causal: a tile past all of this wave's rows has nothing for it
      if (wmax >= 0 && k0 <= (MASKED ? kmax : wmax)) {
        const uint8_t* tb = ring + (st & 1) * C::kStageBytes + ks * C::kTileBytes;
        f32x4_t c[NKB];
        if constexpr (C::kF32) {
          const float* kt = (const float*)tb;
#pragma unroll
          for (int b = 0; b < NKB; ++b) {
            const int row = 16 * b + r16;
            f32x4_t ka[D / 16];
#pragma unroll
            for (int j = 0; j < D / 16; ++j)
              ka[j] = *reinterpret_cast<const f32x4_t*>(kt + row * D + 4 * ((4 * j + g) ^ f32_swz<D>(row)));
            c[b] = products_f32<D / 16>([&](int n) { return ka[n >> 2][n & 3]; }, [&](int n) { return qx[n >> 2][n & 3]; });
          }
        } else {
          const uint16_t* kt = (const uint16_t*)tb;
          bf16x8_t ka[C::NDC][NKB];
#pragma unroll
          for (int dc = 0; dc < C::NDC; ++dc)
#pragma unroll
            for (int b = 0; b < NKB; ++b)
              ka[dc][b] = *reinterpret_cast<const bf16x8_t*>(kt + (dc >> 1) * TK * 64 + 1024 * b + L.ko[dc & 1]);
#pragma unroll
          for (int b = 0; b < NKB; ++b) c[b] = mfma16<IDT>(ka[0][b], qf[0], f32x4_t{0.f, 0.f, 0.f, 0.f});
#pragma unroll
          for (int dc = 1; dc < C::NDC; ++dc)
#pragma unroll
            for (int b = 0; b < NKB; ++b) c[b] = mfma16<IDT>(ka[dc][b], qf[dc], c[b]);
        }
        // scores in log2 units: s * scale (+ mask); -inf for keys past the row
        float s[NKB][4], tmax = -INFINITY;
        const bool cut = k0 + TK - 1 > (MASKED ? kmax : wmin);
        const int last = (MASKED ? kmax : tq) - k0 - 4 * g;
#pragma unroll
        for (int b = 0; b < NKB; ++b) {
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            float x = c[b][i];
            if constexpr (MASKED) x = __builtin_fmaf(x, sl2, kLog2e * mc[b][i]);
            else if constexpr (!kFused<IDT>) x *= sl2;
            if (cut && 16 * b + i > last) x = -INFINITY;
            s[b][i] = x;
            tmax = fmaxf(tmax, x);
          }
        }
        tmax = max_over_rows4(tmax);
        if constexpr (!MASKED && kFused<IDT>) tmax *= sl2;  // sl2 > 0, -inf stays
        if (__ballot(tmax > m) != 0) {  // some row's maximum rises
          const float mn = fmaxf(m, tmax);
          const float alpha = mn == -INFINITY ? 1.f : exp2_p<IDT>(m - mn);
          l *= alpha;
#pragma unroll
          for (int db = 0; db < NDB; ++db)
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[db][i] *= alpha;
          m = mn;
        }
        const float moff = m == -INFINITY ? 0.f : m;  // m = -inf: only -inf scores so far
        float ps[NKB];
#pragma unroll
        for (int b = 0; b < NKB; ++b) {
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const float x = MASKED || !kFused<IDT> ? s[b][i] - moff : __builtin_fmaf(s[b][i], sl2, -moff);
            s[b][i] = exp2_p<IDT>(x) * kPScale<IDT>;
          }
          ps[b] = (s[b][0] + s[b][1]) + (s[b][2] + s[b][3]);
        }
        l += tree_sum(ps);
        if constexpr (C::kF32) {
          // V^T rows are the dims NDB * m + db (db < 4; the second 64 dims
          // for db >= 4): one read per key serves every db.  A tile's products
          // are summed by themselves and then added, so that the sums stay
          // short
          const float* vt = (const float*)(tb + C::kHalfBytes);
          float va[4 * NKB][NDB];
#pragma unroll
          for (int n = 0; n < 4 * NKB; ++n) {
            const int row = 16 * (n >> 2) + 4 * g + (n & 3);
            const float* vr = vt + row * D;
            if constexpr (NDB >= 4) {
#pragma unroll
              for (int h = 0; h < NDB / 4; ++h)
                __builtin_memcpy(va[n] + 4 * h, __builtin_assume_aligned(vr + 4 * ((16 * h + r16) ^ f32_swz<D>(row)), 16),
                                 16);
            } else {
              const int d0 = NDB * r16;
              __builtin_memcpy(va[n], __builtin_assume_aligned(vr + 4 * ((d0 >> 2) ^ f32_swz<D>(row)) + (d0 & 3), 4 * NDB),
                               4 * NDB);
            }
          }
#pragma unroll
          for (int db = 0; db < NDB; ++db)
            acc[db] += products_f32<NKB>([&](int n) { return va[n][db]; }, [&](int n) { return s[n >> 2][n & 3]; });
        } else {
          const uint16_t* vt = (const uint16_t*)(tb + C::kHalfBytes);
          // (int8 results are f32: the tile by itself, as above)
          f32x4_t ta[NDB];
          auto& to = pick<IDT == PFA_I8>(ta, acc);
          if constexpr (IDT == PFA_I8) {
#pragma unroll
            for (int db = 0; db < NDB; ++db) ta[db] = f32x4_t{0.f, 0.f, 0.f, 0.f};
          }
#pragma unroll
          for (int kc = 0; kc < NKB / 2; ++kc) {
            float p[8];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              p[i] = s[2 * kc][i];
              p[4 + i] = s[2 * kc + 1][i];
            }
            bf16x8_t part[kParts];
            split_p<IDT>(p, part);
#pragma unroll
            for (int db = 0; db < NDB; ++db) {
              const uint16_t* vr = vt + (db >> 2) * TK * 64 + 64 * 32 * kc + L.vo[db & 3];
              const i16x4_t v0 = ds_tr4(vr), v1 = ds_tr4(vr + 64 * 16);
              bf16x8_t va;
              __builtin_memcpy(&va, &v0, 8);
              __builtin_memcpy(reinterpret_cast<char*>(&va) + 8, &v1, 8);
#pragma unroll
              for (int n = kParts - 1; n >= 0; --n) to[db] = mfma16<IDT>(va, part[n], to[db]);
            }
          }
          if constexpr (IDT == PFA_I8) {
#pragma unroll
            for (int db = 0; db < NDB; ++db) acc[db] += ta[db];
          }
        }
      }
      if constexpr (IDT == PFA_I8) {
        if (st + 1 < nstep) stash8(st + 1);
      }
    }
    l += __shfl_xor(l, 16, 64);
    l += __shfl_xor(l, 32, 64);

    if constexpr (KS > 1) {
      // the splits' states meet in LDS: wave (rg, 0) merges its row group
      constexpr int W = 4 * NDB + 2;
      static_assert(4 * W * 64 * 4 <= 2 * C::kStageBytes, "merge area");
      __syncthreads();  // every wave is done with the tiles
      float* mine = (float*)ring + (int64_t)wid * W * 64 + lane;
      if (ks > 0) {
        mine[0] = m;
        mine[64] = l;
#pragma unroll
        for (int db = 0; db < NDB; ++db)
#pragma unroll
          for (int i = 0; i < 4; ++i) mine[64 * (2 + 4 * db + i)] = acc[db][i];
      }
      __syncthreads();
      if (ks == 0) {
        for (int k = 1; k < KS; ++k) {
          const float* o = (const float*)ring + (int64_t)(rg + RG * k) * W * 64 + lane;
          const float mo = o[0], mn = fmaxf(m, mo);
          const float fa = m == -INFINITY ? 0.f : exp2_p<IDT>(m - mn);
          const float fb = mo == -INFINITY ? 0.f : exp2_p<IDT>(mo - mn);
          l = l * fa + o[64] * fb;
#pragma unroll
          for (int db = 0; db < NDB; ++db)
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[db][i] = acc[db][i] * fa + o[64 * (2 + 4 * db + i)] * fb;
          m = mn;
        }
      }
    }

    if (ks == 0 && wmax >= 0) {
      bool bad = false;
      const float inv = 1.f / l;
      const float vs = IDT == PFA_I8 ? a.v_scale[bh] : 1.f;
#pragma unroll
      for (int db = 0; db < NDB; ++db)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          acc[db][i] = normalise<IDT>(acc[db][i], l, inv, vs);
          bad |= !(fabsf(acc[db][i]) <= 3.402823466e38f);
          if (l == 0.f) acc[db][i] = __builtin_nanf("");  // every score -inf
        }
      bad = bad && qv && l != 0.f;
      uint64_t redo = __ballot(bad);
      redo = (redo | (redo >> 16) | (redo >> 32) | (redo >> 48)) & 0xffffull;
      const int osz = odt == PFA_F32 ? 4 : 2;
      uint8_t* ob = (uint8_t*)a.out.ptr + (bb * a.out.s_b + hh * a.out.s_h) * osz;
      if (qv && !((redo >> r16) & 1)) {
        void* orow = ob + (int64_t)tq * a.out.s_t * osz;
        if constexpr (C::kF32) {
          // lane's dims NDB * (4g + i) + db (db < 4)
          constexpr int Q = NDB < 4 ? NDB : 4;
#pragma unroll
          for (int h = 0; h < (NDB + 3) / 4; ++h)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              float o[Q];
#pragma unroll
              for (int db = 0; db < Q; ++db) o[db] = acc[4 * h + db][i];
              store_n<Q>(orow, odt, 64 * h + Q * (4 * g + i), o);
            }
        } else {
#pragma unroll
          for (int db = 0; db < NDB; ++db) {
            const float o[4] = {acc[db][0], acc[db][1], acc[db][2], acc[db][3]};
            store_n<4>(orow, odt, 16 * db + 4 * g, o);
          }
        }
      }
      while (redo) {
        const int i = __builtin_ctzll(redo);
        redo &= redo - 1;
        const int t = __shfl(tq, i, 64);
        float ra[8], rl;
        attend_row<IDT, D>(a, r0 + 16 * rg + i, t, bh, MASKED ? (int64_t)kmax + 1 : (int64_t)t + 1, nullptr, ra, rl);
        if (lane < D / 8) {
          const float rinv = 1.f / rl;
#pragma unroll
          for (int e = 0; e < 8; ++e) ra[e] = rl == 0.f ? __builtin_nanf("") : ra[e] * rinv;
          store_n<8>(ob + (int64_t)t * a.out.s_t * osz, odt, 8 * lane, ra);
        }
      }
    }
    __syncthreads();  // the ring is free for the next segment
    s0 = s1;
  }
}

template <int IDT, int D, int KS>
static int launch_ks(const AttnArgs& a, int odt, hipStream_t s) {
  constexpr int kRows = 16 * Cfg<IDT, D, KS>::RG;
  int64_t blocks = (a.N + kRows - 1) / kRows;
  blocks = (blocks + 7) / 8 * 8;
  PFA_CHECK_ARG(blocks < INT32_MAX, "pfa_sparse_attn_fwd: too many rows");
  if (a.mode == kModeCausal) tile_attn_kernel<IDT, D, KS, kTileCausal><<<(unsigned)blocks, 256, 0, s>>>(a, odt);
  else if (a.mask_dtype == PFA_F32) tile_attn_kernel<IDT, D, KS, kTileMask32><<<(unsigned)blocks, 256, 0, s>>>(a, odt);
  else tile_attn_kernel<IDT, D, KS, kTileMask16><<<(unsigned)blocks, 256, 0, s>>>(a, odt);
  PFA_CHECK_LAUNCH("pfa_sparse_attn_fwd");
  return PFA_OK;
}

// Key splits by the number of 64-row blocks, against the chip's 256 CUs.
// Measured on one box (us; key splits 1 / 2 / 4, D = 64 unless named):
//   125 blocks, int8 causal, D = 32, T 1,000:   21.8 /  17.1 /  14.6
//   188 blocks, f32 masked, T 1,500:           187.3 / 123.2 /  93.5
//   188 blocks, bf16 masked, T 1,500:           68.0 /  47.4 /  41.1
//   512 blocks, f16 causal, T 4,096:            82.2 /  73.5 /  85.1
//   512 blocks, f32 causal, T 4,096:           230.6 / 239.3 / 248.7
//   768 blocks, f16 causal, T 4,096:            99.2 /  98.4 / 122.6
//   2,048 blocks, f16 causal, T 8,192:         368   / 428   / 553
// Below one block per CU the splits fill the chip; up to three, two splits
// even out the causal lengths of 16-bit rows (f32 rows are bound by the
// matrix unit already); above, the whole blocks read each tile least often.
template <int IDT, int D>
static int launch_d(const AttnArgs& a, int odt, hipStream_t s) {
  const int64_t blocks = (a.N + 63) / 64;
  if (blocks <= 256) return launch_ks<IDT, D, D <= 64 ? 4 : 2>(a, odt, s);
  if constexpr (IDT != PFA_F32 && D <= 64) {
    if (blocks <= 768) return launch_ks<IDT, D, 2>(a, odt, s);
  }
  return launch_ks<IDT, D, 1>(a, odt, s);
}

template <int IDT>
static int launch(const AttnArgs& a, int odt, int D, hipStream_t s) {
  switch (D) {
    case 16: return launch_d<IDT, 16>(a, odt, s);
    case 32: return launch_d<IDT, 32>(a, odt, s);
    case 64: return launch_d<IDT, 64>(a, odt, s);
    default: return launch_d<IDT, 128>(a, odt, s);
  }
}

}  // namespace tile
}  // namespace pfa
