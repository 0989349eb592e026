// Arguments and the one-row gather loop of the packed sparse attention
// kernels: the row kernel (one wave per row) and the tile kernel, which
// recomputes a row that came out non-finite.
#pragma once

#include "pfa_common.h"

namespace pfa {

constexpr int kAttnWaves = 4;
constexpr float kLog2e = 1.4426950408889634f;

enum AttnMode { kModeCand = 0, kModeCausal = 1, kModeMasked = 2 };

template <int DT>
__device__ __forceinline__ float load_mask(const void* m, int64_t off, int mdt) {
  if (mdt == PFA_F32) return ((const float*)m)[off];
  if (mdt == PFA_BF16) return bf16_to_f32(((const uint16_t*)m)[off]);
  return f16_to_f32(((const uint16_t*)m)[off]);
}

struct AttnArgs {
  pfa_tensor4 q, k, v, out;
  int H;
  int64_t T;
  const int32_t* token_idx;
  const int32_t* row_head;
  const int32_t* head_map;
  int64_t N;                // rows launched
  const int32_t* n_rows;    // device row count bounding N, or null
  const int32_t* cand;
  int64_t cand_stride;
  const int32_t* cand_len;
  const void* mask;
  int mask_dtype;
  const int32_t* head_max;
  float scale;
  const float* q_scale;
  const float* k_scale;
  const float* v_scale;
  int mode;
  // candidate rows: one byte per sixteen rows (the union kernel's verdict: 1
  // where the row kernel is to attend them), or null
  uint8_t* flags;
};

// Rows to process: the launch size, bounded by the device row count when one
// is given.
__device__ __forceinline__ int64_t attn_rows(const AttnArgs& a) {
  return a.n_rows ? min<int64_t>(a.N, (int64_t)a.n_rows[0]) : a.N;
}

// The grid is launched with a multiple of 8 workgroups, so this is a
// bijection on [0, gridDim.x).
__device__ __forceinline__ int64_t remap_block(int64_t P, int64_t nblk) {
  int64_t per = nblk / 8;
  return (P % 8) * per + P / 8;
}

// Attention of packed row r by one wave, unnormalised: the wave is split into
// 512/D key groups of D/8 lanes; every lane ends with its 8 dims (8 * (lane
// mod D/8) ..+7) of the accumulator and the row's probability sum l.
// n keys: crow[0..n) (candidates), or 0..n-1.
template <int IDT, int D>
__device__ __forceinline__ void attend_row(const AttnArgs& a, int64_t r, int64_t t, int bh, int64_t n,
                                           const int32_t* crow, float (&acc)[8], float& l) {
  using IT = typename Elem<IDT>::T;
  constexpr int LPK = D / 8;       // lanes per key
  constexpr int KPI = 64 / LPK;    // keys per iteration
  constexpr int U = (KPI >= 16) ? 2 : 4;  // iterations per softmax step
  const int lane = threadIdx.x & 63;
  const int grp = lane / LPK;
  const int e = lane % LPK;
  const int64_t bb = bh / a.H, hh = bh % a.H;
  const IT* qp = (const IT*)a.q.ptr + bb * a.q.s_b + hh * a.q.s_h + t * a.q.s_t + 8 * e;
  const IT* kb = (const IT*)a.k.ptr + bb * a.k.s_b + hh * a.k.s_h + 8 * e;
  const IT* vb = (const IT*)a.v.ptr + bb * a.v.s_b + hh * a.v.s_h + 8 * e;

  float qf[8];
  load8<IDT>(qp, qf);
  float qmul = a.scale * kLog2e;
  float kmul = 1.f, vmul = 1.f;
  if constexpr (IDT == PFA_I8) {
    qmul *= a.q_scale[bh];
    kmul = a.k_scale[bh];
    vmul = a.v_scale[bh];
  }
#pragma unroll
  for (int i = 0; i < 8; ++i) qf[i] *= qmul;

  const bool has_mask = a.mask != nullptr;

#pragma unroll
  for (int i = 0; i < 8; ++i) acc[i] = 0.f;
  float m = -INFINITY;
  l = 0.f;

  for (int64_t i0 = 0; i0 < n; i0 += (int64_t)KPI * U) {
    float kf[U][8], vf[U][8], s[U];
    int64_t key[U];
    bool ok[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      int64_t i = i0 + u * KPI + grp;
      ok[u] = i < n;
      int64_t kk = 0;
      if (ok[u]) kk = crow ? (int64_t)crow[i] : i;
      kk = kk < 0 ? 0 : (kk >= a.T ? a.T - 1 : kk);
      key[u] = kk;
      load8<IDT>(kb + kk * a.k.s_t, kf[u]);
      load8<IDT>(vb + kk * a.v.s_t, vf[u]);
    }
    float cmax = -INFINITY;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      float d = 0.f;
#pragma unroll
      for (int i = 0; i < 8; ++i) d = __builtin_fmaf(qf[i], kf[u][i], d);
#pragma unroll
      for (int off = 1; off < LPK; off <<= 1) d += __shfl_xor(d, off, 64);
      d *= kmul;
      if (has_mask) d += kLog2e * load_mask<IDT>(a.mask, t * a.T + key[u], a.mask_dtype);
      s[u] = ok[u] ? d : -INFINITY;
      cmax = fmaxf(cmax, s[u]);
    }
#pragma unroll
    for (int off = LPK; off < 64; off <<= 1) cmax = fmaxf(cmax, __shfl_xor(cmax, off, 64));
    float mn = fmaxf(m, cmax);
    if (mn == -INFINITY) continue;  // nothing finite yet
    float alpha = exp2f(m - mn);    // m == -inf -> 0
    l *= alpha;
#pragma unroll
    for (int i = 0; i < 8; ++i) acc[i] *= alpha;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      float p = exp2f(s[u] - mn);
      l += p;
      float pv = p * vmul;
#pragma unroll
      for (int i = 0; i < 8; ++i) acc[i] = __builtin_fmaf(pv, vf[u][i], acc[i]);
    }
    m = mn;
  }
  // combine key groups
#pragma unroll
  for (int off = LPK; off < 64; off <<= 1) {
    l += __shfl_xor(l, off, 64);
#pragma unroll
    for (int i = 0; i < 8; ++i) acc[i] += __shfl_xor(acc[i], off, 64);
  }
}

// Host side (pfa_tile_attn_<type>.hip): the tile kernel on rows that the
// dispatch of pfa_sparse_attn_fwd gives it.
int tile_attn_launch_f32(const AttnArgs& a, int out_dtype, int D, hipStream_t s);
int tile_attn_launch_f16(const AttnArgs& a, int out_dtype, int D, hipStream_t s);
int tile_attn_launch_bf16(const AttnArgs& a, int out_dtype, int D, hipStream_t s);
int tile_attn_launch_i8(const AttnArgs& a, int out_dtype, int D, hipStream_t s);
// The candidate kernel (pfa_cand_attn_<type>.hip), candidate rows without a mask.
int cand_attn_launch_f32(const AttnArgs& a, int out_dtype, int D, hipStream_t s);
int cand_attn_launch_f16(const AttnArgs& a, int out_dtype, int D, hipStream_t s);
int cand_attn_launch_bf16(const AttnArgs& a, int out_dtype, int D, hipStream_t s);
int cand_attn_launch_i8(const AttnArgs& a, int out_dtype, int D, hipStream_t s);

}  // namespace pfa
