// Packed attention over candidate lists on the matrix cores: sixteen rows of
// one head at a time, over the union of their lists.
//
// Neighbouring rows' candidates (a window, shared prototypes, anchors) mostly
// coincide.  A workgroup takes sixteen consecutive packed rows, marks every
// candidate in an LDS table (a 16-bit row mask per key, 8,192 keys at a time),
// compacts the marked keys into a list of (key, row mask), and its four waves
// take every fourth tile of that list: S^T = K Q^T with the rows that do not
// list a key at -inf, an online softmax, O^T += V^T P^T.  Lists in any order
// give the same sets.  A workgroup leaves its rows to the row kernel, launched
// behind it, by a flag (a.flags) where a list names a key twice (counted
// twice there), a result is not finite, or the lists share too little
// (kShare).  Precision is the tile kernel's (pfa_tile_attn.h).
//
// The row kernel fetches K and V once per (row, candidate) and multiplies on
// the vector unit; here they are fetched once per (sixteen rows, key).
// 16,400 rows of 8 heads x 64 dims, T = 8,192, 393 candidates a row: bf16 132
// -> 49 us, f32 139 -> 88 us.  Bound by latency: marking and listing a
// workgroup's keys takes about half of it, two workgroups fit a CU (72 KB of
// LDS, up to 256 VGPRs), and a tile's keys are gathered one tile ahead.
#pragma once

#include "pfa_tile_attn.h"

namespace pfa {
namespace cand {

using tile::exp2_p;
using tile::f32_swz;
using tile::i8_bf16;
using tile::kFused;
using tile::kParts;
using tile::kPScale;
using tile::mfma16;
using tile::negate_q;
using tile::normalise;
using tile::products_f32;
using tile::split_p;
using tile::store_n;
using tile::tree_sum;

constexpr int kRange = 8192;  // keys marked at a time
constexpr int kCap = 4096;    // listed keys between two flushes
constexpr int kFew = 1024;

template <int IDT, int D>
struct Cfg {
  static constexpr bool kF32 = IDT == PFA_F32;
  static constexpr int NH = D > 64 ? 2 : 1;
  static constexpr int TK = kF32 && D >= 64 ? 16 : 32;  // keys per tile
  static constexpr int NKB = TK / 16;
  static constexpr int NDC = D > 32 ? D / 32 : 1;
  static constexpr int NDB = D / 16;
  // Entries per listed key below which more than kFew listed keys are left to
  // the row kernel: a listed key costs as much here as this many entries there
  // (random lists of 512 over 8,192 keys, 1.6 entries a key, attended here: f32
  // 317 us, by rows 190).  Few keys stay in any case: the row kernel takes as
  // long for one row as for a full chip of them.
  static constexpr float kShare = kF32 ? 2.75f : 2.f;
  static constexpr int kVBytes = kF32 ? TK * D * 4 : TK * 128 * NH;  // V tile in LDS
};

template <int IDT, int D>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(D <= 64 ? 2 : 1, 8)))
cand_attn_kernel(AttnArgs a, int odt) {
  using C = Cfg<IDT, D>;
  using IT = typename Elem<IDT>::T;
  constexpr int TK = C::TK, NKB = C::NKB, NDC = C::NDC, NDB = C::NDB;
  __shared__ __align__(16) uint8_t vring[4][2][C::kVBytes];
  __shared__ __align__(16) uint32_t marks[kRange / 2];
  __shared__ __align__(16) int32_t ukey[kCap];
  __shared__ __align__(16) uint16_t umask[kCap];
  __shared__ int wsum[4], psum[4];
  __shared__ int s_more;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r16 = lane & 15, g = lane >> 4;
  const int64_t lb = remap_block(blockIdx.x, gridDim.x);
  const int64_t r0 = lb * 16;
  const int64_t nrow = attn_rows(a);
  if (r0 >= nrow) return;
  bool leave = false;  // some rows are left to the row kernel (uniform)
  // lane l < 16 of every wave: row l's token, head and list length
  int t_l = -1, h_l = -1, n_l = 0;
  if (lane < 16 && r0 + lane < nrow) {
    t_l = a.token_idx[r0 + lane];
    h_l = t_l >= 0 ? a.row_head[r0 + lane] : -1;
    n_l = (int)min<int64_t>(a.cand_len[r0 + lane], a.cand_stride);
  }
  SwzLane L;
  if constexpr (!C::kF32) L.init();
  const uint32_t vr_lds = __builtin_amdgcn_readfirstlane(lds_addr(&vring[0][0][0]) + (uint32_t)wid * 2u * C::kVBytes);
  const int osz = odt == PFA_F32 ? 4 : 2;

  for (int s0 = 0; s0 < 16;) {
    const int hp = __builtin_amdgcn_readlane(h_l, s0);
    const uint64_t other = __ballot(lane > s0 && (h_l != hp || lane >= 16));
    const int s1 = __builtin_ctzll(other);  // lane 16 is always among the others
    if (hp < 0) {
      s0 = s1;
      continue;
    }
    const int bh = a.head_map ? a.head_map[hp] : hp;
    const int64_t bb = bh / a.H, hh = bh % a.H;
    const IT* kb = (const IT*)a.k.ptr + bb * a.k.s_b + hh * a.k.s_h;
    const IT* vb = (const IT*)a.v.ptr + bb * a.v.s_b + hh * a.v.s_h;
    uint8_t* ob = (uint8_t*)a.out.ptr + (bb * a.out.s_b + hh * a.out.s_h) * osz;
    const int tq = __shfl(t_l, r16, 64);
    const bool qv = r16 >= s0 && r16 < s1;
    const IT* qp = (const IT*)a.q.ptr + bb * a.q.s_b + hh * a.q.s_h + (int64_t)(qv ? tq : 0) * a.q.s_t;

    // ---- the lane's query row ----
    bf16x8_t qf[NDC];
    f32x4_t qx[D / 16];
    if constexpr (C::kF32) {
#pragma unroll
      for (int j = 0; j < D / 16; ++j) qx[j] = *reinterpret_cast<const f32x4_t*>(qp + 16 * j + 4 * g);
    } else {
#pragma unroll
      for (int dc = 0; dc < NDC; ++dc) {
        qf[dc] = bf16x8_t{};
        if (D >= 32 || g < 2) {
          if constexpr (IDT == PFA_I8) {
            const uint2 w = *reinterpret_cast<const uint2*>(qp + 32 * dc + 8 * g);
            qf[dc] = i8_bf16(w.x, w.y);
          } else {
            qf[dc] = *reinterpret_cast<const bf16x8_t*>(qp + 32 * dc + 8 * g);
          }
        }
      }
    }
    float sl2 = a.scale * kLog2e;
    if constexpr (IDT == PFA_I8) sl2 *= a.q_scale[bh] * a.k_scale[bh];
    if (sl2 < 0.f) {  // (as in the tile kernel)
      sl2 = -sl2;
      negate_q<C::kF32>(qx, qf);
    }
    float m = -INFINITY, l = 0.f;
    f32x4_t acc[NDB];
#pragma unroll
    for (int db = 0; db < NDB; ++db) acc[db] = f32x4_t{0.f, 0.f, 0.f, 0.f};

    // ---- tiles of the key list: the wave's own, no barrier between them ----
    constexpr int kKReg = C::kF32 ? D / 16 : NDC;
    constexpr int kVr = IDT == PFA_I8 ? TK * (D / 8) / 64 : 1;
    struct Regs {
      uint4 k[kKReg][NKB];  // K fragments
      uint2 v[kVr];         // int8: V chunks (the others' V goes to LDS by DMA)
    };
    auto fetch = [&](int tile, int buf, Regs& x) {
      const int32_t* uk = ukey + tile * TK;
      if constexpr (IDT == PFA_I8) {
#pragma unroll
        for (int j = 0; j < kVr; ++j) {
          const int n = lane + 64 * j, row = n / (D / 8), c = n % (D / 8);
          x.v[j] = *reinterpret_cast<const uint2*>(vb + (int64_t)uk[row] * a.v.s_t + 8 * c);
        }
      } else {
#pragma unroll
        for (int j = 0; j < C::kVBytes / 1024; ++j) {
          const int slot = 64 * j + lane;
          int row, elem;
          if constexpr (C::kF32) {
            constexpr int CPR = D / 4;
            row = slot / CPR;
            elem = 4 * ((slot % CPR) ^ f32_swz<D>(row));
          } else {
            row = (slot / 8) % TK;
            elem = 64 * (slot / (8 * TK)) + 8 * (((slot & 7) ^ tile_swz(row)) & (D >= 64 ? 7 : D / 8 - 1));
          }
          lds_dma16(vb + (int64_t)uk[row] * a.v.s_t + elem, vr_lds + buf * C::kVBytes + 1024u * j);
        }
      }
#pragma unroll
      for (int b = 0; b < NKB; ++b) {
        const IT* kr = kb + (int64_t)uk[16 * b + r16] * a.k.s_t;
#pragma unroll
        for (int j = 0; j < kKReg; ++j) {
          if constexpr (C::kF32) x.k[j][b] = *reinterpret_cast<const uint4*>(kr + 16 * j + 4 * g);
          else if constexpr (IDT == PFA_I8) {
            const uint2 w = *reinterpret_cast<const uint2*>(kr + 32 * j + 8 * (D >= 32 ? g : g & 1));
            x.k[j][b] = make_uint4(w.x, w.y, 0u, 0u);
          } else x.k[j][b] = *reinterpret_cast<const uint4*>(kr + 32 * j + 8 * (D >= 32 ? g : g & 1));
        }
      }
    };
    auto compute = [&](int tile, int buf, const Regs& x) {
      f32x4_t c[NKB];
      if constexpr (C::kF32) {
#pragma unroll
        for (int b = 0; b < NKB; ++b) {
          f32x4_t ka[D / 16];
#pragma unroll
          for (int j = 0; j < D / 16; ++j) __builtin_memcpy(&ka[j], &x.k[j][b], 16);
          c[b] = products_f32<D / 16>([&](int n) { return ka[n >> 2][n & 3]; }, [&](int n) { return qx[n >> 2][n & 3]; });
        }
      } else {
#pragma unroll
        for (int dc = 0; dc < NDC; ++dc)
#pragma unroll
          for (int b = 0; b < NKB; ++b) {
            bf16x8_t ka;
            if constexpr (IDT == PFA_I8) ka = i8_bf16(x.k[dc][b].x, x.k[dc][b].y);
            else __builtin_memcpy(&ka, &x.k[dc][b], 16);
            c[b] = mfma16<IDT>(ka, qf[dc], dc == 0 ? f32x4_t{0.f, 0.f, 0.f, 0.f} : c[b]);
          }
      }
      if constexpr (IDT == PFA_I8) {
#pragma unroll
        for (int j = 0; j < kVr; ++j) {
          const int n = lane + 64 * j, row = n / (D / 8), ch = n % (D / 8);
          const bf16x8_t h = i8_bf16(x.v[j].x, x.v[j].y);
          __builtin_memcpy(__builtin_assume_aligned(&vring[wid][buf][(ch >> 3) * TK * 128 + row * 128 +
                                                                      16 * ((ch & 7) ^ tile_swz(row))], 16), &h, 16);
        }
        wave_sync();
      }
      // scores (unscaled where kFused); -inf where the row does not list the key
      float s[NKB][4], tmax = -INFINITY;
#pragma unroll
      for (int b = 0; b < NKB; ++b) {
        const uint2 mw = *reinterpret_cast<const uint2*>(umask + tile * TK + 16 * b + 4 * g);
        const uint32_t mk[4] = {mw.x, mw.x >> 16, mw.y, mw.y >> 16};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          s[b][i] = (mk[i] >> r16) & 1u ? (kFused<IDT> ? c[b][i] : c[b][i] * sl2) : -INFINITY;
          tmax = fmaxf(tmax, s[b][i]);
        }
      }
      tmax = max_over_rows4(tmax);
      if constexpr (kFused<IDT>) tmax *= sl2;  // sl2 > 0, -inf stays
      if (__ballot(tmax > m) != 0) {
        const float mn = fmaxf(m, tmax);
        const float alpha = mn == -INFINITY ? 1.f : exp2_p<IDT>(m - mn);
        l *= alpha;
#pragma unroll
        for (int db = 0; db < NDB; ++db)
#pragma unroll
          for (int i = 0; i < 4; ++i) acc[db][i] *= alpha;
        m = mn;
      }
      const float moff = m == -INFINITY ? 0.f : m;
      float ps[NKB];
#pragma unroll
      for (int b = 0; b < NKB; ++b) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float x = kFused<IDT> ? __builtin_fmaf(s[b][i], sl2, -moff) : s[b][i] - moff;
          s[b][i] = exp2_p<IDT>(x) * kPScale<IDT>;
        }
        ps[b] = (s[b][0] + s[b][1]) + (s[b][2] + s[b][3]);
      }
      l += tree_sum(ps);
      if constexpr (C::kF32) {
        const float* vt = (const float*)&vring[wid][buf][0];
        float va[4 * NKB][NDB];
#pragma unroll
        for (int n = 0; n < 4 * NKB; ++n) {
          const int row = 16 * (n >> 2) + 4 * g + (n & 3);
          const float* vr = vt + row * D;
          if constexpr (NDB >= 4) {
#pragma unroll
            for (int h = 0; h < NDB / 4; ++h)
              __builtin_memcpy(va[n] + 4 * h, __builtin_assume_aligned(vr + 4 * ((16 * h + r16) ^ f32_swz<D>(row)), 16), 16);
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
        const uint16_t* vt = (const uint16_t*)&vring[wid][buf][0];
        float p[8];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          p[i] = s[0][i];
          p[4 + i] = s[NKB - 1][i];
        }
        bf16x8_t part[kParts];
        split_p<IDT>(p, part);
#pragma unroll
        for (int db = 0; db < NDB; ++db) {
          const uint16_t* vr = vt + (db >> 2) * TK * 64 + L.vo[db & 3];
          const i16x4_t v0 = ds_tr4(vr), v1 = ds_tr4(vr + 64 * 16);
          bf16x8_t va;
          __builtin_memcpy(&va, &v0, 8);
          __builtin_memcpy(reinterpret_cast<char*>(&va) + 8, &v1, 8);
#pragma unroll
          for (int n = kParts - 1; n >= 0; --n) acc[db] = mfma16<IDT>(va, part[n], acc[db]);
        }
      }
    };
    // The list's cnt keys, then the list is free again.  Entered and left with
    // the whole workgroup.
    bool begun = false;
    auto flush = [&](int cnt) {
      begun = true;
      const int ntile = (cnt + TK - 1) / TK;
      if (cnt + tid < ntile * TK) {  // fewer than 256 entries of padding
        ukey[cnt + tid] = ukey[cnt - 1];
        umask[cnt + tid] = 0;
      }
      __syncthreads();
      // the wave's tiles, one in flight while one is computed
      Regs x0, x1;
      int t = wid;
      if (t < ntile) {
        fetch(t, 0, x0);
        for (;;) {
          asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
          if (t + 4 < ntile) fetch(t + 4, 1, x1);
          compute(t, 0, x0);
          if ((t += 4) >= ntile) break;
          asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
          if (t + 4 < ntile) fetch(t + 4, 0, x0);
          compute(t, 1, x1);
          if ((t += 4) >= ntile) break;
        }
      }
      __syncthreads();
    };

    // ---- mark, list, attend ----
    // Wave w marks the rows 4w .. 4w+3.  Their lists' first 512 entries stay in
    // registers (one memory latency, for every range of keys); the rest of a
    // longer list is read again for each range.
    constexpr int kReg = 8;  // entries per lane and row
    int kk[4][kReg], nr[4];
    int nmax = 0;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = 4 * wid + r;
      nr[r] = row >= s0 && row < s1 ? __builtin_amdgcn_readlane(n_l, row) : 0;
      nmax = max(nmax, nr[r]);
    }
    auto load_entries = [&](int i0) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int32_t* crow = a.cand + (r0 + 4 * wid + r) * a.cand_stride;
#pragma unroll
        for (int j = 0; j < kReg; ++j) {
          const int i = i0 + 64 * j + lane;
          kk[r][j] = i < nr[r] ? crow[i] : INT32_MIN;
        }
      }
    };
    load_entries(0);
    int pairs = 0;  // distinct (row, key) pairs that this thread saw in the table
    auto all_pairs = [&]() {  // of the workgroup (which it synchronises)
      int n = pairs;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) n += __shfl_xor(n, o, 64);
      if (lane == 0) psum[wid] = n;
      __syncthreads();
      return psum[0] + psum[1] + psum[2] + psum[3];
    };
    bool skip = false;  // this segment is left to the row kernel (uniform)
    int cnt = 0;  // listed keys (uniform)
    for (int64_t base = 0; base < a.T; base += kRange) {
#pragma unroll
      for (int j = 0; j < kRange / 2 / 4 / 256; ++j)  // 16 bytes each
        reinterpret_cast<uint4*>(marks)[tid + 256 * j] = make_uint4(0u, 0u, 0u, 0u);
      if (tid == 0) s_more = 0;
      __syncthreads();
      bool more = false;
      for (int i0 = 0; i0 < nmax; i0 += 64 * kReg) {
        if (nmax > 64 * kReg && (i0 > 0 || base > 0)) load_entries(i0);
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
          for (int j = 0; j < kReg; ++j) {
            if (i0 + 64 * j >= nr[r]) continue;  // uniform
            const int e = kk[r][j];
            const bool has = i0 + 64 * j + lane < nr[r];
            const int o = min(max(e, 0), (int)a.T - 1) - (int)base;
            if (has && o >= 0 && o < kRange) atomicOr(&marks[o >> 1], 1u << (4 * wid + r + 16 * (o & 1)));
            more |= has && o >= kRange;
          }
      }
      if (more) s_more = 1;
      __syncthreads();
      // 32 keys per thread
      constexpr int kW = kRange / 2 / 256;
      uint32_t w[kW];
      __builtin_memcpy(w, &marks[kW * tid], 4 * kW);
      int mine = 0;
#pragma unroll
      for (int j = 0; j < kW; ++j) {
        mine += ((w[j] & 0xffffu) != 0) + ((w[j] >> 16) != 0);
        pairs += __popc(w[j]);
      }
      int incl = mine;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const int y = __shfl_up(incl, o, 64);
        if (lane >= o) incl += y;
      }
      if (lane == 63) wsum[wid] = incl;
      const bool again = s_more != 0;
      __syncthreads();
      int pos = incl - mine, total = 0;
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        pos += k < wid ? wsum[k] : 0;
        total += wsum[k];
      }
      // into the list, in halves of the range when they do not fit together
      const bool whole = cnt + total <= kCap;
      if (!whole && !begun && (float)all_pairs() < C::kShare * (float)(cnt + total)) {
        skip = true;
        break;
      }
      if (!whole && cnt > 0) {
        flush(cnt);
        cnt = 0;
      }
      const bool split = total > kCap;  // more than half of the range is listed
      int at = pos + cnt;
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        // half 0: everything, or the threads of the first half of the range
        const bool take = half == 0 ? (!split || tid < 128) : (split && tid >= 128);
        if (half == 1) {
          if (!split) break;
          const int first = wsum[0] + wsum[1];
          __syncthreads();
          if (first > 0) flush(first);
          at = pos - first;
          total -= first;
        }
        if (take) {
#pragma unroll
          for (int j = 0; j < 2 * kW; ++j) {
            const uint32_t mk = (w[j >> 1] >> (16 * (j & 1))) & 0xffffu;
            if (mk != 0) {
              ukey[at] = (int)base + 2 * kW * tid + j;
              umask[at] = (uint16_t)mk;
              ++at;
            }
          }
        }
      }
      cnt += total;
      __syncthreads();
      if (!again) break;
    }
    int entries = lane >= s0 && lane < s1 ? n_l : 0;
#pragma unroll
    for (int o = 1; o < 16; o <<= 1) entries += __shfl_xor(entries, o, 64);
    entries = __builtin_amdgcn_readlane(entries, 0);
    // every list's entries found once: otherwise a list names a key twice
    if (!skip) {
      const int seen = all_pairs();
      skip = seen != entries || (!begun && cnt > kFew && (float)seen < C::kShare * (float)cnt);
    }
    if (skip) {
      leave = true;
      __syncthreads();
      s0 = s1;
      continue;
    }
    if (cnt > 0) flush(cnt);

    // ---- the waves' states meet in LDS: wave 0 merges and stores ----
    l += __shfl_xor(l, 16, 64);
    l += __shfl_xor(l, 32, 64);
    constexpr int W = 4 * NDB + 2;
    static_assert(3 * W * 64 * 4 <= 8 * C::kVBytes, "merge area");
    float* area = (float*)&vring[0][0][0];
    if (wid > 0) {
      float* mine = area + (wid - 1) * W * 64 + lane;
      mine[0] = m;
      mine[64] = l;
#pragma unroll
      for (int db = 0; db < NDB; ++db)
#pragma unroll
        for (int i = 0; i < 4; ++i) mine[64 * (2 + 4 * db + i)] = acc[db][i];
    }
    __syncthreads();
    if (wid == 0) {
      for (int k = 0; k < 3; ++k) {
        const float* o = area + k * W * 64 + lane;
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
      bool bad = false;
      const float inv = 1.f / l;
      const float vs = IDT == PFA_I8 ? a.v_scale[bh] : 1.f;
#pragma unroll
      for (int db = 0; db < NDB; ++db)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          acc[db][i] = normalise<IDT>(acc[db][i], l, inv, vs);
          bad |= !(fabsf(acc[db][i]) <= 3.402823466e38f);
          if (l == 0.f) acc[db][i] = __builtin_nanf("");  // every score -inf, or no candidate
        }
      leave = leave || __ballot(bad && qv && l != 0.f) != 0;
      if (qv) {
        void* orow = ob + (int64_t)tq * a.out.s_t * osz;
        if constexpr (C::kF32) {
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
    }
    __syncthreads();  // LDS is free for the next segment
    s0 = s1;
  }
  if (tid == 0) a.flags[lb] = leave ? 1 : 0;  // (wave 0 holds the non-finite results)
}

template <int IDT, int D>
static int launch_d(const AttnArgs& a, int odt, hipStream_t s) {
  int64_t blocks = (a.N + 15) / 16;
  blocks = (blocks + 7) / 8 * 8;
  PFA_CHECK_ARG(blocks < INT32_MAX, "pfa_sparse_attn_fwd: too many rows");
  cand_attn_kernel<IDT, D><<<(unsigned)blocks, 256, 0, s>>>(a, odt);
  PFA_CHECK_LAUNCH("pfa_sparse_attn_fwd");
  return PFA_OK;
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

}  // namespace cand
}  // namespace pfa
