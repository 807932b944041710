// dK / dV of a tile of 64 keys whose queries are a range of the sequence (compressed and window attention), head_dim 64 and 128,
// GQA groups of which a pass of 64 rows holds whole ones.  Same work list, partial sums and reduction as the kernel for gathered rows
// (dkdv_kernel.h), which remains for the other shapes and for q or dO that are not aligned.
//
// Two of the four waves share 32 keys, two 32 of the pass's rows: S = Q K^T, dP = dO V^T, dV^T += dO^T P and dK^T += Q^T dS of 32 rows
// and 32 keys, whose K (and, at head_dim 64, V) fragments stay in registers; the other V fragments lie in LDS in the order of the
// lanes.  (16 keys a wave, as for gathered rows, read every row of Q and dO twice as often: 128 KB of LDS traffic for 64 keys x 32
// rows, 1000 clocks beside 512 of products.)  Q, dO and the statistics of the next pass are on their way to LDS past the registers
// while this one is computed; exponentials stand beside the products of dP, dS beside those of dV.  No unit is full (4 x 8192 tokens:
// matrix 51 %, vector issue 49 %, LDS 40 %): the rest is the chain of a pass on two waves per SIMD, at the 1.7 GHz that the chip
// keeps up under this load.  Both branches of a layer, us, before -> after: 4 x 8192 tokens x 32 heads of 128, window 512, 1550 ->
// 1075; 5003 233 -> 161; 2 x 1000 x 8, window 128, 21.1 -> 17.4; 6000 x 32 heads of 64 152 -> 114.
#pragma once
#include "attn_rows.h"
#include "dkdv_kernel.h"

namespace fsa {

template <int D> struct DenseKv {
  static constexpr int ROWS = 64, NT = 256;                  // rows of a pass; four waves
  static constexpr int TILE = ROWS * D * 2;                  // Q or dO of a pass
  static constexpr int STAGE = 2 * TILE + ROWS * 8;          // Q, dO, [lse | delta] of the rows
  static constexpr int V_REGS = D >= 128 ? 1 : D / 16;  // k-steps of V that stay in registers; the others come from LDS
  static constexpr int BYTES = 2 * STAGE + 2 * (D / 16 - V_REGS) * 1024;   // (the epilogue's four 32 x D partial sums fit)
};

inline bool dense_kv_shape_ok(int g, int d) { return d <= 128 && g <= 64 && (g & (g - 1)) == 0; }
// Host: a pass has whole queries, rows are 16-byte aligned, and an offset from the first row of a pass to any of its rows has 32 bits
inline bool dense_kv_rows_ok(const void* q, int64_t q_sn, int64_t q_sh, const void* d_o, int64_t do_sn, int64_t do_sh, int64_t n_tokens,
                             int g, int d) {
  auto ok = [&](const void* x, int64_t sn, int64_t sh) {
    return ((uintptr_t)x % 16 | (sn | sh) % 8) == 0 && 2 * (66 * sn + g * sh + d) < (int64_t)0xFFFFFF00;
  };
  return dense_kv_shape_ok(g, d) && (n_tokens + 64) * g < (1 << 30) && ok(q, q_sn, q_sh) && ok(d_o, do_sn, do_sh);
}

// upper_seg by a whole wave: a look-up of a chain of log64 n loads, not log2 n
__device__ __forceinline__ int wave_upper_seg(const int32_t* __restrict__ a, int n, int x) {
  const int lane = threadIdx.x & 63;
  int lo = 0;
  for (int span = n; span > 1;) {   // a[lo] <= x, a[lo + span] > x (virtual)
    const int step = (span + 63) / 64, i = lane * step;
    const int below = __popcll(__ballot(i < span && a[lo + min(i, span - 1)] <= x));
    const int skip = (below - 1) * step;
    lo += skip;
    span = min(step, span - skip);
  }
  return lo;
}

template <typename T, int D, int MODE, bool GATED>
__device__ __forceinline__ void dense_dkdv_tile(const SelBwdParams& p, const int w, const int h) {
  typedef typename Elem<T>::vec8 vec8;
  typedef DenseKv<D> C;
  constexpr int BK = 64, NKS = D / 16, NDT = D / 32, CPR = D / 8, RPI = 64 / CPR, N = 16 / RPI;
  constexpr bool SHIFTED = GATED && std::is_same_v<T, _Float16>;   // as in attn_bwd_dkdv_tile
  constexpr float P_SHIFT = 15.f, P_UNDO = 0x1p-15f;
  const float ds_scale = SHIFTED ? p.scale * P_UNDO : p.scale;
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];

  const int64_t nbp1 = p.max_blocks + 1;
  const int32_t* tp = p.tile_prefix + h * nbp1;
  if (w >= tp[p.max_blocks]) return;
  const int gb = __builtin_amdgcn_readfirstlane(wave_upper_seg(tp, (int)p.max_blocks, w));
  KvBlock<MODE, BK> blk;
  blk.init(p, gb);
  const int rows = p.counts[h * p.max_blocks + gb] * p.g;
  const int ntile_b = tp[gb + 1] - tp[gb];
  const int share = ((rows + ntile_b - 1) / ntile_b + C::ROWS - 1) / C::ROWS * C::ROWS;
  const int row_lo = __builtin_amdgcn_readfirstlane((w - tp[gb]) * share);
  const int row_hi = __builtin_amdgcn_readfirstlane(min(rows, row_lo + share));

  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6), col = lane & 31, hh = lane >> 5;
  const int kgp = wv & 1, rh = wv >> 1;   // this wave's 32 keys, its 32 rows of a pass
  const int key = kgp * 32 + col, ktok = blk.key_row0 + key;
  const bool key_ok = key < blk.n_keys_valid;
  constexpr int NV = C::V_REGS;
  vec8 kf[NKS], vf[NV];
  const uint32_t lds = lds_addr(smem), v_lds = lds + 2 * C::STAGE + (kgp * (NKS - NV) * 64 + lane) * 16;
  const int q_first = blk.seq_start + blk.q_first, shift = p.g_shift, gmask = p.g - 1;
  // A pass on its way to a stage: load j of the wave takes RPI rows, the offset of which is one of the first row (scalar) plus one
  // of the lane.  Past the end of the share its last row again.
  const uint32_t q_sn = 2u * (uint32_t)p.q_sn, q_sh = 2u * (uint32_t)p.q_sh, do_sn = 2u * (uint32_t)p.do_sn, do_sh = 2u * (uint32_t)p.do_sh;
  const int ld_row = lane / CPR;
  const uint32_t q_lane = (ld_row >> shift) * q_sn + (ld_row & gmask) * q_sh, do_lane = (ld_row >> shift) * do_sn + (ld_row & gmask) * do_sh;
  // Statistics of the rows: pairs, or two arrays by head.
  const uint32_t st_t = p.stat2 ? 8u * p.hq : 4u, st_h = p.stat2 ? 8u : 4u * (uint32_t)p.n_tokens;
  const char* lse = p.stat2 ? reinterpret_cast<const char*>(p.stat2) : reinterpret_cast<const char*>(p.lse);
  const char* delta = p.stat2 ? lse + 4 : reinterpret_cast<const char*>(p.delta);
  auto issue = [&](int base, uint32_t stage) {
    const int64_t t0 = q_first + (base >> shift);
    const __amdgpu_buffer_rsrc_t qr = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<T*>(reinterpret_cast<const T*>(p.q) + t0 * p.q_sn + (int64_t)h * p.g * p.q_sh), 0, 0xFFFFFF00u, 0x00020000);
    const __amdgpu_buffer_rsrc_t dr = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<T*>(reinterpret_cast<const T*>(p.d_o) + t0 * p.do_sn + (int64_t)h * p.g * p.do_sh), 0, 0xFFFFFF00u, 0x00020000);
    const bool whole = base + C::ROWS <= row_hi;
#pragma unroll
    for (int j = 0; j < N; ++j) {
      const int u = wv * 16 + j * RPI;
      const uint32_t c = (uint32_t)((lane % CPR) ^ chunk_swizzle<D>(u + ld_row)) * 16;
      uint32_t qo = q_lane + c, oo = do_lane + c, qs = (u >> shift) * q_sn + (u & gmask) * q_sh, os = (u >> shift) * do_sn + (u & gmask) * do_sh;
      if (!whole) {
        const int r = min(base + u + ld_row, row_hi - 1) - base;
        qo = (r >> shift) * q_sn + (r & gmask) * q_sh + c;
        oo = (r >> shift) * do_sn + (r & gmask) * do_sh + c;
        qs = os = 0;
      }
      const uint32_t to = stage + (wv * N + j) * 1024;
      asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %1, %3 offen lds" :: "v"(qo), "s"(qr), "s"(to), "s"(qs) : "memory");
      asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %1, %3 offen lds" :: "v"(oo), "s"(dr), "s"(to + C::TILE), "s"(os) : "memory");
    }
    if (rh == 0) {   // one array each by two waves
      const int r = min(base + lane, row_hi - 1) - base;
      const uint32_t so = (r >> shift) * st_t + (r & gmask) * st_h;
      const __amdgpu_buffer_rsrc_t sr = __builtin_amdgcn_make_buffer_rsrc(
          const_cast<char*>((kgp ? delta : lse) + t0 * st_t + (int64_t)h * p.g * st_h), 0, 0xFFFFFF00u, 0x00020000);
      asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tbuffer_load_dword %0, %1, 0 offen lds" :: "v"(so), "s"(sr), "s"(stage + 2 * C::TILE + kgp * 256) : "memory");
    }
  };
  // First query, counted from the block's first, that sees a key of the block; the first that sees all of the wave's keys, and
  // (window) the last that still sees the first of them.  (Keys behind the end of the sequence have positions beyond any query's.)
  auto see = [&](int key_) {
    if (MODE == KV_MODE_WINDOW) return blk.key_base + key_ - blk.q_first;
    return (int)min((int64_t)(blk.key_base + key_) * p.kernel_stride + (p.kernel_size - 1 - blk.q_first), (int64_t)INT32_MAX);
  };
  const int see_all = see(32 * kgp + 31), see_first = MODE == KV_MODE_WINDOW ? see(32 * kgp) + p.window : INT32_MAX;

  f32x16 dk[NDT], dv[NDT];
#pragma unroll
  for (int t = 0; t < NDT; ++t)
#pragma unroll
    for (int i = 0; i < 16; ++i) dk[t][i] = dv[t][i] = 0.f;
  const TileFrags<D> f;

  auto pass = [&](int base, uint32_t stage) {
    const uint32_t q_tile = stage + rh * 32 * D * 2, o_tile = q_tile + C::TILE;
    const float* st = lds_ptr<float>(stage + 2 * C::TILE + (rh * 32 + 4 * hh) * 4);
    auto stat4 = [&](int which, int qd) { return *reinterpret_cast<const f32x4*>(st + which * 64 + 8 * qd); };
    constexpr int AHEAD = 2;
    vec8 fr[AHEAD + 1], vl[2];
    f32x16 s, dp;
#pragma unroll
    for (int i = 0; i < 16; ++i) s[i] = dp[i] = 0.f;
    // S, then dP with the exponentials beside it
    auto read = [&](int i) { fr[i % (AHEAD + 1)] = load16<vec8>(lds_ptr<T>((i < NKS ? q_tile : o_tile) + (f.k ^ (16u * (i % NKS))))); };
#pragma unroll
    for (int i = 0; i < AHEAD; ++i) read(i);
#pragma unroll
    for (int i = 0; i < 2 * NKS; ++i) {
      if (i + AHEAD < 2 * NKS) read(i + AHEAD);
      if (i + 1 - NKS >= NV && i + 1 < 2 * NKS) vl[(i + 1) % 2] = load16<vec8>(lds_ptr<T>(v_lds + (i + 1 - NKS - NV) * 1024));
      if (i < NKS) s = Elem<T>::mfma32(fr[i % (AHEAD + 1)], kf[i % NKS], s);
      else dp = Elem<T>::mfma32(fr[i % (AHEAD + 1)], i - NKS < NV ? vf[(i - NKS) % NV] : vl[i % 2], dp);
      if (i >= NKS) {
#pragma unroll
        for (int x = (i - NKS) * 16 / NKS; x < (i - NKS + 1) * 16 / NKS; ++x) {
          if (x % 4 == 0) {
            const f32x4 l4 = stat4(0, x / 4);
#pragma unroll
            for (int e = 0; e < 4; ++e) s[x + e] = s[x + e] * p.scale_log2 - (SHIFTED ? l4[e] - P_SHIFT : l4[e]);
          }
          s[x] = fast_exp2(s[x]);
          if ((x & 3) == 3) asm volatile("" : "+v"(s[x - 3]), "+v"(s[x - 2]), "+v"(s[x - 1]), "+v"(s[x]));   // (here, not in front of its use)
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    const int rb = base + 32 * rh;   // (the rows of the wave's share of the pass: does every one of them see all of the wave's keys?)
    if (!(rb + 32 <= row_hi && (rb >> shift) >= see_all && ((rb + 31) >> shift) <= see_first)) {
      asm volatile("" ::: "memory");   // (a branch, not selects in every pass)
      const int from = see(key), to = MODE == KV_MODE_WINDOW ? from + p.window : INT32_MAX;
#pragma unroll
      for (int x = 0; x < 16; ++x) {
        const int r = rb + 8 * (x >> 2) + 4 * hh + (x & 3), t = r >> shift;
        if (!(r < row_hi && t >= from && t <= to)) s[x] = 0.f;
      }
    }
    vec8 pk[2], dsk[2];
#pragma unroll
    for (int i = 0; i < 16; ++i) pk[i >> 3][i & 7] = (T)s[i];
    // dV with dS beside it, then dK
    constexpr int AH = 2;
    vec8 tr[AH + 1];
    auto readt = [&](int i) { tr[i % (AH + 1)] = swizzled_tr_frag<T, D>((i < 2 * NDT ? o_tile : q_tile) + (f.v ^ (64u * (i % NDT))), i / NDT % 2); };
#pragma unroll
    for (int i = 0; i < AH; ++i) readt(i);
#pragma unroll
    for (int i = 0; i < 4 * NDT; ++i) {
      if (i + AH < 4 * NDT) readt(i + AH);
      if (i < 2 * NDT) {
        dv[i % NDT] = Elem<T>::mfma32(tr[i % (AH + 1)], pk[i / NDT], dv[i % NDT]);
#pragma unroll
        for (int x = i * 8 / NDT; x < (i + 1) * 8 / NDT; ++x) {
          if (x % 4 == 0) {
            const f32x4 del = stat4(1, x / 4);
#pragma unroll
            for (int e = 0; e < 4; ++e) dp[x + e] -= del[e];
          }
          dsk[x >> 3][x & 7] = (T)(s[x] * dp[x] * ds_scale);
          if ((x & 7) == 7) asm volatile("" : "+v"(dsk[x >> 3]));
        }
      } else {
        dk[i % NDT] = Elem<T>::mfma32(tr[i % (AH + 1)], dsk[i / NDT - 2], dk[i % NDT]);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  if (row_lo < row_hi) {
    issue(row_lo, lds);
    // K and V of the block by way of the other stage: a load instruction of whole rows touches four of them instead of 32
    {
      const T* kb = reinterpret_cast<const T*>(p.k) + (int64_t)blk.key_row0 * p.k_sn + (int64_t)h * p.k_sh;
      const T* vb = reinterpret_cast<const T*>(p.v) + (int64_t)blk.key_row0 * p.v_sn + (int64_t)h * p.v_sh;
      constexpr int NL = BK * CPR / C::NT;
      vec8 xk[NL], xv[NL];
#pragma unroll
      for (int j = 0; j < NL; ++j) {
        const int r = j * (C::NT / CPR) + tid / CPR, c = tid % CPR * 8;
        xk[j] = xv[j] = zero8<T>();
        if (r < blk.n_keys_valid) {
          xk[j] = load16<vec8>(kb + (int64_t)r * p.k_sn + c);
          xv[j] = load16<vec8>(vb + (int64_t)r * p.v_sn + c);
        }
      }
#pragma unroll
      for (int j = 0; j < NL; ++j) {
        const int r = j * (C::NT / CPR) + tid / CPR, at = r * D + (tid % CPR ^ chunk_swizzle<D>(r)) * 8;
        store16(reinterpret_cast<T*>(smem + C::STAGE) + at, xk[j]);
        store16(reinterpret_cast<T*>(smem + C::STAGE + C::TILE) + at, xv[j]);
      }
    }
    tiles_arrived();
    const uint32_t k_tile = lds + C::STAGE + kgp * 32 * D * 2;
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) {
      kf[ks] = load16<vec8>(lds_ptr<T>(k_tile + (f.k ^ (16u * ks))));
      const vec8 x = load16<vec8>(lds_ptr<T>(k_tile + C::TILE + (f.k ^ (16u * ks))));
      if (ks < NV) vf[ks] = x;
      else if (rh == 0) store16(const_cast<T*>(lds_ptr<T>(v_lds + (ks - NV) * 1024)), x);
    }
    // settled in front of the loop
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) asm volatile("" : "+v"(kf[ks]));
#pragma unroll
    for (int ks = 0; ks < NV; ++ks) asm volatile("" : "+v"(vf[ks]));
    tiles_arrived();
    uint32_t stage = 0;
    for (int base = row_lo; base < row_hi; base += C::ROWS) {
      const uint32_t next = C::STAGE - stage;
      if (base + C::ROWS < row_hi) issue(base + C::ROWS, lds + next);
      pass(base, lds + stage);
      tiles_arrived();
      stage = next;
    }
  }

  // The two waves of 32 keys: the first keeps dK, the second dV, as [32][D] fp32 with 16-byte chunk c of row r at c ^ r.  The rows
  // leave whole: pieces of 32 bytes straight from the registers cost a work-group of one pass 5 us.
  constexpr int CH = D / 4, XM = CH - 1 < 31 ? CH - 1 : 31;
  f32x4* give = reinterpret_cast<f32x4*>(smem + wv * (32 * D * 4));
  f32x4* keep = reinterpret_cast<f32x4*>(smem + (wv ^ 2) * (32 * D * 4));
  auto piece = [&](const f32x16& x, int qd) { return f32x4{x[4 * qd], x[4 * qd + 1], x[4 * qd + 2], x[4 * qd + 3]}; };
#pragma unroll
  for (int t = 0; t < NDT; ++t)
#pragma unroll
    for (int qd = 0; qd < 4; ++qd) {
      const f32x4 a = piece(dk[t], qd), b = piece(dv[t], qd);
      give[col * CH + ((8 * t + 2 * qd + hh) ^ (col & XM))] = rh == 0 ? b : a;
    }
  __syncthreads();
#pragma unroll
  for (int t = 0; t < NDT; ++t)
#pragma unroll
    for (int qd = 0; qd < 4; ++qd) {
      f32x4* at = keep + col * CH + ((8 * t + 2 * qd + hh) ^ (col & XM));
      f32x4 x = (rh == 0 ? piece(dk[t], qd) : piece(dv[t], qd)) + *at;
      if constexpr (SHIFTED) x *= rh == 0 ? 1.f : P_UNDO;
      *at = x;
    }
  __builtin_amdgcn_wave_barrier();
  if (ntile_b == 1) {
    T* out = reinterpret_cast<T*>(rh == 0 ? p.dk : p.dv) + (int64_t)(blk.key_row0 + 32 * kgp) * p.dk_sn + (int64_t)h * p.dk_sh;
#pragma unroll
    for (int j = 0; j < 32 / RPI; ++j) {
      const int r = j * RPI + lane / CPR, c = 2 * (lane % CPR);
      const f32x4 lo = keep[r * CH + (c ^ (r & XM))], hi = keep[r * CH + ((c + 1) ^ (r & XM))];
      vec8 y;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        y[e] = (T)lo[e];
        y[4 + e] = (T)hi[e];
      }
      if (32 * kgp + r < blk.n_keys_valid) store16(out + (int64_t)r * p.dk_sn + 4 * c, y);
    }
  } else {
    f32x4* part = reinterpret_cast<f32x4*>(p.dkdv_part + ((int64_t)h * p.max_tiles + w) * (2 * BK * D) + (rh * BK + 32 * kgp) * D);
#pragma unroll
    for (int j = 0; j < 32 * CH / 64; ++j) {
      const int r = (j * 64 + lane) / CH, c = lane % CH;
      __builtin_nontemporal_store(keep[r * CH + (c ^ (r & XM))], part + j * 64 + lane);
    }
  }
}

template <typename T, int D, int MODE>
__global__ void __launch_bounds__(DenseKv<D>::NT, 2)
dense_dkdv_kernel(SelBwdParams p, HeadOrder order) {
  int h, w;
  head_tile(order, h, w);
  dense_dkdv_tile<T, D, MODE, false>(p, w, h);
}
// compressed and window attention of one layer in one launch: the first `na` work-groups of a kv head take tiles of a
template <typename T, int D>
__global__ void __launch_bounds__(DenseKv<D>::NT, 2)
dense_dkdv_pair_kernel(SelBwdParams a, SelBwdParams b, int na, HeadOrder order) {
  int h, w;
  head_tile(order, h, w);
  if (w < na) dense_dkdv_tile<T, D, KV_MODE_COMPRESSED, true>(a, w, h);
  else dense_dkdv_tile<T, D, KV_MODE_WINDOW, true>(b, w - na, h);
}

}  // namespace fsa
