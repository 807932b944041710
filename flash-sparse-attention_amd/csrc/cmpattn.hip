// Compressed attention (queries against the compressed keys / values), the
// block-importance scores derived from it and the top-k block selection, gfx950.
//
//   cmpattn_fwd   : query-major flash attention over tiles of 32 compressed keys
//                   that go straight to LDS; rows are (query, head-in-group) pairs so one
//                   K/V tile serves the whole GQA group; S^T = K Q^T with one row
//                   per lane, online softmax in registers, O^T += V^T P^T.
//   cmpattn_bwd   : delta, a query-major dQ kernel of the same shape, and the
//                   key-major dK/dV kernel (dense_dkdv.h, dkdv_kernel.h).
//   cmp_score     : probabilities of the first head of every group, fp32.
//   cmp_topk      : per query: weighted 5-tap re-binning into selection blocks,
//                   forced blocks, cast to bf16, top-k by (value desc, id asc),
//                   ascending ids, ids above the own block -> -1.
//
// Semantics: nsa_ref/ops/compressed_attention.py:27-156 (forward; key j visible
// to query i iff i >= j*stride + ks - 1, rows without a visible key give O = 0,
// LSE = -inf), :195-518 (backward), :832-930 (score), :1006-1158 (transform),
// :1272-1315 (selection).
#include "attn_rows.h"
#include "dkdv_kernel.h"
#include "dense_dkdv.h"

#include <algorithm>

namespace fsa {

struct CmpParams {
  const void* q;
  const void* k;
  const void* v;
  const void* d_o;
  void* o;
  void* dq;
  float* lse;          // [Hq, N]
  const float* delta;  // [Hq, N]
  const float2* stat2; // backward, optional: (lse, delta) pairs [N, Hq] instead of the two arrays above
  int64_t q_sn, q_sh, k_sn, k_sh, v_sn, v_sh, o_sn, o_sh, do_sn, do_sh;
  const int32_t* cu_q;
  const int32_t* cu_k;
  int64_t n_tokens;
  int g, hkv;
  int nx;              // query tiles of the longest sequence
  int kernel_size, kernel_stride;
  int window;  // sliding-window mode: key p visible to query i iff i - window <= p <= i
  float scale, scale_log2;
  // score / top-k
  float* score;        // [Hkv, N, score_ld]
  int64_t score_ld;
  int score_head_step;  // q head that scores kv head h = h * score_head_step (g: first head of the group)
  int rebin;           // cmp_score writes block scores (taps 1 2 2 2 1 over groups of 4 keys) instead of probabilities
};

constexpr int CMP_MODE_COMPRESSED = 0;
constexpr int CMP_MODE_WINDOW = 1;   // the same query-major kernels over raw keys with a causal band mask
constexpr int CMP_BK = 64;      // compressed keys per tile
constexpr int CMP_ROWS = 128;   // rows per work-group (4 waves x 32)

template <int D> struct CmpLds {   // keys of the score kernel
  static constexpr int KS = D + 8;  // 16 B pad: fragments of 16 bytes from 32 rows without bank conflicts
  static constexpr int BYTES = CMP_BK * KS * 2;
};

// A tile of CMP_BK keys travels as 16-byte chunks, chunk c = tid + 256 j of thread tid: row c / (D / 8),
// which is tid / (D / 8) + j * ROWS_PER_STEP.  The loads are buffer loads: step j has a scalar descriptor of its
// own (first row of the step, as many bytes as the step has rows left in the sequence) and every step uses the
// same 32-bit lane offset (k_tile_offset), which never changes - no per-load vector arithmetic at all, and the
// rows past the end of the sequence (last tile only) come back as zeros from the descriptor's range check.
template <typename T, int D>
__device__ __forceinline__ uint32_t k_tile_offset(int64_t sn, int tid) {
  constexpr int CPR = D / 8;
  return (uint32_t)((tid / CPR) * sn * (int64_t)sizeof(T)) + (tid % CPR) * 16;   // host: CMP_BK * sn * sizeof(T) < 2^32
}
template <typename T, int D>
__device__ __forceinline__ void stage_k_tile(const T* base, int64_t sn, uint32_t off, int row0, int n_valid, T* Ks, int tid) {
  constexpr int CPR = D / 8, RPS = 256 / CPR, N = CMP_BK / RPS;   // chunks per row, rows per step, steps
  const int64_t row_bytes = sn * (int64_t)sizeof(T);
  const char* tile = reinterpret_cast<const char*>(base) + row0 * row_bytes;
  typename Elem<T>::vec8 r[N];
#pragma unroll
  for (int j = 0; j < N; ++j) {
    const int rows = min(n_valid - j * RPS, RPS);  // rows of this step inside the sequence
    const uint32_t bytes = rows > 0 ? (uint32_t)((rows - 1) * row_bytes) + D * (uint32_t)sizeof(T) : 0u;
    const __amdgpu_buffer_rsrc_t rsrc =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(tile + j * RPS * row_bytes), 0, (int)bytes, 0x00020000);
    r[j] = __builtin_bit_cast(typename Elem<T>::vec8, __builtin_amdgcn_raw_buffer_load_b128(rsrc, off, 0, 0));
  }
#pragma unroll
  for (int j = 0; j < N; ++j) store16(&Ks[(tid / CPR + j * RPS) * CmpLds<D>::KS + tid % CPR * 8], r[j]);
}

// Work-group -> (query tile, sequence, kv head).  Consecutive work-groups go to the eight XCDs in turn: with the kv head
// running fastest an XCD keeps to few heads, whose keys and values then stay in its L2.  The tiles of a sequence run from
// its end: late queries see the most compressed keys, and the long tiles should not start last.  Many sequences and a long
// one among them: the sequences go into the second dimension of the grid (dense_grid).
__device__ __forceinline__ void tile_of(const CmpParams& p, int id, int& x, int& s, int& h) {
  h = id % p.hkv;
  const int rest = id / p.hkv;
  x = p.nx - 1 - rest % p.nx;
  s = blockIdx.y + rest / p.nx;
}

// Per-row and per-work-group visible key range [lo, hi] (inclusive) in both modes.
template <int MODE> struct KeyRange {
  static __device__ __forceinline__ int hi(const CmpParams& p, int qi, int nc) {
    if (MODE == CMP_MODE_WINDOW) return min(qi, nc - 1);
    const int j = qi >= p.kernel_size - 1 ? (qi - p.kernel_size + 1) / p.kernel_stride : -1;
    return min(j, nc - 1);
  }
  static __device__ __forceinline__ int lo(const CmpParams& p, int qi) {
    return MODE == CMP_MODE_WINDOW ? max(0, qi - p.window) : 0;
  }
};

// ---------------------------------------------------------------- forward ----
// Four waves of 32 rows share the tiles of K and V, 32 keys a step, two tiles of each in LDS; the products of one step stand beside
// the exponentials of another.  What a step takes, about 1 us for the two waves of a SIMD, is less than half of it products; a
// work-group has 6 us in front of and behind its steps, with one other work-group on the CU to cover them.  Hence q and o by way
// of LDS, too: a load or store instruction of whole rows touches four of them, not 32 (16384 tokens x 8 heads of 256 138 -> 120
// us).  Against 64-key tiles by way of the registers, products and exponentials in turn, window of 512 / compressed, us: 5003 x 32
// heads of 128 74 -> 64 / 37 -> 32, 4 x 8192 x 32 400 -> 362 / 248 -> 221, 5003 x 32 of 64 42 -> 36 / 21 -> 18, 16384 x 8 of 256
// 148 -> 117 / 129 -> 100.
template <typename T, int D> struct CmpFwdLds {
  static constexpr int TILE = TileLoads<T, D>::BYTES, BYTES = 8 * TILE;   // two tiles of K, two of V, one of q / o for every wave
};
// ANY: keys or values that are not aligned, or whose rows lie on top of each other.
template <typename T, int D, int MODE, bool ANY>
__device__ __forceinline__ void attn_fwd_tile(const CmpParams& p, int id) {
  typedef typename Elem<T>::vec8 vec8;
  typedef TileLoads<T, D, ANY> Loads;
  constexpr int TILE = Loads::BYTES;
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];

  int bx, s, h;
  tile_of(p, id, bx, s, h);
  const int q0 = p.cu_q[s], lq = p.cu_q[s + 1] - q0;
  const int k0 = MODE == CMP_MODE_WINDOW ? q0 : p.cu_k[s];
  const int nc = MODE == CMP_MODE_WINDOW ? lq : p.cu_k[s + 1] - k0;
  const int rows_total = lq * p.g;
  const int row_lo = bx * CMP_ROWS;
  if (row_lo >= rows_total) return;
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), col = lane & 31, hh = lane >> 5;
  const int row = row_lo + wv * 32 + col;
  const bool valid = row < rows_total;
  const int rr = valid ? row : rows_total - 1;
  const int qi = rr / p.g, hq_i = h * p.g + rr - qi * p.g;
  // the range of keys of the work-group, in steps of 32
  const int qi_first = row_lo / p.g, qi_last = (min(rows_total, row_lo + CMP_ROWS) - 1) / p.g;
  const int jt0 = __builtin_amdgcn_readfirstlane(KeyRange<MODE>::lo(p, qi_first) & ~31);
  const int n_steps = __builtin_amdgcn_readfirstlane((KeyRange<MODE>::hi(p, qi_last, nc) + 1 - jt0 + 31) >> 5);
  const Loads kl(p.k, p.k_sn, p.k_sh, k0, h, nc), vl(p.v, p.v_sn, p.v_sh, k0, h, nc);
  const uint32_t k_lds = lds_addr(smem), v_lds = k_lds + 2 * TILE;
  // this wave's share of a tile: even waves K, odd ones V, each half a tile where that has loads enough
  constexpr int PARTS = Loads::N >= 2 * Loads::NV ? 2 : 1;
  auto issue_k = [&](int t) {
    if ((wv & 1) == 0 && wv < 2 * PARTS) kl.template issue<PARTS>(jt0 + 32 * t, k_lds + (t & 1) * TILE, wv >> 1);
  };
  auto issue_v = [&](int t) {
    if ((wv & 1) == 1 && wv < 2 * PARTS) vl.template issue<PARTS>(jt0 + 32 * t, v_lds + (t & 1) * TILE, wv >> 1);
  };
  // ANY: every wave requests a quarter of either tile at the start of a step and puts it into LDS at its end.  (Put there at once,
  // as in front of the loop, the waves waited for every tile: keys and values one element off, window / compressed, us, 16384 x 32 of
  // 128 285 / 296 -> 213 / 199, 16384 x 16 of 64 114 / 107 -> 64 / 58, 9000 x 8 of 256 215 / 104 -> 118 / 63; 64-key tiles 241 / 210, 72 /
  // 60, 139 / 73.)
  vec8 next_k[Loads::N / 4], next_v[Loads::N / 4];
  auto fetch = [&](int t) {
    kl.template fetch<4>(next_k, jt0 + 32 * (t + 2), wv);
    vl.template fetch<4>(next_v, jt0 + 32 * (t + 1), wv);
  };
  auto land = [&](uint32_t k_to, uint32_t v_to) {
    kl.template land<4>(next_k, k_to, wv);
    vl.template land<4>(next_v, v_to, wv);
  };
  AttnRows<T, D> r;
  r.scale_log2 = p.scale_log2;
  r.clear();
  T* rows_lds = reinterpret_cast<T*>(smem + (4 + wv) * TILE);
  if (n_steps > 0) {
    issue_k(0);
    issue_v(0);
    issue_k(1);
    const int jmax = KeyRange<MODE>::hi(p, qi, nc) - jt0, jmin = KeyRange<MODE>::lo(p, qi) - jt0;
    auto mask = [&](f32x16& x, int t) {   // a step that every row of the wave sees completely needs none
      const int limit = jmax - 32 * t, limit_lo = jmin - 32 * t;
      if (!__all(limit >= 31 && limit_lo <= 0)) {
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const int key = 8 * (i >> 2) + 4 * hh + (i & 3);
          if (!(key <= limit && key >= limit_lo)) x[i] = -INFINITY;
        }
      }
    };
    const TileFrags<D> f;
    r.load_q_rows(reinterpret_cast<const T*>(p.q) + (int64_t)(q0 + qi) * p.q_sn + (int64_t)hq_i * p.q_sh, rows_lds, f);
    vec8 pk[2];
    auto step = [&](f32x16& x, f32x16& next, int t) {   // scores of this step in x, those of the next one into `next`
      tiles_arrived();   // K of the next step, V of this one
      if constexpr (ANY) {
        fetch(t);
      } else {
        issue_k(t + 2);    // (behind the last key: zeros, and nothing is read)
        issue_v(t + 1);
      }
      r.template scores<true>(next, x, r.reference(true), pk, k_lds + ((t + 1) & 1) * TILE, f);
      mask(next, t + 1);
      r.raise(r.values(next, pk, v_lds + (t & 1) * TILE, f), true);
      if constexpr (ANY) land(k_lds + (t & 1) * TILE, v_lds + ((t + 1) & 1) * TILE);
    };
    f32x16 sa, sb;
    tiles_arrived();
    r.template scores<false>(sa, sb, 0.f, pk, k_lds, f);
    mask(sa, 0);
    r.raise(r.lane_max(sa), true);
    for (int t = 0;;) {
      step(sa, sb, t);
      if (++t >= n_steps) break;
      step(sb, sa, t);
      if (++t >= n_steps) break;
    }
    vm_wait<0>();
  }
  r.l = sum32(r.l);
  r.store_rows(reinterpret_cast<T*>(p.o) + (int64_t)(q0 + qi) * p.o_sn + (int64_t)hq_i * p.o_sh, valid, r.l > 0.f ? 1.f / r.l : 0.f, rows_lds);
  if (valid && hh == 0) p.lse[(int64_t)hq_i * p.n_tokens + q0 + qi] = r.l > 0.f ? r.mref + log2f(r.l) : -INFINITY;
}

// --------------------------------------------------------------------- dq ----
// The structure of the forward: dP of a step beside its exponentials, scores of the next step beside dS of this one, then the products
// of K^T and dS; K of two steps and what is on its way in three tiles.  Matrix unit 50 %, vector issue 47 %, LDS 36 %: as in the kernel
// of dK / dV, the chain of a step is the rest.  Against 64-key tiles by way of the registers, phases in turn, q, dO and dQ in pieces of
// 16 bytes, both branches of a layer, us: 4 x 8192 tokens x 32 heads of 128, window 512, 980 -> 778; 12000 x 32 336 -> 276; 5003 x 32
// 143 -> 118; 2 x 1000 x 8, window 128, 21.3 -> 15.6; 6000 x 32 of 64 100 -> 84; window alone, 9000 x 8 of 256, 128 -> 127.  At head_dim
// 256 the registers do not suffice: 28 of either branch and 52 of both in one launch are spilled, which leaves it level (both, 9000 x
// 8 194 -> 194, 16384 x 16 720 -> 703).
template <typename T, int D> struct CmpDqLds {
  static constexpr int TILE = TileLoads<T, D>::BYTES, BYTES = 9 * TILE;   // three tiles of K, two of V, one of q / dO / dQ for every wave
};
template <typename T, int D, int MODE, bool ANY>
__device__ __forceinline__ void attn_bwd_dq_tile(const CmpParams& p, int id) {
  typedef typename Elem<T>::vec8 vec8;
  typedef TileLoads<T, D, ANY> Loads;
  constexpr int TILE = Loads::BYTES, NKS = D / 16, NDT = D / 32;
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];

  int bx, s, h;
  tile_of(p, id, bx, s, h);
  const int q0 = p.cu_q[s], lq = p.cu_q[s + 1] - q0;
  const int k0 = MODE == CMP_MODE_WINDOW ? q0 : p.cu_k[s];
  const int nc = MODE == CMP_MODE_WINDOW ? lq : p.cu_k[s + 1] - k0;
  const int rows_total = lq * p.g;
  const int row_lo = bx * CMP_ROWS;
  if (row_lo >= rows_total) return;
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), col = lane & 31, hh = lane >> 5;
  const int row = row_lo + wv * 32 + col;
  const bool valid = row < rows_total;
  const int rr = valid ? row : rows_total - 1;
  const int qi = rr / p.g, hq_i = h * p.g + rr - qi * p.g;
  // the range of keys of the work-group, in steps of 32
  const int qi_first = row_lo / p.g, qi_last = (min(rows_total, row_lo + CMP_ROWS) - 1) / p.g;
  const int jt0 = __builtin_amdgcn_readfirstlane(KeyRange<MODE>::lo(p, qi_first) & ~31);
  const int n_steps = __builtin_amdgcn_readfirstlane((KeyRange<MODE>::hi(p, qi_last, nc) + 1 - jt0 + 31) >> 5);
  const Loads kl(p.k, p.k_sn, p.k_sh, k0, h, nc), vl(p.v, p.v_sn, p.v_sh, k0, h, nc);
  const uint32_t k_lds = lds_addr(smem), v_lds = k_lds + 3 * TILE;
  // this wave's share of a tile: as in the forward
  constexpr int PARTS = Loads::N >= 2 * Loads::NV ? 2 : 1;
  auto issue_k = [&](int t, uint32_t to) {
    if ((wv & 1) == 0 && wv < 2 * PARTS) kl.template issue<PARTS>(jt0 + 32 * t, to, wv >> 1);
  };
  auto issue_v = [&](int t) {
    if ((wv & 1) == 1 && wv < 2 * PARTS) vl.template issue<PARTS>(jt0 + 32 * t, v_lds + (t & 1) * TILE, wv >> 1);
  };
  // ANY: as in the forward; window / compressed, us, 16384 x 32 of 128 337 / 386 -> 297 / 261, 16384 x 16 of 64 121 / 130 -> 79 / 73,
  // 9000 x 8 of 256 258 / 184 -> 158 / 83; 64-key tiles 304 / 286, 88 / 82, 155 / 83
  vec8 next_k[Loads::N / 4], next_v[Loads::N / 4];
  auto fetch = [&](int t) {
    kl.template fetch<4>(next_k, jt0 + 32 * (t + 2), wv);
    vl.template fetch<4>(next_v, jt0 + 32 * (t + 1), wv);
  };
  auto land = [&](uint32_t k_to, uint32_t v_to) {
    kl.template land<4>(next_k, k_to, wv);
    vl.template land<4>(next_v, v_to, wv);
  };
  AttnRows<T, D> r;   // q, and dQ in its accumulators
  r.clear();
  T* rows_lds = reinterpret_cast<T*>(smem + (5 + wv) * TILE);
  if (n_steps > 0) {
    uint32_t k_old = k_lds + 2 * TILE, k_now = k_lds, k_next = k_lds + TILE;   // where K of the last, this and the next step lies
    issue_k(0, k_now);
    issue_v(0);
    issue_k(1, k_next);
    const TileFrags<D> f;
    // ANY, head_dim 256: dO of the row tile stays in LDS.  Beside K and V on their way 73 registers were spilled, and dQ took 279 / 128
    // us, window / compressed, in the last example above.
    constexpr bool DO_LDS = ANY && D >= 256;
    vec8 xq[Loads::N], xd[Loads::N], dorow[NKS];
    r.rows_fetch(xq, reinterpret_cast<const T*>(p.q) + (int64_t)(q0 + qi) * p.q_sn + (int64_t)hq_i * p.q_sh);
    r.rows_fetch(xd, reinterpret_cast<const T*>(p.d_o) + (int64_t)(q0 + qi) * p.do_sn + (int64_t)hq_i * p.do_sh);
    const int64_t stat = (int64_t)hq_i * p.n_tokens + q0 + qi;
    // a row without any visible key has lse = -inf: +inf instead turns every probability of it into 0, not NaN
    const float2 pair = p.stat2 ? p.stat2[(int64_t)(q0 + qi) * (p.g * p.hkv) + hq_i] : make_float2(p.lse[stat], p.delta[stat]);
    const float lse = pair.x == -INFINITY ? INFINITY : pair.x, delta = pair.y * p.scale;
    const int jmax = KeyRange<MODE>::hi(p, qi, nc) - jt0, jmin = KeyRange<MODE>::lo(p, qi) - jt0;
    auto mask = [&](f32x16& x, int t) {   // a step that every row of the wave sees completely needs none
      const int limit = jmax - 32 * t, limit_lo = jmin - 32 * t;
      if (!__all(limit >= 31 && limit_lo <= 0)) {
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const int key = 8 * (i >> 2) + 4 * hh + (i & 3);
          if (!(key <= limit && key >= limit_lo)) x[i] = -INFINITY;
        }
      }
    };
    r.rows_to_frags(r.q, xq, rows_lds, f);
    r.rows_to_frags(dorow, xd, rows_lds, f);
    r.settle_q();
    if constexpr (!DO_LDS) {
#pragma unroll
      for (int ks = 0; ks < NKS; ++ks) asm volatile("" : "+v"(dorow[ks]));
    }
    const uint32_t do_lds = lds_addr(rows_lds);
    auto step = [&](f32x16& x, f32x16& next, int t) {   // scores of this step in x, those of the next one into `next`
      tiles_arrived();   // K of the next step, V of this one
      if constexpr (ANY) {
        fetch(t);
      } else {
        issue_k(t + 2, k_old);    // (behind the last key: zeros, and nothing is read)
        issue_v(t + 1);
      }
      const uint32_t v_tile = v_lds + (t & 1) * TILE;
      constexpr int AHEAD = 2;
      vec8 fr[AHEAD + 1], ds[2];
      f32x16 dp;
#pragma unroll
      for (int i = 0; i < 16; ++i) dp[i] = next[i] = 0.f;
      auto read = [&](int i) {
        fr[i % (AHEAD + 1)] = load16<vec8>(lds_ptr<T>((i < NKS ? v_tile : k_next) + (f.k ^ (16u * (i % NKS)))));
        if (DO_LDS && i < NKS) dorow[i % (AHEAD + 1)] = load16<vec8>(lds_ptr<T>(do_lds + (f.k ^ (16u * i))));
      };
#pragma unroll
      for (int i = 0; i < AHEAD; ++i) read(i);
      // dP of this step beside its exponentials, then scores of the next step beside dS = P (dP - delta) scale of this one
      constexpr int LATE = NKS / 4;   // dS starts that many products after the last one of dP
#pragma unroll
      for (int i = 0; i < 2 * NKS; ++i) {
        if (i + AHEAD < 2 * NKS) read(i + AHEAD);
        if (i < NKS) {
          dp = Elem<T>::mfma32(fr[i % (AHEAD + 1)], dorow[DO_LDS ? i % (AHEAD + 1) : i % NKS], dp);
#pragma unroll
          for (int e = i * 16 / NKS; e < (i + 1) * 16 / NKS; ++e) {
            x[e] = fast_exp2(x[e] * p.scale_log2 - lse);
            asm volatile("" : "+v"(x[e]));   // (here, not in front of its use)
          }
        } else {
          next = Elem<T>::mfma32(fr[i % (AHEAD + 1)], r.q[i % NKS], next);
          constexpr int SLOTS = NKS - LATE;
          const int j = i - NKS - LATE;
#pragma unroll
          for (int e = j < 0 ? 0 : j * 16 / SLOTS; e < (j < 0 ? 0 : (j + 1) * 16 / SLOTS); ++e) {
            ds[e >> 3][e & 7] = (T)(x[e] * (dp[e] * p.scale - delta));
            if ((e & 7) == 7) asm volatile("" : "+v"(ds[e >> 3]));
          }
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      // dQ^T += K^T dS
      constexpr int AH = 3;
      vec8 tr[AH + 1];
      auto readt = [&](int i) { tr[i % (AH + 1)] = swizzled_tr_frag<T, D>(k_now + (f.v ^ (64u * (i % NDT))), i / NDT); };
#pragma unroll
      for (int i = 0; i < AH; ++i) readt(i);
#pragma unroll
      for (int i = 0; i < 2 * NDT; ++i) {
        if (i + AH < 2 * NDT) readt(i + AH);
        r.o[i % NDT] = Elem<T>::mfma32(tr[i % (AH + 1)], ds[i / NDT], r.o[i % NDT]);
        __builtin_amdgcn_sched_barrier(0);
      }
      mask(next, t + 1);
      if constexpr (ANY) land(k_old, v_lds + ((t + 1) & 1) * TILE);
      const uint32_t k = k_old;
      k_old = k_now;
      k_now = k_next;
      k_next = k;
    };
    f32x16 sa, sb;
    tiles_arrived();
#pragma unroll
    for (int i = 0; i < 16; ++i) sa[i] = 0.f;
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) sa = Elem<T>::mfma32(load16<vec8>(lds_ptr<T>(k_now + (f.k ^ (16u * ks)))), r.q[ks], sa);
    mask(sa, 0);
    for (int t = 0;;) {
      step(sa, sb, t);
      if (++t >= n_steps) break;
      step(sb, sa, t);
      if (++t >= n_steps) break;
    }
    vm_wait<0>();
  }
  r.store_rows(reinterpret_cast<T*>(p.dq) + ((int64_t)(q0 + qi) * (p.g * p.hkv) + hq_i) * D, valid, 1.f, rows_lds);
}

template <typename T, int D, int MODE, bool ANY>
__global__ void __launch_bounds__(256, (D <= 128 ? 2 : 1))
cmpattn_fwd_kernel(CmpParams p) {
  attn_fwd_tile<T, D, MODE, ANY>(p, blockIdx.x);
}
template <typename T, int D, int MODE, bool ANY>
__global__ void __launch_bounds__(256, (D <= 128 ? 2 : 1))
cmpattn_bwd_dq_kernel(CmpParams p) {
  attn_bwd_dq_tile<T, D, MODE, ANY>(p, blockIdx.x);
}
// Compressed (blockIdx.z == 0, in front) and window attention of one layer in one launch.  At small sizes either alone
// leaves most of the chip idle.
template <typename T, int D, bool ANY>
__global__ void __launch_bounds__(256, (D <= 128 ? 2 : 1))
attn_fwd_pair_kernel(CmpParams a, CmpParams b) {
  if (blockIdx.z == 0) attn_fwd_tile<T, D, CMP_MODE_COMPRESSED, ANY>(a, blockIdx.x);
  else attn_fwd_tile<T, D, CMP_MODE_WINDOW, ANY>(b, blockIdx.x);
}
template <typename T, int D>
__global__ void __launch_bounds__(256)
cmp_delta_kernel(const T* __restrict__ o, int64_t o_sn, int64_t o_sh, const T* __restrict__ d_o,
                 int64_t do_sn, int64_t do_sh, int64_t n_tokens, int hq, float* __restrict__ delta) {
  typedef typename Elem<T>::vec8 vec8;
  constexpr int LPR = D / 8, RPB = 256 / LPR;
  const int64_t R = (int64_t)blockIdx.x * RPB + threadIdx.x / LPR;
  const int sub = threadIdx.x % LPR;
  if (R >= n_tokens * hq) return;
  const int64_t tok = R / hq;
  const int h = (int)(R - tok * hq);
  vec8 a = load16<vec8>(o + tok * o_sn + (int64_t)h * o_sh + sub * 8);
  vec8 b = load16<vec8>(d_o + tok * do_sn + (int64_t)h * do_sh + sub * 8);
  float s = 0.f;
#pragma unroll
  for (int e = 0; e < 8; ++e) s += (float)a[e] * (float)b[e];
#pragma unroll
  for (int o_ = LPR / 2; o_ >= 1; o_ >>= 1) s += __shfl_xor(s, o_, LPR);
  if (sub == 0) delta[(int64_t)h * n_tokens + tok] = s;
}

// Work list of the key-major dK/dV kernel, one work-group per kv head: a "block" is a tile of 64 keys.  Compressed mode:
// its rows are the queries from the first one that sees its first key to the end of the sequence; window mode: the
// queries from the tile's first key to `window` tokens past its last key.  Writes the counts, cu_tiles (tiles of the
// sequences before s) and the tile prefix in one launch.
constexpr int KT_THREADS = 256;
struct KvTiles {
  const int32_t *cu_q, *cu_k;
  int64_t max_blocks;
  int kernel_size, kernel_stride, window, tile_rows;
  int32_t *cu_tiles, *counts, *tile_prefix;
};
template <int MODE> __device__ __forceinline__ void kv_tiles(const KvTiles& p, int batch, int g, int h) {
  const int32_t *__restrict__ cu_q = p.cu_q, *__restrict__ cu_k = p.cu_k;
  const int64_t max_blocks = p.max_blocks;
  const int kernel_size = p.kernel_size, kernel_stride = p.kernel_stride, window = p.window, tile_rows = p.tile_rows;
  int32_t *cu_tiles = p.cu_tiles, *counts = p.counts, *tile_prefix = p.tile_prefix;
  __shared__ int wave_total[KT_THREADS / WAVE];
  const int tid = threadIdx.x, lane = tid & (WAVE - 1), w = tid / WAVE;
  // exclusive scan over the work-group, and the total
  auto scan = [&](int v, int& total) {
    int inc = v;
#pragma unroll
    for (int o = 1; o < WAVE; o <<= 1) {
      const int x = __shfl_up(inc, o, WAVE);
      if (lane >= o) inc += x;
    }
    if (lane == WAVE - 1) wave_total[w] = inc;
    __syncthreads();
    total = 0;
    for (int ww = 0; ww < KT_THREADS / WAVE; ++ww) {
      if (ww == w) inc += total;
      total += wave_total[ww];
    }
    __syncthreads();
    return inc - v;
  };
  const int32_t* cu = MODE == CMP_MODE_WINDOW ? cu_q : cu_k;
  int n_blocks = 0;   // every head writes the same cu_tiles; each work-group reads back only what it wrote itself
  for (int s0 = 0; s0 < batch; s0 += KT_THREADS) {
    const int s = s0 + tid;
    const int nb = s < batch ? (cu[s + 1] - cu[s] + CMP_BK - 1) / CMP_BK : 0;
    int total;
    const int at = n_blocks + scan(nb, total);
    if (s < batch) cu_tiles[s] = at;
    n_blocks += total;
  }
  if (tid == 0) cu_tiles[batch] = n_blocks;
  __syncthreads();
  int run = 0;
  for (int64_t b0 = 0; b0 < max_blocks; b0 += KT_THREADS) {
    const int64_t gb = b0 + tid;
    int c = 0;
    if (gb < n_blocks) {
      const int s = upper_seg(cu_tiles, batch, (int)gb);
      const int len = cu_q[s + 1] - cu_q[s], first = (int)(gb - cu_tiles[s]) * CMP_BK;
      c = MODE == CMP_MODE_WINDOW ? max(0, min(len, first + CMP_BK + window) - first)
                                  : max(0, len - (first * kernel_stride + kernel_size - 1));
    }
    int total;
    const int at = run + scan((int)(((int64_t)c * g + tile_rows - 1) / tile_rows), total);
    if (gb < max_blocks) {
      counts[h * max_blocks + gb] = c;
      tile_prefix[h * (max_blocks + 1) + gb] = at;
    }
    run += total;
  }
  if (tid == 0) tile_prefix[h * (max_blocks + 1) + max_blocks] = run;
}
template <int MODE>
__global__ void __launch_bounds__(KT_THREADS)
kv_tiles_kernel(KvTiles p, int batch, int g) {
  kv_tiles<MODE>(p, batch, g, blockIdx.x);
}

// dQ of a pair; the first 2 hkv work-groups write the two work lists that the dK/dV launch behind it needs (their places in
// the other rows of the grid stay empty).
template <typename T, int D, bool ANY>
__global__ void __launch_bounds__(256, (D <= 128 ? 2 : 1))
attn_bwd_dq_pair_kernel(CmpParams a, CmpParams b, KvTiles ta, KvTiles tb, int batch) {
  const int hkv = a.hkv, id = (int)blockIdx.x - 2 * hkv;
  if (id < 0) {
    if (blockIdx.y != 0 || blockIdx.z != 0) return;
    if (id < -hkv) kv_tiles<CMP_MODE_COMPRESSED>(ta, batch, a.g, id + 2 * hkv);
    else kv_tiles<CMP_MODE_WINDOW>(tb, batch, a.g, id + hkv);
  } else if (blockIdx.z == 0) {
    attn_bwd_dq_tile<T, D, CMP_MODE_COMPRESSED, ANY>(a, id);
  } else {
    attn_bwd_dq_tile<T, D, CMP_MODE_WINDOW, ANY>(b, id);
  }
}

// ------------------------------------------------------------------ score ----
// score[h, token, j] = 2^(c q[token, h*g] . ck[j, h] - lse[h*g, token]) for visible j
// REBIN (compression window of 2 strides, selection block of 4): the block scores - taps 4 b - 1 .. 4 b + 3 with
// weights 1 2 2 2 1 - are formed in registers and written instead of the per-key probabilities, a quarter of the
// bytes.  A lane holds groups of four consecutive keys, i.e. the last four taps of a block; the first tap is the
// last key of the group before, which the other half of the wave holds (one exchange per group, and one value
// carried over from the previous key tile).
template <typename T, int D, bool REBIN>
__global__ void __launch_bounds__(256)
cmp_score_kernel(CmpParams p) {
  typedef typename Elem<T>::vec8 vec8;
  constexpr int KS = CmpLds<D>::KS;
  constexpr int NA = CMP_BK / 32, NKS = D / 16;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  T* Ks = reinterpret_cast<T*>(smem);

  int bx, s, h;
  tile_of(p, blockIdx.x, bx, s, h);
  const int q0 = p.cu_q[s], lq = p.cu_q[s + 1] - q0;
  const int k0 = p.cu_k[s], nc = p.cu_k[s + 1] - k0;
  const int row_lo = bx * CMP_ROWS;
  if (row_lo >= lq) return;
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int col = lane & 31, hh = lane >> 5;
  const int r = row_lo + wv * 32 + col;
  const bool valid = r < lq;
  const int qi = valid ? r : lq - 1;
  const int hq_i = h * p.score_head_step;  // first head of the group (as written: q head = kv head)
  const T* qrow = reinterpret_cast<const T*>(p.q) + (int64_t)(q0 + qi) * p.q_sn + (int64_t)hq_i * p.q_sh + hh * (D / 2);
  vec8 qreg[NKS];
#pragma unroll
  for (int ks = 0; ks < NKS; ++ks) qreg[ks] = load16<vec8>(qrow + ks * 8);
  const float lse_r = p.lse[(int64_t)hq_i * p.n_tokens + q0 + qi];
  int jmax = qi >= p.kernel_size - 1 ? (qi - p.kernel_size + 1) / p.kernel_stride : -1;
  jmax = min(jmax, nc - 1);
  const int qi_last = min(lq, row_lo + CMP_ROWS) - 1;
  const int n_keys = qi_last >= p.kernel_size - 1 ? min(nc, (qi_last - p.kernel_size + 1) / p.kernel_stride + 1) : 0;
  const T* kbase = reinterpret_cast<const T*>(p.k) + (int64_t)h * p.k_sh;
  float* srow = p.score + ((int64_t)h * p.n_tokens + q0 + qi) * p.score_ld;
  const uint32_t k_off = k_tile_offset<T, D>(p.k_sn, tid);

  // REBIN: one more tile when the visible keys end on a tile boundary - the block that starts there still owns the
  // last key before it
  const int n_keys_loop = REBIN && n_keys > 0 ? n_keys + 1 : n_keys;
  float carry = 0.f;  // REBIN, lower half of the wave: probability of the key just before this tile
  for (int jt = 0; jt < n_keys_loop; jt += CMP_BK) {
    if (jt) __syncthreads();
    stage_k_tile<T, D>(kbase, p.k_sn, k_off, k0 + jt, nc - jt, Ks, tid);
    __syncthreads();
    f32x16 acc[NA];
#pragma unroll
    for (int a = 0; a < NA; ++a) {
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[a][i] = 0.f;
#pragma unroll
      for (int ks = 0; ks < NKS; ++ks) {
        vec8 kf = load16<vec8>(&Ks[(a * 32 + col) * KS + hh * (D / 2) + ks * 8]);
        acc[a] = Elem<T>::mfma32(kf, qreg[ks], acc[a]);
      }
    }
    const int limit = jmax - jt;
    if constexpr (REBIN) {
      static_assert(NA == 2, "two 32-key halves per tile");
      float x[NA][16], last[NA * 4], recv[NA * 4];
#pragma unroll
      for (int a = 0; a < NA; ++a)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const int key = a * 32 + 8 * (i >> 2) + 4 * hh + (i & 3);
          x[a][i] = key <= limit ? fast_exp2(acc[a][i] * p.scale_log2 - lse_r) : 0.f;
        }
#pragma unroll
      for (int f = 0; f < NA * 4; ++f) {
        last[f] = x[f >> 2][4 * (f & 3) + 3];
        recv[f] = __shfl_xor(last[f], 32, 64);
      }
#pragma unroll
      for (int f = 0; f < NA * 4; ++f) {
        // the key before this group: the other half's group f (upper half) or f - 1 (lower half)
        const float before = hh ? recv[f] : (f ? recv[f > 0 ? f - 1 : 0] : carry);
        const int a = f >> 2, qd = f & 3;
        float bsum = before;
        bsum += 2.f * x[a][4 * qd];
        bsum += 2.f * x[a][4 * qd + 1];
        bsum += 2.f * x[a][4 * qd + 2];
        bsum += x[a][4 * qd + 3];
        const int blk = jt / 4 + a * 8 + 2 * qd + hh;
        if (valid && blk < p.score_ld) srow[blk] = bsum;
      }
      carry = recv[NA * 4 - 1];
    } else if (valid) {
#pragma unroll
      for (int a = 0; a < NA; ++a)
#pragma unroll
        for (int qd = 0; qd < 4; ++qd) {
          const int key0 = a * 32 + 8 * qd + 4 * hh;
          if (jt + key0 < p.score_ld) {
            f32x4 x;
#pragma unroll
            for (int e = 0; e < 4; ++e)
              x[e] = key0 + e <= limit ? fast_exp2(acc[a][4 * qd + e] * p.scale_log2 - lse_r) : 0.f;
            *reinterpret_cast<f32x4*>(srow + jt + key0) = x;
          }
        }
    }
  }
}

// ------------------------------------------------------- transform + top-k ----
struct TopkParams {
  const float* score;   // [Hkv, N, score_ld]; only the visible prefix of each row is defined
  int64_t score_ld;
  const int32_t* cu_q;
  const int32_t* cu_k;
  int batch;
  int64_t n_tokens;
  int hkv;
  int kernel_size, kernel_stride, block_size;
  int na, ne;           // kernel_size / kernel_stride, block_size / kernel_stride
  int rebin;            // `score` already holds the block scores before forcing and rounding
  int nblk;             // columns of the block-score matrix: ceil(max_seqlen_q / block_size)
  int t_out;            // min(topk, nblk)
  int init_blocks, local_blocks;
  int to_bf16;
  int32_t* topk_idx;    // [Hkv, N, t_out]
  float* block_score;   // optional [Hkv, N, nblk] fp32 (after the optional bf16 rounding)
};

__device__ __forceinline__ float round_bf16(float x) { return (float)(__bf16)x; }

// One wave per (kv head, query).  NREG > 0 (scores rounded to bf16, at most 64 * NREG blocks): the scores live in
// registers as 16-bit keys, and the t_out-th largest of them is found bit by bit: a step is NREG compares and ballots,
// the counting is scalar work.  The chosen ids come out in ascending order by themselves (position = number of chosen
// lanes in front).  Bound by vector issue; against t_out rounds of a maximum over the wave and a rank sort: 8 heads, 32K
// tokens and up to 225 blocks 230 -> 176 us, 5K tokens 31 -> 22 us.  NREG == 0: fp32 scores in LDS, (value, id) compared
// explicitly.
// BIG (more than 64 selected blocks per query, or more blocks than four waves can keep in LDS): one wave per
// work-group, the chosen ids are collected in LDS behind the scores and ranked from there.
template <int NREG, bool BIG = false>
__global__ void __launch_bounds__(BIG ? 64 : 256)
cmp_topk_kernel(TopkParams p) {
  constexpr int WPB = BIG ? 1 : 4;   // waves (= queries) per work-group
  extern __shared__ float bs_all[];  // [WPB waves][nblk] (+ [t_out] ids when BIG), NREG == 0 only
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int h = blockIdx.y;
  const int tok = blockIdx.x * WPB + wv;  // the same for every lane of the wave
  if (tok >= p.n_tokens) return;
  float* bs = bs_all + wv * p.nblk;
  int* sel = reinterpret_cast<int*>(bs_all + p.nblk);  // BIG only
  const int s = upper_seg(p.cu_q, p.batch, tok);
  const int qi = tok - p.cu_q[s];
  const int nc = p.cu_k[s + 1] - p.cu_k[s];
  const int n_vis = qi >= p.kernel_size - 1 ? min(nc, (qi - p.kernel_size + 1) / p.kernel_stride + 1) : 0;
  const int na = p.na, ne = p.ne;
  const int n_off = na + ne - 1, pad = na - 1;
  const int bq = qi / p.block_size;
  const float* srow = p.score + ((int64_t)h * p.n_tokens + tok) * p.score_ld;
  // the usual geometry (compression window of 2 strides, selection block of 4): taps 4 b - 1 .. 4 b + 3 with
  // weights 1 2 2 2 1, four of them one aligned 16-byte load (score rows start 16-byte aligned)
  const bool taps_12221 = na == 2 && ne == 4;
  auto block_score = [&](int b) {
    float acc = 0.f;
    const int c0 = b * ne - pad;
    if (p.rebin) {
      acc = max(4 * b - 1, 0) < n_vis ? srow[b] : 0.f;  // blocks without a visible tap were not written
    } else if (taps_12221) {
      const int c = 4 * b;
      f32x4 x = {0.f, 0.f, 0.f, 0.f};
      if (c + 3 < n_vis) {
        x = *reinterpret_cast<const f32x4*>(srow + c);
      } else {
#pragma unroll
        for (int e = 0; e < 3; ++e)
          if (c + e < n_vis) x[e] = srow[c + e];
      }
      const float xm = (c >= 1 && c - 1 < n_vis) ? srow[c - 1] : 0.f;
      acc = xm;
      acc += 2.f * x[0];
      acc += 2.f * x[1];
      acc += 2.f * x[2];
      acc += x[3];
    } else
    for (int o = 0; o < n_off; ++o) {
      const int c = c0 + o;
      if (c >= 0 && c < n_vis) {
        const int wgt = min(min(o, n_off - 1 - o), min(na, ne) - 1) + 1;
        acc += (float)wgt * srow[c];
      }
    }
    if (b < p.init_blocks || (bq >= b && bq < b + p.local_blocks)) acc = INFINITY;
    if (p.to_bf16) acc = round_bf16(acc);
    if (p.block_score) p.block_score[((int64_t)h * p.n_tokens + tok) * p.nblk + b] = acc;
    return acc;
  };
  int my_id = -1;  // lane t keeps the id chosen in round t
  if constexpr (NREG > 0) {
    int32_t* out = p.topk_idx + ((int64_t)h * p.n_tokens + tok) * p.t_out;
    const int n_cand = min(bq + 1, p.nblk);   // later blocks score zero and would be masked: they only fill up the list
    if (n_cand <= p.t_out) {                  // every block is taken (uniform)
      if (p.block_score)
        for (int b = lane; b < p.nblk; b += 64) block_score(b);
      if (lane < p.t_out) out[lane] = lane < n_cand ? lane : -1;
      return;
    }
    // bf16 bits + 1; 0: no candidate.  A NaN is a large score; the largest of them is cut to the 15 bits that the search
    // below runs over, a key above every threshold would be taken however many there are.
    uint32_t key[NREG];
#pragma unroll
    for (int r = 0; r < NREG; ++r) {
      const int b = lane + 64 * r;
      const float sc = (b < p.nblk && (b < n_cand || p.block_score)) ? block_score(b) : 0.f;
      key[r] = b < n_cand ? min(__float_as_uint(sc) >> 16 & 0x7FFFu, 0x7FFEu) + 1u : 0u;
    }
    // largest threshold that at least t_out keys reach, bit by bit; counts come from ballots, in scalar registers
    auto count_from = [&](uint32_t t) {
      int c = 0;
#pragma unroll
      for (int r = 0; r < NREG; ++r) c += (int)__popcll(__ballot(key[r] >= t));
      return c;
    };
    uint32_t thr = 0;
    int at_thr = n_cand;
#pragma unroll 1
    for (int bit = 14; bit >= 0 && at_thr != p.t_out; --bit) {
      const uint32_t t = thr | (1u << bit);
      const int c = count_from(t);
      if (c >= p.t_out) {
        thr = t;
        at_thr = c;
      }
    }
    // of the keys equal to the threshold the lowest ids are taken
    int need = p.t_out - (at_thr == p.t_out ? 0 : count_from(thr + 1));
    int base = 0;
#pragma unroll
    for (int r = 0; r < NREG; ++r) {
      bool take = key[r] >= thr;
      if (at_thr != p.t_out) {
        const uint64_t eq = __ballot(key[r] == thr);
        const int rank = __builtin_amdgcn_mbcnt_hi((uint32_t)(eq >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)eq, 0));
        take = key[r] > thr || (key[r] == thr && rank < need);
        need = max(0, need - (int)__popcll(eq));
      }
      const uint64_t m = __ballot(take);
      if (take) out[base + __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0))] = lane + 64 * r;
      base += (int)__popcll(m);
    }
    return;
  } else {
    for (int b = lane; b < p.nblk; b += 64) bs[b] = block_score(b);
    __builtin_amdgcn_wave_barrier();
    // t_out rounds of arg-max by (value desc, id asc).  Scores are >= 0 or NaN, which is a large score, as in the other
    // form; taken entries are marked -1.  As 64-bit keys, score bits + 1 above (0: taken) and the complement of the id
    // below, the larger key is the larger score or, on equal scores, the lower id; t_out <= nblk entries are never all taken.
    for (int t = 0; t < p.t_out; ++t) {
      uint64_t best = 0;
      for (int b = lane; b < p.nblk; b += 64) {
        const uint32_t bits = __float_as_uint(bs[b]);
        const uint64_t k = bits == 0xBF800000u ? 0ull : ((uint64_t)((bits & 0x7FFFFFFFu) + 1u) << 32) | (0xFFFFFFFFu - (uint32_t)b);
        best = k > best ? k : best;
      }
      const uint64_t top = wave_max_u64(best);
      const int best_id = (int)(0xFFFFFFFFu - (uint32_t)top);
      if (!BIG && lane == t) my_id = best_id;
      if (lane == 0) {
        bs[best_id] = -1.f;
        if (BIG) sel[t] = best_id;
      }
      __builtin_amdgcn_wave_barrier();
    }
  }
  if (BIG) {  // ascending order by rank counting over the list in LDS, then the mask
    for (int i = lane; i < p.t_out; i += 64) {
      const int id = sel[i];
      int rank = 0;
      for (int j = 0; j < p.t_out; ++j) rank += sel[j] < id;
      p.topk_idx[((int64_t)h * p.n_tokens + tok) * p.t_out + rank] = id > bq ? -1 : id;
    }
    return;
  }
  // ascending order by rank counting (ids are distinct), then mask ids above the own block
  const int t_eff = min(p.t_out, 64);
  int rank = 0;
  for (int t = 0; t < t_eff; ++t) {
    const int other = __builtin_amdgcn_readlane(my_id, t);  // uniform lane index: no trip through the LDS crossbar
    if (other < my_id) ++rank;
  }
  if (lane < t_eff)
    p.topk_idx[((int64_t)h * p.n_tokens + tok) * p.t_out + rank] = my_id > bq ? -1 : my_id;
}

// -------------------------------------------------------------- host side ----
// Grid of 256 threads per tile: one dimension, but not beyond the 2^32 work-items that it may have (600 sequences x 8 kv
// heads of which one sequence has 131072 tokens x 4 heads).  `lists`: work-groups in front of each row.
static dim3 dense_grid(int nx, int hkv, int batch, int lists = 0) {
  const int64_t all = (int64_t)nx * hkv * batch + lists;
  if (all * 256 < ((int64_t)1 << 32)) return dim3((unsigned)all);
  return dim3((unsigned)(nx * hkv + lists), (unsigned)batch);
}
static dim3 dense_pair_grid(int nx, int hkv, int batch, int lists = 0) {   // both branches of a layer: blockIdx.z
  dim3 g = dense_grid(nx, hkv, batch, lists);
  g.z = 2;
  return g;
}

// Rows per work-group of the dK/dV kernel.  A work-group alone on a CU takes 1.3 us for a pass of 64 rows of 128 dims, two there
// 2.5, so one for every CU is as good as two, and every share of a key tile costs 64 KB of partial sums, written and read.  Kernel
// and reduction of both branches, us, two per slot (as for gathered rows) | 384 work-groups a branch | 256: 2000 tokens x 8 heads of
// 128, window 128, 30.1 | 29.7 | 29.1, 3000 x 16, window 512, 71.9 | 64.4 | 72.6, 4000 x 8 79 | 64 | 70, 5003 x 32 210 | 174 | 173,
// 12000 x 32 421 | 400 | 398; 6000 x 32 heads of 64 162 | 140 | 122, 20000 x 32 244 | 220 | 221.  `straight` false: the kernel for gathered
// rows runs, and with these shares it would be slower (rows that are not aligned, 16384 x 32 of 128, window | compressed, 545 | 649
// against 496 | 528, 16384 x 16 of 64 compressed 235 against 146).
static int dense_tile_rows(int64_t rows_total, int g, int d, bool straight) {
  if (!straight) return kv_tile_rows(rows_total, g, d, CMP_BK);
  const int64_t r = rows_total / (d > 64 ? 384 : 256) / 64 * 64;
  return (int)std::max<int64_t>(kv_tile_rows(rows_total, g, d, CMP_BK), std::min<int64_t>(r, KV_TILE_ROWS_MAX));
}
// rows of all (key tile, query head) pairs: a key tile of a sequence is seen by about half of its queries
static int64_t cmp_rows_total(int64_t max_blocks, int64_t max_q, int hq) { return max_blocks * max_q * hq / 2; }
static int64_t win_rows_total(int64_t max_blocks, int window, int hq) { return max_blocks * (CMP_BK + window) * hq; }

struct CmpBwdWs {
  size_t off_delta, off_cu_tiles, off_counts, off_tiles, off_part, total;
  int64_t max_blocks, max_tiles;
  int tile_rows;
};

// The work list and the partial sums of key tiles that at most `rows` rows see each.  The room for the sums is that of the shares
// that gathered rows would have, as callers know it: shares for one work-group per CU are never shorter.
static void dense_tiles(CmpBwdWs& w, int64_t rows, int64_t rows_total, int g, int hkv, int d, bool straight) {
  const int64_t gathered = kv_tile_rows(rows_total, g, d, CMP_BK);
  w.tile_rows = dense_tile_rows(rows_total, g, d, straight);
  w.max_tiles = w.max_blocks * ((rows + w.tile_rows - 1) / w.tile_rows);   // as kv_tiles deals them
  w.total = w.off_part + align_up((size_t)hkv * w.max_blocks * ((rows + gathered - 1) / gathered) * 2 * CMP_BK * d * 4, 256);
}
static CmpBwdWs cmp_bwd_ws(int64_t n, int64_t n_k, int64_t max_q, int batch, int hq, int hkv, int d, bool straight) {
  CmpBwdWs w;
  const int g = hq / hkv;
  w.max_blocks = (n_k + CMP_BK - 1) / CMP_BK + batch;
  w.off_delta = 0;
  w.off_cu_tiles = align_up((size_t)n * hq * 4, 256);
  w.off_counts = w.off_cu_tiles + align_up((size_t)(batch + 1) * 4, 256);
  w.off_tiles = w.off_counts + align_up((size_t)hkv * w.max_blocks * 4, 256);
  w.off_part = w.off_tiles + align_up((size_t)hkv * (w.max_blocks + 1) * 4, 256);
  // a key tile is seen by at most max_q queries of its sequence; rows = queries * g
  dense_tiles(w, max_q * g, cmp_rows_total(w.max_blocks, max_q, hq), g, hkv, d, straight);
  return w;
}

// Whether keys and values can go to LDS past the registers: rows 16-byte aligned, and none on top of another.
static bool rows_go_straight(const CmpParams& p, int d) {
  auto ok = [&](const void* x, int64_t sn, int64_t sh) { return ((uintptr_t)x % 16 | (sn | sh) % 8) == 0 && sn >= d; };
  return ok(p.k, p.k_sn, p.k_sh) && ok(p.v, p.v_sn, p.v_sh);
}

template <typename T, int D, int MODE, bool ANY>
static int attn_fwd_launch_as(CmpParams p, int batch, int hkv, int64_t max_rows, hipStream_t stream) {
  static LdsAllowed lds;
  if (int rc_ = allow_lds(lds, (const void*)cmpattn_fwd_kernel<T, D, MODE, ANY>, CmpFwdLds<T, D>::BYTES)) return rc_;
  p.hkv = hkv;
  p.nx = (int)((max_rows + CMP_ROWS - 1) / CMP_ROWS);
  const dim3 grid = dense_grid(p.nx, hkv, batch);
  ProfScope ps_(MODE == CMP_MODE_WINDOW ? "winattn_fwd" : "cmpattn_fwd", stream);
  cmpattn_fwd_kernel<T, D, MODE, ANY><<<grid, 256, CmpFwdLds<T, D>::BYTES, stream>>>(p);
  return 0;
}
template <typename T, int D, int MODE>
static int attn_fwd_launch(const CmpParams& p, int batch, int hkv, int64_t max_rows, hipStream_t stream) {
  return rows_go_straight(p, D) ? attn_fwd_launch_as<T, D, MODE, false>(p, batch, hkv, max_rows, stream)
                                : attn_fwd_launch_as<T, D, MODE, true>(p, batch, hkv, max_rows, stream);
}
template <typename T, int D>
static int cmp_fwd_launch(const CmpParams& p, int batch, int hkv, int64_t max_rows, hipStream_t stream) {
  return attn_fwd_launch<T, D, CMP_MODE_COMPRESSED>(p, batch, hkv, max_rows, stream);
}
template <typename T, int D>
static int win_fwd_launch(const CmpParams& p, int batch, int hkv, int64_t max_rows, hipStream_t stream) {
  return attn_fwd_launch<T, D, CMP_MODE_WINDOW>(p, batch, hkv, max_rows, stream);
}

template <typename T, int D, int MODE, bool ANY>
static int attn_dq_launch_as(const CmpParams& p, int batch, hipStream_t stream) {
  static LdsAllowed lds;
  if (int rc_ = allow_lds(lds, (const void*)cmpattn_bwd_dq_kernel<T, D, MODE, ANY>, CmpDqLds<T, D>::BYTES)) return rc_;
  ProfScope ps_(MODE == CMP_MODE_WINDOW ? "winattn_bwd_dq" : "cmpattn_bwd_dq", stream);
  cmpattn_bwd_dq_kernel<T, D, MODE, ANY><<<dense_grid(p.nx, p.hkv, batch), 256, CmpDqLds<T, D>::BYTES, stream>>>(p);
  return 0;
}
template <typename T, int D, int MODE>
static int attn_bwd_launch(CmpParams p, const SelBwdParams& kv, int batch, int hq, int hkv,
                           int64_t max_rows, int64_t n, bool straight, hipStream_t stream) {
  constexpr int KVM = MODE == CMP_MODE_WINDOW ? KV_MODE_WINDOW : KV_MODE_COMPRESSED;
  static LdsAllowed lds2;
  if (int rc_ = allow_lds(lds2, (const void*)attn_bwd_dkdv_kernel<T, D, CMP_BK, KVM>, KvCfg<D, CMP_BK>::BYTES)) return rc_;
  static LdsAllowed lds3;
  if constexpr (D <= 128)
    if (int rc_ = allow_lds(lds3, (const void*)dense_dkdv_kernel<T, D, KVM>, DenseKv<D>::BYTES)) return rc_;
  p.hkv = hkv;
  p.nx = (int)((max_rows + CMP_ROWS - 1) / CMP_ROWS);
  {
    ProfScope ps_(MODE == CMP_MODE_WINDOW ? "winattn_bwd_delta" : "cmpattn_bwd_delta", stream);
    constexpr int RPB = 256 / (D / 8);
    cmp_delta_kernel<T, D><<<(unsigned)((n * hq + RPB - 1) / RPB), 256, 0, stream>>>(
        (const T*)p.o, p.o_sn, p.o_sh, (const T*)p.d_o, p.do_sn, p.do_sh, n, hq, (float*)p.delta);
  }
  if (int rc_ = rows_go_straight(p, D) ? attn_dq_launch_as<T, D, MODE, false>(p, batch, stream)
                                       : attn_dq_launch_as<T, D, MODE, true>(p, batch, stream))
    return rc_;
  {
    const HeadOrder order = head_order(hkv, n * kv.g * D * 2);
    ProfScope ps_(MODE == CMP_MODE_WINDOW ? "winattn_bwd_dkdv" : "cmpattn_bwd_dkdv", stream);
    bool done = false;
    if constexpr (D <= 128)
      if ((done = straight))
        dense_dkdv_kernel<T, D, KVM><<<head_tile_grid(kv.max_tiles, order), DenseKv<D>::NT, DenseKv<D>::BYTES, stream>>>(kv, order);
    if (!done)
      attn_bwd_dkdv_kernel<T, D, CMP_BK, KVM>
          <<<head_tile_grid(kv.max_tiles, order), KvCfg<D, CMP_BK>::NT, KvCfg<D, CMP_BK>::BYTES, stream>>>(kv, order);
  }
  {
    ProfScope ps_(MODE == CMP_MODE_WINDOW ? "winattn_bwd_dkdv_reduce" : "cmpattn_bwd_dkdv_reduce", stream);
    const unsigned spans = (unsigned)((kv.max_blocks + KV_REDUCE_SPAN - 1) / KV_REDUCE_SPAN);
    attn_bwd_dkdv_reduce_kernel<T, D, CMP_BK, KVM>
        <<<dim3(spans, hkv, kv_reduce_split((int64_t)spans * hkv)), 256, 0, stream>>>(kv);
  }
  return 0;
}

template <typename T, int D, bool ANY>
static int pair_fwd_launch_as(CmpParams a, CmpParams b, int batch, int hkv, int64_t max_rows, hipStream_t stream) {
  static LdsAllowed lds;
  if (int rc_ = allow_lds(lds, (const void*)attn_fwd_pair_kernel<T, D, ANY>, CmpFwdLds<T, D>::BYTES)) return rc_;
  a.hkv = b.hkv = hkv;
  a.nx = b.nx = (int)((max_rows + CMP_ROWS - 1) / CMP_ROWS);
  ProfScope ps_("attn_fwd_pair", stream);
  attn_fwd_pair_kernel<T, D, ANY><<<dense_pair_grid(a.nx, hkv, batch), 256, CmpFwdLds<T, D>::BYTES, stream>>>(a, b);
  return 0;
}
template <typename T, int D>
static int pair_fwd_launch(const CmpParams& a, const CmpParams& b, int batch, int hkv, int64_t max_rows, hipStream_t stream) {
  return rows_go_straight(a, D) && rows_go_straight(b, D) ? pair_fwd_launch_as<T, D, false>(a, b, batch, hkv, max_rows, stream)
                                                          : pair_fwd_launch_as<T, D, true>(a, b, batch, hkv, max_rows, stream);
}
template <typename T, int D, bool ANY>
static int pair_dq_launch_as(const CmpParams& a, const CmpParams& b, const KvTiles& ta, const KvTiles& tb, int batch, hipStream_t stream) {
  static LdsAllowed lds;
  if (int rc_ = allow_lds(lds, (const void*)attn_bwd_dq_pair_kernel<T, D, ANY>, CmpDqLds<T, D>::BYTES)) return rc_;
  ProfScope ps_("attn_bwd_dq_pair", stream);
  attn_bwd_dq_pair_kernel<T, D, ANY><<<dense_pair_grid(a.nx, a.hkv, batch, 2 * a.hkv), 256, CmpDqLds<T, D>::BYTES, stream>>>(a, b, ta, tb, batch);
  return 0;
}
template <typename T, int D>
static int pair_bwd_launch(CmpParams a, CmpParams b, const SelBwdParams& ka, const SelBwdParams& kb, const KvTiles& ta,
                           const KvTiles& tb, int batch, int hkv, int64_t max_rows, bool straight, hipStream_t stream) {
  typedef KvCfg<D, CMP_BK> C;
  static LdsAllowed lds2;
  if (int rc_ = allow_lds(lds2, (const void*)attn_bwd_dkdv_pair_kernel<T, D, CMP_BK>, C::BYTES)) return rc_;
  static LdsAllowed lds3;
  if constexpr (D <= 128)
    if (int rc_ = allow_lds(lds3, (const void*)dense_dkdv_pair_kernel<T, D>, DenseKv<D>::BYTES)) return rc_;
  a.hkv = b.hkv = hkv;
  a.nx = b.nx = (int)((max_rows + CMP_ROWS - 1) / CMP_ROWS);
  if (int rc_ = rows_go_straight(a, D) && rows_go_straight(b, D) ? pair_dq_launch_as<T, D, false>(a, b, ta, tb, batch, stream)
                                                                 : pair_dq_launch_as<T, D, true>(a, b, ta, tb, batch, stream))
    return rc_;
  {
    const HeadOrder order = head_order(hkv, ka.n_tokens * ka.g * D * 2);
    ProfScope ps_("attn_bwd_dkdv_pair", stream);
    const dim3 grid = head_tile_grid(ka.max_tiles + kb.max_tiles, order);
    bool done = false;
    if constexpr (D <= 128)
      if ((done = straight))
        dense_dkdv_pair_kernel<T, D><<<grid, DenseKv<D>::NT, DenseKv<D>::BYTES, stream>>>(ka, kb, (int)ka.max_tiles, order);
    if (!done) attn_bwd_dkdv_pair_kernel<T, D, CMP_BK><<<grid, C::NT, C::BYTES, stream>>>(ka, kb, (int)ka.max_tiles, order);
  }
  {
    ProfScope ps_("attn_bwd_dkdv_pair_reduce", stream);
    const int sa = (int)((ka.max_blocks + KV_REDUCE_SPAN - 1) / KV_REDUCE_SPAN), sb = (int)((kb.max_blocks + KV_REDUCE_SPAN - 1) / KV_REDUCE_SPAN);
    const int za = kv_reduce_split((int64_t)sa * hkv), zb = kv_reduce_split((int64_t)sb * hkv);
    attn_bwd_dkdv_pair_reduce_kernel<T, D, CMP_BK><<<dim3(sa + sb, hkv, std::max(za, zb)), 256, 0, stream>>>(ka, kb, sa, za, zb);
  }
  return 0;
}

template <typename T, int D>
static int cmp_bwd_launch(const CmpParams& p, const SelBwdParams& kv, int batch, int hq, int hkv,
                          int64_t max_rows, int64_t n, bool straight, hipStream_t stream) {
  return attn_bwd_launch<T, D, CMP_MODE_COMPRESSED>(p, kv, batch, hq, hkv, max_rows, n, straight, stream);
}
template <typename T, int D>
static int win_bwd_launch(const CmpParams& p, const SelBwdParams& kv, int batch, int hq, int hkv,
                          int64_t max_rows, int64_t n, bool straight, hipStream_t stream) {
  return attn_bwd_launch<T, D, CMP_MODE_WINDOW>(p, kv, batch, hq, hkv, max_rows, n, straight, stream);
}

template <typename T, int D>
static int cmp_score_launch(CmpParams p, int batch, int hkv, int64_t max_q, hipStream_t stream) {
  ProfScope ps_("cmp_score", stream);
  p.hkv = hkv;
  p.nx = (int)((max_q + CMP_ROWS - 1) / CMP_ROWS);
  const dim3 grid = dense_grid(p.nx, hkv, batch);
  if (p.rebin) cmp_score_kernel<T, D, true><<<grid, 256, CmpLds<D>::BYTES, stream>>>(p);
  else cmp_score_kernel<T, D, false><<<grid, 256, CmpLds<D>::BYTES, stream>>>(p);
  return 0;
}

// the lane offsets inside a K / V tile are 32-bit: CMP_BK rows have to span less than 4 GiB
static int cmp_check_strides(int64_t k_sn, int64_t v_sn) {
  const int64_t lim = ((int64_t)1 << 32) / (CMP_BK * 2);
  FSA_CHECK_ARG(k_sn >= 0 && k_sn < lim && v_sn >= 0 && v_sn < lim,
                "compressed / window attention: key or value row stride too large");
  return 0;
}
static int cmp_check_strides(const CmpParams& p) { return cmp_check_strides(p.k_sn, p.v_sn); }

#define FSA_CMP_DISPATCH(FN, P, ...)                                                      \
  do {                                                                                    \
    if (int rc_ = cmp_check_strides(P)) return rc_;                                       \
    if (dtype == FSA_BF16) {                                                              \
      if (head_dim == 64) return FN<__bf16, 64>(P, __VA_ARGS__);                          \
      if (head_dim == 128) return FN<__bf16, 128>(P, __VA_ARGS__);                           \
      if (head_dim == 256) return FN<__bf16, 256>(P, __VA_ARGS__);                           \
    } else {                                                                              \
      if (head_dim == 64) return FN<_Float16, 64>(P, __VA_ARGS__);                           \
      if (head_dim == 128) return FN<_Float16, 128>(P, __VA_ARGS__);                         \
      if (head_dim == 256) return FN<_Float16, 256>(P, __VA_ARGS__);                         \
    }                                                                                     \
    set_error("compressed attention: head_dim=%d not supported (64, 128, 256)", head_dim); \
    return FSA_ERR_UNSUPPORTED;                                                           \
  } while (0)

static int cmp_fwd_dispatch(int dtype, int head_dim, const CmpParams& p, int batch, int hkv,
                            int64_t max_rows, hipStream_t stream) {
  FSA_CMP_DISPATCH(cmp_fwd_launch, p, batch, hkv, max_rows, stream);
}
static int cmp_bwd_dispatch(int dtype, int head_dim, const CmpParams& p, const SelBwdParams& kv, int batch,
                            int hq, int hkv, int64_t max_rows, int64_t n, bool straight, hipStream_t stream) {
  FSA_CMP_DISPATCH(cmp_bwd_launch, p, kv, batch, hq, hkv, max_rows, n, straight, stream);
}
static int win_fwd_dispatch(int dtype, int head_dim, const CmpParams& p, int batch, int hkv,
                            int64_t max_rows, hipStream_t stream) {
  FSA_CMP_DISPATCH(win_fwd_launch, p, batch, hkv, max_rows, stream);
}
static int win_bwd_dispatch(int dtype, int head_dim, const CmpParams& p, const SelBwdParams& kv, int batch,
                            int hq, int hkv, int64_t max_rows, int64_t n, bool straight, hipStream_t stream) {
  FSA_CMP_DISPATCH(win_bwd_launch, p, kv, batch, hq, hkv, max_rows, n, straight, stream);
}
static int pair_fwd_dispatch(int dtype, int head_dim, const CmpParams& a, const CmpParams& b, int batch, int hkv,
                             int64_t max_rows, hipStream_t stream) {
  FSA_CMP_DISPATCH(pair_fwd_launch, a, b, batch, hkv, max_rows, stream);
}
static int pair_bwd_dispatch(int dtype, int head_dim, const CmpParams& a, const CmpParams& b, const SelBwdParams& ka,
                             const SelBwdParams& kb, const KvTiles& ta, const KvTiles& tb, int batch, int hkv, int64_t max_rows,
                             bool straight, hipStream_t stream) {
  FSA_CMP_DISPATCH(pair_bwd_launch, a, b, ka, kb, ta, tb, batch, hkv, max_rows, straight, stream);
}
static int cmp_score_dispatch(int dtype, int head_dim, const CmpParams& p, int batch, int hkv,
                              int64_t max_q, hipStream_t stream) {
  FSA_CMP_DISPATCH(cmp_score_launch, p, batch, hkv, max_q, stream);
}

}  // namespace fsa

using namespace fsa;

static int cmp_check_common(const char* who, int32_t dtype, int32_t hq, int32_t hkv, int32_t ks,
                            int32_t stride, int32_t batch, int64_t n) {
  FSA_CHECK_ARG(dtype == FSA_BF16 || dtype == FSA_FP16, "%s: dtype must be bf16 or fp16", who);
  FSA_CHECK_ARG(hkv >= 1 && hq % hkv == 0, "%s: num_q_heads must be a multiple of num_kv_heads", who);
  FSA_CHECK_ARG(ks >= 1 && stride >= 1 && ks % stride == 0,
                "%s: kernel_size must be a positive multiple of kernel_stride", who);
  FSA_CHECK_ARG(batch >= 1 && n >= 1, "%s: empty problem", who);
  return 0;
}

extern "C" int fsa_cmpattn_fwd(const void* q, const void* ck, const void* cv, int32_t dtype,
                               int64_t q_stride_n, int64_t q_stride_h, int64_t k_stride_n,
                               int64_t k_stride_h, int64_t v_stride_n, int64_t v_stride_h,
                               const int32_t* cu_seqlens_q, const int32_t* cu_seqlens_k, int32_t batch,
                               int64_t total_q, int64_t max_seqlen_q, int32_t num_q_heads,
                               int32_t num_kv_heads, int32_t head_dim, int32_t kernel_size,
                               int32_t kernel_stride, float softmax_scale, void* o, int64_t o_stride_n,
                               int64_t o_stride_h, float* lse, void* stream_) {
  FSA_CHECK_ARG(q && ck && cv && o && lse && cu_seqlens_q && cu_seqlens_k, "fsa_cmpattn_fwd: null pointer");
  int rc = cmp_check_common("fsa_cmpattn_fwd", dtype, num_q_heads, num_kv_heads, kernel_size, kernel_stride,
                            batch, total_q);
  if (rc) return rc;
  FSA_CHECK_ARG(max_seqlen_q >= 1 && max_seqlen_q <= total_q, "fsa_cmpattn_fwd: bad max_seqlen_q");
  CmpParams p = {};
  p.q = q; p.k = ck; p.v = cv; p.o = o; p.lse = lse;
  p.q_sn = q_stride_n; p.q_sh = q_stride_h; p.k_sn = k_stride_n; p.k_sh = k_stride_h;
  p.v_sn = v_stride_n; p.v_sh = v_stride_h; p.o_sn = o_stride_n; p.o_sh = o_stride_h;
  p.cu_q = cu_seqlens_q; p.cu_k = cu_seqlens_k; p.n_tokens = total_q;
  p.g = num_q_heads / num_kv_heads; p.kernel_size = kernel_size; p.kernel_stride = kernel_stride;
  p.scale = softmax_scale; p.scale_log2 = softmax_scale * LOG2E;
  rc = cmp_fwd_dispatch(dtype, head_dim, p, batch, num_kv_heads, max_seqlen_q * p.g, (hipStream_t)stream_);
  if (rc) return rc;
  FSA_CHECK_LAUNCH("fsa_cmpattn_fwd");
  return 0;
}

extern "C" size_t fsa_cmpattn_bwd_workspace_bytes(int64_t total_q, int64_t total_k, int64_t max_seqlen_q,
                                                  int32_t batch, int32_t num_q_heads,
                                                  int32_t num_kv_heads, int32_t head_dim) {
  return cmp_bwd_ws(total_q, total_k, max_seqlen_q, batch, num_q_heads, num_kv_heads, head_dim, false).total;   // (of either kernel)
}

extern "C" int fsa_cmpattn_bwd(const void* q, const void* ck, const void* cv, const void* o,
                               const void* d_o, const float* lse, int32_t dtype, int64_t q_stride_n,
                               int64_t q_stride_h, int64_t k_stride_n, int64_t k_stride_h,
                               int64_t v_stride_n, int64_t v_stride_h, int64_t o_stride_n,
                               int64_t o_stride_h, int64_t do_stride_n, int64_t do_stride_h,
                               const int32_t* cu_seqlens_q, const int32_t* cu_seqlens_k, int32_t batch,
                               int64_t total_q, int64_t total_k, int64_t max_seqlen_q,
                               int32_t num_q_heads, int32_t num_kv_heads, int32_t head_dim,
                               int32_t kernel_size, int32_t kernel_stride, float softmax_scale, void* dq,
                               void* dck, void* dcv, void* workspace, size_t workspace_bytes,
                               void* stream_) {
  hipStream_t stream = (hipStream_t)stream_;
  FSA_CHECK_ARG(q && ck && cv && o && lse && d_o && dq && dck && dcv && cu_seqlens_q && cu_seqlens_k,
                "fsa_cmpattn_bwd: null pointer");
  int rc = cmp_check_common("fsa_cmpattn_bwd", dtype, num_q_heads, num_kv_heads, kernel_size, kernel_stride,
                            batch, total_q);
  if (rc) return rc;
  FSA_CHECK_ARG(total_k >= 1, "fsa_cmpattn_bwd: no compressed keys");
  FSA_CHECK_ARG(max_seqlen_q >= 1 && max_seqlen_q <= total_q, "fsa_cmpattn_bwd: bad max_seqlen_q");
  const bool straight = dense_kv_rows_ok(q, q_stride_n, q_stride_h, d_o, do_stride_n, do_stride_h, total_q,
                                         num_q_heads / num_kv_heads, head_dim);
  CmpBwdWs ws = cmp_bwd_ws(total_q, total_k, max_seqlen_q, batch, num_q_heads, num_kv_heads, head_dim, straight);
  if (!workspace || workspace_bytes < ws.total) {
    set_error("fsa_cmpattn_bwd: workspace too small (%zu < %zu)", workspace_bytes, ws.total);
    return FSA_ERR_WORKSPACE;
  }
  char* wsp = (char*)workspace;
  const int g = num_q_heads / num_kv_heads;
  FSA_CHECK_ARG(kv_qdo_strides_ok(q_stride_n, q_stride_h, do_stride_n, do_stride_h, g, head_dim),
                "fsa_cmpattn_bwd: q / d_o strides too large or negative");
  if (int rc_ = cmp_check_strides(k_stride_n, v_stride_n)) return rc_;
  float* delta = (float*)(wsp + ws.off_delta);
  int32_t* cu_tiles = (int32_t*)(wsp + ws.off_cu_tiles);
  int32_t* counts = (int32_t*)(wsp + ws.off_counts);
  int32_t* tile_prefix = (int32_t*)(wsp + ws.off_tiles);
  const KvTiles tiles = {cu_seqlens_q, cu_seqlens_k, ws.max_blocks, kernel_size, kernel_stride, 0, ws.tile_rows, cu_tiles, counts,
                         tile_prefix};
  kv_tiles_kernel<CMP_MODE_COMPRESSED><<<num_kv_heads, KT_THREADS, 0, stream>>>(tiles, batch, g);

  CmpParams p = {};
  p.q = q; p.k = ck; p.v = cv; p.o = (void*)o; p.d_o = d_o; p.dq = dq; p.lse = (float*)lse; p.delta = delta;
  p.q_sn = q_stride_n; p.q_sh = q_stride_h; p.k_sn = k_stride_n; p.k_sh = k_stride_h;
  p.v_sn = v_stride_n; p.v_sh = v_stride_h; p.o_sn = o_stride_n; p.o_sh = o_stride_h;
  p.do_sn = do_stride_n; p.do_sh = do_stride_h;
  p.cu_q = cu_seqlens_q; p.cu_k = cu_seqlens_k; p.n_tokens = total_q;
  p.g = g; p.kernel_size = kernel_size; p.kernel_stride = kernel_stride;
  p.scale = softmax_scale; p.scale_log2 = softmax_scale * LOG2E;

  SelBwdParams kv = {};
  kv.q = q; kv.k = ck; kv.v = cv; kv.d_o = d_o; kv.lse = lse; kv.delta = delta; kv.hq = num_q_heads;
  kv.q_sn = q_stride_n; kv.q_sh = q_stride_h; kv.k_sn = k_stride_n; kv.k_sh = k_stride_h;
  kv.v_sn = v_stride_n; kv.v_sh = v_stride_h; kv.do_sn = do_stride_n; kv.do_sh = do_stride_h;
  kv.cu_seqlens = cu_seqlens_q; kv.cu_blocks = cu_tiles; kv.counts = counts; kv.starts = nullptr;
  kv.sel_tokens = nullptr; kv.tile_prefix = tile_prefix;
  kv.batch = batch; kv.max_blocks = ws.max_blocks; kv.cap = 0; kv.n_tokens = total_q; kv.g = g; kv.g_shift = group_shift(g);
  kv.scale = softmax_scale; kv.scale_log2 = softmax_scale * LOG2E;
  kv.dq_part = nullptr; kv.dkdv_part = (float*)(wsp + ws.off_part); kv.max_tiles = ws.max_tiles;
  kv.dk = dck; kv.dv = dcv; kv.dk_sn = (int64_t)num_kv_heads * head_dim; kv.dk_sh = head_dim;
  kv.cu_seqlens_k = cu_seqlens_k; kv.kernel_size = kernel_size; kv.kernel_stride = kernel_stride;

  rc = cmp_bwd_dispatch(dtype, head_dim, p, kv, batch, num_q_heads, num_kv_heads, max_seqlen_q * g, total_q,
                        straight, stream);
  if (rc) return rc;
  FSA_CHECK_LAUNCH("fsa_cmpattn_bwd");
  return 0;
}

extern "C" size_t fsa_cmp_topk_workspace_bytes(int64_t total_q, int32_t num_kv_heads, int64_t max_seqlen_k) {
  const int64_t ld = (max_seqlen_k + 3) / 4 * 4;
  return align_up((size_t)total_q * num_kv_heads * ld * 4, 256);
}

extern "C" int fsa_cmp_topk(const void* q, const void* ck, const float* lse, int32_t dtype,
                            int64_t q_stride_n, int64_t q_stride_h, int64_t k_stride_n, int64_t k_stride_h,
                            const int32_t* cu_seqlens_q, const int32_t* cu_seqlens_k, int32_t batch,
                            int64_t total_q, int64_t max_seqlen_q, int64_t max_seqlen_k,
                            int32_t num_q_heads, int32_t num_kv_heads, int32_t head_dim,
                            int32_t kernel_size, int32_t kernel_stride, int32_t block_size, int32_t topk,
                            int32_t init_blocks, int32_t local_blocks, int32_t scores_to_bf16,
                            int32_t score_head_as_written, float softmax_scale, int32_t* topk_idx,
                            float* block_score, void* workspace,
                            size_t workspace_bytes, void* stream_) {
  hipStream_t stream = (hipStream_t)stream_;
  FSA_CHECK_ARG(q && ck && lse && topk_idx && cu_seqlens_q && cu_seqlens_k, "fsa_cmp_topk: null pointer");
  int rc = cmp_check_common("fsa_cmp_topk", dtype, num_q_heads, num_kv_heads, kernel_size, kernel_stride,
                            batch, total_q);
  if (rc) return rc;
  FSA_CHECK_ARG(block_size >= kernel_stride && block_size % kernel_stride == 0,
                "fsa_cmp_topk: block_size must be a multiple of kernel_stride");
  FSA_CHECK_ARG(topk >= 1 && max_seqlen_q >= 1 && max_seqlen_k >= 1, "fsa_cmp_topk: bad sizes");
  const int nblk = (int)((max_seqlen_q + block_size - 1) / block_size);
  const int t_out = topk < nblk ? topk : nblk;
  // more than 64 selected blocks per query or more than 4096 blocks per sequence: one-wave work-groups with
  // scores and chosen ids in LDS, which bounds their sum
  const bool big = t_out > 64 || nblk > 4096;
  FSA_CHECK_ARG(!big || ((int64_t)nblk + t_out) * 4 <= 160 * 1024,
                "fsa_cmp_topk: blocks per sequence + selected blocks per query exceed 40960");
  // usual geometry (window of 2 strides, block of 4): the score kernel writes block scores, at most
  // max_seqlen_k / 4 + 1 per query, instead of one probability per compressed key
  const bool rebin = kernel_size == 2 * kernel_stride && block_size == 4 * kernel_stride;
  const int64_t score_cols = rebin ? max_seqlen_k / 4 + 1 : max_seqlen_k;
  const size_t need = fsa_cmp_topk_workspace_bytes(total_q, num_kv_heads, score_cols);
  if (!workspace || workspace_bytes < need) {
    set_error("fsa_cmp_topk: workspace too small (%zu < %zu)", workspace_bytes, need);
    return FSA_ERR_WORKSPACE;
  }
  CmpParams p = {};
  p.q = q; p.k = ck; p.lse = (float*)lse;
  p.q_sn = q_stride_n; p.q_sh = q_stride_h; p.k_sn = k_stride_n; p.k_sh = k_stride_h;
  p.cu_q = cu_seqlens_q; p.cu_k = cu_seqlens_k; p.n_tokens = total_q;
  p.g = num_q_heads / num_kv_heads; p.kernel_size = kernel_size; p.kernel_stride = kernel_stride;
  p.scale = softmax_scale; p.scale_log2 = softmax_scale * LOG2E;
  p.rebin = rebin;
  p.score_head_step = score_head_as_written ? 1 : p.g;
  p.score = (float*)workspace;
  p.score_ld = (score_cols + 3) / 4 * 4;
  rc = cmp_score_dispatch(dtype, head_dim, p, batch, num_kv_heads, max_seqlen_q, stream);
  if (rc) return rc;
  FSA_CHECK_LAUNCH("fsa_cmp_topk score");
  TopkParams tp = {};
  tp.score = p.score; tp.score_ld = p.score_ld; tp.cu_q = cu_seqlens_q; tp.cu_k = cu_seqlens_k;
  tp.batch = batch; tp.n_tokens = total_q; tp.hkv = num_kv_heads;
  tp.kernel_size = kernel_size; tp.kernel_stride = kernel_stride; tp.block_size = block_size;
  tp.na = kernel_size / kernel_stride; tp.ne = block_size / kernel_stride; tp.rebin = p.rebin;
  tp.nblk = nblk; tp.t_out = t_out; tp.init_blocks = init_blocks; tp.local_blocks = local_blocks;
  tp.to_bf16 = scores_to_bf16; tp.topk_idx = topk_idx; tp.block_score = block_score;
  {
    ProfScope ps_("cmp_topk", stream);
    const dim3 grid((unsigned)((total_q + 3) / 4), (unsigned)num_kv_heads);
    if (big) {
      const int lds = (nblk + t_out) * 4;
      if (lds > 48 * 1024)
        if (int rc_ = set_lds_limit((const void*)cmp_topk_kernel<0, true>, lds)) return rc_;
      cmp_topk_kernel<0, true><<<dim3((unsigned)total_q, (unsigned)num_kv_heads), 64, lds, stream>>>(tp);
    } else if (scores_to_bf16 && nblk <= 128) cmp_topk_kernel<2><<<grid, 256, 0, stream>>>(tp);
    else if (scores_to_bf16 && nblk <= 256) cmp_topk_kernel<4><<<grid, 256, 0, stream>>>(tp);
    else if (scores_to_bf16 && nblk <= 512) cmp_topk_kernel<8><<<grid, 256, 0, stream>>>(tp);
    else if (scores_to_bf16 && nblk <= 1024) cmp_topk_kernel<16><<<grid, 256, 0, stream>>>(tp);
    else cmp_topk_kernel<0><<<grid, 256, (size_t)4 * nblk * 4, stream>>>(tp);
  }
  FSA_CHECK_LAUNCH("fsa_cmp_topk select");
  return 0;
}

// ------------------------------------------------------------------------------------------------
// Sliding-window attention (causal band of `window` + 1 keys): the third branch of the module.
extern "C" int fsa_winattn_fwd(const void* q, const void* k, const void* v, int32_t dtype,
                               int64_t q_stride_n, int64_t q_stride_h, int64_t k_stride_n,
                               int64_t k_stride_h, int64_t v_stride_n, int64_t v_stride_h,
                               const int32_t* cu_seqlens, int32_t batch, int64_t total_tokens,
                               int64_t max_seqlen, int32_t num_q_heads, int32_t num_kv_heads,
                               int32_t head_dim, int32_t window, float softmax_scale, void* o,
                               int64_t o_stride_n, int64_t o_stride_h, float* lse, void* stream_) {
  FSA_CHECK_ARG(q && k && v && o && lse && cu_seqlens, "fsa_winattn_fwd: null pointer");
  int rc = cmp_check_common("fsa_winattn_fwd", dtype, num_q_heads, num_kv_heads, 1, 1, batch, total_tokens);
  if (rc) return rc;
  FSA_CHECK_ARG(window >= 0 && max_seqlen >= 1 && max_seqlen <= total_tokens, "fsa_winattn_fwd: bad sizes");
  CmpParams p = {};
  p.q = q; p.k = k; p.v = v; p.o = o; p.lse = lse;
  p.q_sn = q_stride_n; p.q_sh = q_stride_h; p.k_sn = k_stride_n; p.k_sh = k_stride_h;
  p.v_sn = v_stride_n; p.v_sh = v_stride_h; p.o_sn = o_stride_n; p.o_sh = o_stride_h;
  p.cu_q = cu_seqlens; p.cu_k = cu_seqlens; p.n_tokens = total_tokens;
  p.g = num_q_heads / num_kv_heads; p.kernel_size = 1; p.kernel_stride = 1; p.window = window;
  p.scale = softmax_scale; p.scale_log2 = softmax_scale * LOG2E;
  rc = win_fwd_dispatch(dtype, head_dim, p, batch, num_kv_heads, max_seqlen * p.g, (hipStream_t)stream_);
  if (rc) return rc;
  FSA_CHECK_LAUNCH("fsa_winattn_fwd");
  return 0;
}

static CmpBwdWs win_bwd_ws(int64_t n, int64_t max_q, int window, int batch, int hq, int hkv, int d, bool straight) {
  CmpBwdWs w = cmp_bwd_ws(n, n, max_q, batch, hq, hkv, d, straight);
  const int g = hq / hkv;
  dense_tiles(w, (int64_t)(CMP_BK + window) * g, win_rows_total(w.max_blocks, window, hq), g, hkv, d, straight);
  return w;
}

extern "C" size_t fsa_winattn_bwd_workspace_bytes(int64_t total_tokens, int64_t max_seqlen, int32_t window,
                                                  int32_t batch, int32_t num_q_heads,
                                                  int32_t num_kv_heads, int32_t head_dim) {
  return win_bwd_ws(total_tokens, max_seqlen, window, batch, num_q_heads, num_kv_heads, head_dim, false).total;
}

extern "C" int fsa_winattn_bwd(const void* q, const void* k, const void* v, const void* o, const void* d_o,
                               const float* lse, int32_t dtype, int64_t q_stride_n, int64_t q_stride_h,
                               int64_t k_stride_n, int64_t k_stride_h, int64_t v_stride_n,
                               int64_t v_stride_h, int64_t o_stride_n, int64_t o_stride_h,
                               int64_t do_stride_n, int64_t do_stride_h, const int32_t* cu_seqlens,
                               int32_t batch, int64_t total_tokens, int64_t max_seqlen,
                               int32_t num_q_heads, int32_t num_kv_heads, int32_t head_dim,
                               int32_t window, float softmax_scale, void* dq, void* dk, void* dv,
                               void* workspace, size_t workspace_bytes, void* stream_) {
  hipStream_t stream = (hipStream_t)stream_;
  FSA_CHECK_ARG(q && k && v && o && lse && d_o && dq && dk && dv && cu_seqlens, "fsa_winattn_bwd: null pointer");
  int rc = cmp_check_common("fsa_winattn_bwd", dtype, num_q_heads, num_kv_heads, 1, 1, batch, total_tokens);
  if (rc) return rc;
  FSA_CHECK_ARG(window >= 0 && max_seqlen >= 1 && max_seqlen <= total_tokens, "fsa_winattn_bwd: bad sizes");
  const bool straight = dense_kv_rows_ok(q, q_stride_n, q_stride_h, d_o, do_stride_n, do_stride_h, total_tokens,
                                         num_q_heads / num_kv_heads, head_dim);
  CmpBwdWs ws = win_bwd_ws(total_tokens, max_seqlen, window, batch, num_q_heads, num_kv_heads, head_dim, straight);
  if (!workspace || workspace_bytes < ws.total) {
    set_error("fsa_winattn_bwd: workspace too small (%zu < %zu)", workspace_bytes, ws.total);
    return FSA_ERR_WORKSPACE;
  }
  char* wsp = (char*)workspace;
  const int g = num_q_heads / num_kv_heads;
  FSA_CHECK_ARG(kv_qdo_strides_ok(q_stride_n, q_stride_h, do_stride_n, do_stride_h, g, head_dim),
                "fsa_winattn_bwd: q / d_o strides too large or negative");
  if (int rc_ = cmp_check_strides(k_stride_n, v_stride_n)) return rc_;
  float* delta = (float*)(wsp + ws.off_delta);
  int32_t* cu_tiles = (int32_t*)(wsp + ws.off_cu_tiles);
  int32_t* counts = (int32_t*)(wsp + ws.off_counts);
  int32_t* tile_prefix = (int32_t*)(wsp + ws.off_tiles);
  const KvTiles tiles = {cu_seqlens, cu_seqlens, ws.max_blocks, 1, 1, window, ws.tile_rows, cu_tiles, counts, tile_prefix};
  kv_tiles_kernel<CMP_MODE_WINDOW><<<num_kv_heads, KT_THREADS, 0, stream>>>(tiles, batch, g);

  CmpParams p = {};
  p.q = q; p.k = k; p.v = v; p.o = (void*)o; p.d_o = d_o; p.dq = dq; p.lse = (float*)lse; p.delta = delta;
  p.q_sn = q_stride_n; p.q_sh = q_stride_h; p.k_sn = k_stride_n; p.k_sh = k_stride_h;
  p.v_sn = v_stride_n; p.v_sh = v_stride_h; p.o_sn = o_stride_n; p.o_sh = o_stride_h;
  p.do_sn = do_stride_n; p.do_sh = do_stride_h;
  p.cu_q = cu_seqlens; p.cu_k = cu_seqlens; p.n_tokens = total_tokens;
  p.g = g; p.kernel_size = 1; p.kernel_stride = 1; p.window = window;
  p.scale = softmax_scale; p.scale_log2 = softmax_scale * LOG2E;

  SelBwdParams kv = {};
  kv.q = q; kv.k = k; kv.v = v; kv.d_o = d_o; kv.lse = lse; kv.delta = delta; kv.hq = num_q_heads;
  kv.q_sn = q_stride_n; kv.q_sh = q_stride_h; kv.k_sn = k_stride_n; kv.k_sh = k_stride_h;
  kv.v_sn = v_stride_n; kv.v_sh = v_stride_h; kv.do_sn = do_stride_n; kv.do_sh = do_stride_h;
  kv.cu_seqlens = cu_seqlens; kv.cu_blocks = cu_tiles; kv.counts = counts; kv.tile_prefix = tile_prefix;
  kv.batch = batch; kv.max_blocks = ws.max_blocks; kv.n_tokens = total_tokens; kv.g = g; kv.g_shift = group_shift(g);
  kv.scale = softmax_scale; kv.scale_log2 = softmax_scale * LOG2E;
  kv.dkdv_part = (float*)(wsp + ws.off_part); kv.max_tiles = ws.max_tiles;
  kv.dk = dk; kv.dv = dv; kv.dk_sn = (int64_t)num_kv_heads * head_dim; kv.dk_sh = head_dim;
  kv.cu_seqlens_k = cu_seqlens; kv.kernel_size = 1; kv.kernel_stride = 1; kv.window = window;

  rc = win_bwd_dispatch(dtype, head_dim, p, kv, batch, num_q_heads, num_kv_heads, max_seqlen * g, total_tokens,
                        straight, stream);
  if (rc) return rc;
  FSA_CHECK_LAUNCH("fsa_winattn_bwd");
  return 0;
}

// ------------------------------------------------------------------------------------------------
// Both dense branches of a layer at once, on contiguous tensors.
static CmpParams pair_params(const LayerAttn& l, bool window) {
  CmpParams p = {};
  const int64_t d = l.head_dim;
  p.q = l.q; p.k = window ? l.k : l.ck; p.v = window ? l.v : l.cv;
  p.o = window ? l.o_win : l.o_cmp; p.lse = window ? l.lse_win : l.lse_cmp;
  p.d_o = l.d_out; p.dq = window ? l.dq_win : l.dq_cmp; p.stat2 = window ? l.stat_win : l.stat_cmp;
  p.q_sn = p.o_sn = p.do_sn = l.hq * d; p.q_sh = p.k_sh = p.v_sh = p.o_sh = p.do_sh = d; p.k_sn = p.v_sn = l.hkv * d;
  p.cu_q = l.cu; p.cu_k = window ? l.cu : l.cu_ck; p.n_tokens = l.n;
  p.g = l.hq / l.hkv; p.kernel_size = window ? 1 : l.kernel_size; p.kernel_stride = window ? 1 : l.kernel_stride;
  p.window = l.window;
  p.scale = l.scale; p.scale_log2 = l.scale * LOG2E;
  return p;
}

int fsa::layer_attn_fwd(const LayerAttn& l, hipStream_t stream) {
  const int dtype = l.dtype, head_dim = l.head_dim;
  if (int rc = pair_fwd_dispatch(dtype, head_dim, pair_params(l, false), pair_params(l, true), l.batch, l.hkv,
                                 l.max_len * (l.hq / l.hkv), stream))
    return rc;
  FSA_CHECK_LAUNCH("fsa_layer attention");
  return 0;
}

size_t fsa::layer_attn_bwd_workspace_bytes(int64_t n, int64_t total_ck, int64_t max_len, int window, int batch, int hq, int hkv, int d) {
  return cmp_bwd_ws(n, total_ck, max_len, batch, hq, hkv, d, false).total + win_bwd_ws(n, max_len, window, batch, hq, hkv, d, false).total;
}

int fsa::layer_attn_bwd(const LayerAttn& l, void* workspace, hipStream_t stream) {
  const int dtype = l.dtype, head_dim = l.head_dim, g = l.hq / l.hkv;
  const int64_t row = (int64_t)l.hq * head_dim;
  const bool straight = dense_kv_rows_ok(l.q, row, head_dim, l.d_out, row, head_dim, l.n, g, head_dim);
  const CmpBwdWs w[2] = {cmp_bwd_ws(l.n, l.total_ck, l.max_len, l.batch, l.hq, l.hkv, head_dim, straight),
                         win_bwd_ws(l.n, l.max_len, l.window, l.batch, l.hq, l.hkv, head_dim, straight)};
  CmpParams p[2];
  SelBwdParams kv[2] = {};
  KvTiles tiles[2];
  char* ws = (char*)workspace;
  for (int i = 0; i < 2; ++i) {
    p[i] = pair_params(l, i == 1);
    int32_t *cu_tiles = (int32_t*)(ws + w[i].off_cu_tiles), *counts = (int32_t*)(ws + w[i].off_counts),
            *prefix = (int32_t*)(ws + w[i].off_tiles);
    tiles[i] = {p[i].cu_q, p[i].cu_k, w[i].max_blocks, p[i].kernel_size, p[i].kernel_stride, p[i].window, w[i].tile_rows,
                cu_tiles, counts, prefix};
    SelBwdParams& k = kv[i];
    k.q = p[i].q; k.k = p[i].k; k.v = p[i].v; k.d_o = p[i].d_o; k.stat2 = p[i].stat2; k.hq = l.hq;
    k.q_sn = p[i].q_sn; k.q_sh = p[i].q_sh; k.k_sn = p[i].k_sn; k.k_sh = p[i].k_sh; k.v_sn = p[i].v_sn; k.v_sh = p[i].v_sh;
    k.do_sn = p[i].do_sn; k.do_sh = p[i].do_sh;
    k.cu_seqlens = p[i].cu_q; k.cu_seqlens_k = p[i].cu_k; k.cu_blocks = cu_tiles; k.counts = counts; k.tile_prefix = prefix;
    k.batch = l.batch; k.max_blocks = w[i].max_blocks; k.n_tokens = l.n; k.g = g; k.g_shift = group_shift(g);
    k.scale = p[i].scale; k.scale_log2 = p[i].scale_log2;
    k.dkdv_part = (float*)(ws + w[i].off_part); k.max_tiles = w[i].max_tiles;
    k.dk = i ? l.dk_win : l.dck; k.dv = i ? l.dv_win : l.dcv; k.dk_sn = p[i].k_sn; k.dk_sh = head_dim;
    k.kernel_size = p[i].kernel_size; k.kernel_stride = p[i].kernel_stride; k.window = p[i].window;
    ws += w[i].total;
  }
  FSA_CHECK_ARG(kv_qdo_strides_ok(kv[0].q_sn, kv[0].q_sh, kv[0].do_sn, kv[0].do_sh, g, head_dim), "fsa_layer: too many heads");
  if (int rc = pair_bwd_dispatch(dtype, head_dim, p[0], p[1], kv[0], kv[1], tiles[0], tiles[1], l.batch, l.hkv, l.max_len * g, straight, stream))
    return rc;
  FSA_CHECK_LAUNCH("fsa_layer attention backward");
  return 0;
}
