// Selected attention of short sequences, straight from the block lists: no inverted index, no partial rows.
//
// Where a sequence has few blocks, the rows (query, head-in-group) of a query tile together select nearly every block they
// may see, and a query-major kernel that visits the union of their blocks does little more arithmetic than the block-major
// pair (selattn_fwd_main / _reduce) while it reads q once and writes o once.
//
// Two kernels.  What a wave does in a step is the same in both: 32 rows against 32 keys, K and V from LDS tiles that buffer loads
// fill past the registers.
//
//   narrow  few row tiles: a work-group takes one, its KG waves share out the visited keys, each with K / V buffers of its own,
//           so there is no barrier between the first step and the merge of the partial results in LDS.
//   wide    many row tiles: a work-group takes RT of them, whose waves go through the keys together and share every tile.
#include "attn_rows.h"

#include <algorithm>
#include <cmath>
#include <type_traits>

namespace fsa {

struct DirectParams {
  const void *q, *k, *v;
  int64_t q_sn, q_sh, k_sn, k_sh, v_sn, v_sh, o_sn, o_sh;
  const int32_t* topk_idx;   // [Hkv, N, T]
  int64_t i_sh, i_sn;
  const int32_t* cu;
  int batch, hkv, g, g_shift, topk, max_blk;   // max_blk: blocks of the longest sequence the tables hold
  int bk_shift;                                // log2 of the block size
  int64_t n_tokens;
  float scale_log2;
  void* o;
  float* lse;
  MergeEpilogue merge;
};

// A row tile.  The rows of the whole buffer are dealt out, so that none of o and lse stays unwritten where the sequences do not
// fill it: segment i runs from cu[i - 1] to cu[i], with the start of the buffer in front and its end behind.  Segment 0, in
// front of the first sequence, has no keys; the last one holds the last sequence and, as queries at the positions behind it,
// the tokens that follow it, which is where the inverted index counts them too.
struct DirectTile {
  int q0, n_q, len;   // first token, queries and keys of its segment
  int tile;           // of the segment
};
// Row tile of work-group `id`, `per_tile` rows each; false: past the last one.  The late tiles of a segment, which see the most
// blocks, come first.
__device__ __forceinline__ bool direct_tile(const int32_t* __restrict__ cu, int batch, int n_tokens, int g, int per_tile, int id,
                                            DirectTile& t) {
  const int lane = threadIdx.x & (WAVE - 1);
  for (int s0 = 0; s0 <= batch; s0 += WAVE) {
    const int si = s0 + lane;
    const int a = cu[min(max(si - 1, 0), batch)], b = cu[min(si, batch)];
    const int q0 = si > 0 ? a : 0, n_q = (si < batch ? b : n_tokens) - q0;
    const int n = si <= batch ? (int)(((int64_t)n_q * g + per_tile - 1) / per_tile) : 0;
    int inc = n;
#pragma unroll
    for (int o = 1; o < WAVE; o <<= 1) {
      const int x = __shfl_up(inc, o, WAVE);
      if (lane >= o) inc += x;
    }
    const uint64_t m = __ballot(inc > id);
    if (m) {
      const int at = __ffsll((unsigned long long)m) - 1;
      t.q0 = __builtin_amdgcn_readlane(q0, at);
      t.n_q = __builtin_amdgcn_readlane(n_q, at);
      t.len = s0 + at > 0 ? __builtin_amdgcn_readlane(b - a, at) : 0;
      t.tile = __builtin_amdgcn_readlane(inc, at) - 1 - id;
      return true;
    }
    id -= __builtin_amdgcn_readlane(inc, WAVE - 1);
  }
  return false;
}

// Chunk `sub` (8 dims) of row r of a row tile, from the partial results of KG waves: partial w at part + w * part_step bytes,
// its statistics at st_m + w * st_step.
template <typename T, int D, bool MERGE, int KG>
__device__ __forceinline__ void direct_store(const DirectParams& p, int h, int q0, int row, int r, int sub, const unsigned char* part, int part_step,
                                             const float* st_m, const float* st_l, int st_step) {
  typedef typename Elem<T>::vec8 vec8;
  constexpr int XM = AttnRows<T, D>::XM;
  float mw[KG], mx = -INFINITY;
#pragma unroll
  for (int w = 0; w < KG; ++w) {
    mw[w] = st_m[w * st_step + r];
    mx = fmaxf(mx, mw[w]);
  }
  float sum = 0.f, out[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) out[e] = 0.f;
#pragma unroll
  for (int w = 0; w < KG; ++w) {
    mw[w] = mx == -INFINITY ? 0.f : fast_exp2(mw[w] - mx);
    sum += mw[w] * st_l[w * st_step + r];
    const float* pw = reinterpret_cast<const float*>(part + w * part_step) + r * D;
    const f32x4 x0 = *reinterpret_cast<const f32x4*>(pw + ((2 * sub) ^ (r & XM)) * 4);
    const f32x4 x1 = *reinterpret_cast<const f32x4*>(pw + ((2 * sub + 1) ^ (r & XM)) * 4);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      out[e] += mw[w] * x0[e];
      out[4 + e] += mw[w] * x1[e];
    }
    }
  const float inv = sum == 0.f ? 0.f : 1.f / sum;   // (a sum that is NaN, from a NaN in q or a key, makes the row NaN)
  vec8 x;
#pragma unroll
  for (int e = 0; e < 8; ++e) x[e] = (T)(out[e] * inv);
  const int qi = div_group(row, p.g, p.g_shift), hq_i = h * p.g + row - qi * p.g;
  const int64_t tok = q0 + qi;
  if constexpr (MERGE) {
    const int64_t at = (tok * (p.hkv * p.g) + hq_i) * D + sub * 8;
    const vec8 xa = load16_stream<vec8>(reinterpret_cast<const T*>(p.merge.a) + at);
    const vec8 xc = load16_stream<vec8>(reinterpret_cast<const T*>(p.merge.c) + at);
    const T* gate = reinterpret_cast<const T*>(p.merge.gate) + tok * 3;
    const float g0 = (float)gate[0], g1 = (float)gate[1], g2 = (float)gate[2];
    vec8 y;
#pragma unroll
    for (int e = 0; e < 8; ++e) y[e] = (T)(g0 * (float)xa[e] + g1 * (float)x[e] + g2 * (float)xc[e]);
    store16(reinterpret_cast<T*>(p.merge.out) + at, y);
    if (!p.o) return;
  }
  store16(reinterpret_cast<T*>(p.o) + tok * p.o_sn + (int64_t)hq_i * p.o_sh + sub * 8, x);
  if (sub == 0) p.lse[(int64_t)hq_i * p.n_tokens + tok] = sum == 0.f ? -INFINITY : mx + log2f(sum);
}

// How often the lane's query names block b.
__device__ __forceinline__ float direct_times(const DirectParams& p, int h, int tok, int b) {
  const int32_t* ids = p.topk_idx + h * p.i_sh + (int64_t)tok * p.i_sn;
  int c = 0;
  for (int i = 0; i < p.topk; ++i) c += ids[i] == b;
  return (float)c;
}

// ---- narrow: one row tile, KG key groups of one wave -----------------------------------------------------------------------
// Bound by the chain of a step (products, maximum, exponentials, products: 0.8 us for a wave that is alone on its SIMD) in the
// longest work-group.  q is settled in front of the loop, and the lists are read a step ahead: without, the compiler waited for q,
// and with it for the tile just requested, in every step, and a step began with two trips to LDS.  Both: 4096 tokens x 4 heads of
// 128 39.3 -> 35.0 us, 4500 x 8 of 64 40 -> 38.  Two row tiles per work-group, a long and a short one, shared out over eight waves:
// 36 and slower elsewhere.
template <int D, int KG> struct NarrowLds {
  static constexpr int TILE = 32 * D * 2;
  static constexpr int WAVE_BYTES = 2 * TILE;               // K and V of a wave; at the end its fp32 partial [32][D]
  static constexpr int STATS = 2 * KG * 32 * 4;             // (m, l) of every wave
  static constexpr int bytes(int max_blk) { return KG * WAVE_BYTES + STATS + 16 + 6 * max_blk; }
};

template <typename T, int D, int KG, bool MERGE>
__global__ void __launch_bounds__(64 * KG, D <= 128 ? 2 : 1)
selattn_direct_narrow_kernel(DirectParams p) {
  typedef typename Elem<T>::vec8 vec8;
  typedef NarrowLds<D, KG> L;
  typedef TileLoads<T, D> Loads;
  constexpr int NKS = D / 16, NDT = D / 32, NT = 64 * KG, NLD = Loads::N;
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
  float* st_m = reinterpret_cast<float*>(smem + KG * L::WAVE_BYTES);   // [wave][row]
  float* st_l = st_m + KG * 32;
  int* info = reinterpret_cast<int*>(st_l + KG * 32);           // [0] list length, [1] a list names a block twice
  uint32_t* sel = reinterpret_cast<uint32_t*>(info + 4);        // [block]: bit i = query q_first + i
  uint16_t* list = reinterpret_cast<uint16_t*>(sel + p.max_blk);   // visited blocks

  const int h = blockIdx.x % p.hkv;
  DirectTile t_;
  if (!direct_tile(p.cu, p.batch, (int)p.n_tokens, p.g, 32, blockIdx.x / p.hkv, t_)) return;
  const int q0 = t_.q0, len = t_.len, rows = t_.n_q * p.g, row0 = t_.tile * 32, bks = p.bk_shift;
  const int q_first = div_group(row0, p.g, p.g_shift), q_last = div_group(min(rows, row0 + 32) - 1, p.g, p.g_shift);
  const int n_blk = min((q_last >> bks) + 1, (len + (1 << bks) - 1) >> bks);
  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6), col = lane & 31;

  AttnRows<T, D> r;
  r.scale_log2 = p.scale_log2;
  {
    const int row = min(row0 + col, rows - 1);
    r.qpos = div_group(row, p.g, p.g_shift);
    r.load_q(reinterpret_cast<const T*>(p.q) + (int64_t)(q0 + r.qpos) * p.q_sn + (int64_t)(h * p.g + row - r.qpos * p.g) * p.q_sh);
  }
  const int qoff = r.qpos - q_first;
  const Loads kl(p.k, p.k_sn, p.k_sh, q0, h, len), vl(p.v, p.v_sn, p.v_sh, q0, h, len);
  const uint32_t k_lds = lds_addr(smem + wv * L::WAVE_BYTES), v_lds = k_lds + L::TILE;

  // ---- which blocks, and which of the queries selected them ----
  const int32_t* ids = p.topk_idx + h * p.i_sh + (int64_t)(q0 + q_first) * p.i_sn;
  const int n_ids = (q_last - q_first + 1) * p.topk;
  constexpr int AHEAD = 512 / NT;   // entries per thread that are requested at once (32 lists of 16)
  int qo[AHEAD], id[AHEAD];
#pragma unroll
  for (int i = 0; i < AHEAD; ++i) {
    const int e = min(tid + i * NT, n_ids - 1);
    qo[i] = (uint32_t)e / (uint32_t)p.topk;
    id[i] = ids[qo[i] * p.i_sn + (e - qo[i] * p.topk)];
  }
  // The first keys of every wave are requested before it is known which blocks are visited: the first blocks of the
  // sequence, as where the union of the lists has no gap at its start.  4096 tokens x 4 heads 40.5 -> 39.3 us.  (The
  // compiler's waits for id[] below do not count these loads, which are younger, and so wait for most of them as well.)
  int guess = 32 * wv;
  if (guess + 32 <= len) {
    kl.issue(guess, k_lds);
    vl.issue(guess, v_lds);
  } else {
    guess = -1;
  }
  for (int b = tid; b < n_blk; b += NT) sel[b] = 0;
  if (tid < 2) info[tid] = 0;
  __syncthreads();
  auto visit = [&](int q, int b) {
    if (b < 0 || b >= n_blk || b > (q_first + q) >> bks) return;   // (a block behind the query's own holds no key it may see)
    if (atomicOr(&sel[b], 1u << q) >> q & 1) info[1] = 1;
  };
#pragma unroll
  for (int i = 0; i < AHEAD; ++i)
    if (tid + i * NT < n_ids) visit(qo[i], id[i]);
  for (int e = tid + AHEAD * NT; e < n_ids; e += NT) {
    const int q = (uint32_t)e / (uint32_t)p.topk;
    visit(q, ids[q * p.i_sn + (e - q * p.topk)]);
  }
  r.settle_q();
  __syncthreads();
  if (wv == 0) {   // the visited blocks, in order
    int at = 0;
    for (int b0 = 0; b0 < n_blk; b0 += WAVE) {
      const int b = b0 + lane;
      const bool any = b < n_blk && sel[b] != 0;
      const uint64_t m = __ballot(any);
      if (any) list[at + __popcll(m & ((1ull << lane) - 1))] = (uint16_t)b;
      at += __popcll(m);
    }
    if (lane == 0) info[0] = at;
  }
  __syncthreads();
  const bool twice = __builtin_amdgcn_readfirstlane(info[1]) != 0;
  const int upb_shift = bks - 5;   // log2 of the steps of 32 keys per block
  const int n_units = __builtin_amdgcn_readfirstlane(info[0]) << upb_shift;
  const int n_steps = (n_units - wv + KG - 1) / KG;   // of this wave
  const TileFrags<D> f;
  auto place = [&](int t) { return wv + KG * min(t, n_steps - 1); };   // in the list of steps
  auto key_of = [&](int u, int b) { return (b << bks) + (u & ((1 << upb_shift) - 1)) * 32; };

  auto attend = [&]() {
    r.clear();
    if (n_steps <= 0) {
      vm_wait<0>();
      return;
    }
    int b = __builtin_amdgcn_readfirstlane(list[place(0) >> upb_shift]), b1 = __builtin_amdgcn_readfirstlane(list[place(1) >> upb_shift]);
    int key = key_of(place(0), b);
    uint32_t mask = (uint32_t)__builtin_amdgcn_readfirstlane((int)sel[b]);
    if (key != guess) {
      vm_wait<0>();   // (what is on its way would land in what comes now)
      kl.issue(key, k_lds);
      vl.issue(key, v_lds);
    }
    for (int t = 0;; ++t) {
      const bool more = t + 1 < n_steps;
      const int key1 = key_of(place(t + 1), b1);
      vm_wait<NLD>();   // K of this step, not its V
      vec8 kf[NKS];
#pragma unroll
      for (int ks = 0; ks < NKS; ++ks) kf[ks] = load16<vec8>(lds_ptr<T>(k_lds + (f.k ^ (16u * ks))));
      // asked for here, looked at behind the products: the mask of the next step, the block of the one after
      const uint32_t mask1 = sel[b1], b2 = list[place(t + 2) >> upb_shift];
      lds_reads_done();
      if (more) kl.issue(key1, k_lds);
      f32x16 s;
#pragma unroll
      for (int i = 0; i < 16; ++i) s[i] = 0.f;
#pragma unroll
      for (int ks = 0; ks < NKS; ++ks) s = Elem<T>::mfma32(kf[ks], r.q[ks], s);
      const bool on = mask >> qoff & 1;
      if (__builtin_expect(key + 31 > q_first, 0)) r.causal(s, key);   // some row may see the keys partly
      r.raise(r.lane_max(s), on);
      const float ref = r.reference(on);
      float sum = 0.f;
      vec8 pk[2];
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const float pv = fast_exp2(s[i] * r.scale_log2 - ref);
        sum += pv;
        pk[i >> 3][i & 7] = (T)pv;
      }
      r.l += sum;   // the lane's own keys: the two lanes of a row are added behind the loop
      if (more) vm_wait<NLD>();   // V of this step, not K of the next
      else vm_wait<0>();
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int dt = 0; dt < NDT; ++dt) r.o[dt] = Elem<T>::mfma32(swizzled_tr_frag<T, D>(v_lds + (f.v ^ (64u * dt)), j), pk[j], r.o[dt]);
      lds_reads_done();
      if (!more) break;
      vl.issue(key1, v_lds);
      key = key1;
      mask = (uint32_t)__builtin_amdgcn_readfirstlane((int)mask1);
      b1 = __builtin_amdgcn_readfirstlane((int)b2);
    }
  };
  bool careful = twice;
  if (!careful) {
    attend();
    careful = __any(r.has_nan());
  }
  if (careful) {
    vm_wait<0>();
    r.clear();
    for (int t = 0; t < n_steps; ++t) {
      const int b = __builtin_amdgcn_readfirstlane(list[place(t) >> upb_shift]);
      r.step_carefully(kl, vl, f, k_lds, key_of(place(t), b), sel[b] >> qoff & 1, twice ? direct_times(p, h, q0 + r.qpos, b) : 1.f);
    }
  }
  r.l = sum32(r.l);

  // ---- merge of the waves ----
  r.park(reinterpret_cast<float*>(smem + wv * L::WAVE_BYTES), st_m + wv * 32, st_l + wv * 32);
  __syncthreads();
  constexpr int CPR = Loads::CPR;
  for (int wr = tid / CPR; wr < 32 && row0 + wr < rows; wr += NT / CPR)
    direct_store<T, D, MERGE, KG>(p, h, q0, row0 + wr, wr, tid % CPR, smem, L::WAVE_BYTES, st_m, st_l, 32);
}

// ---- wide: RT row tiles, KG key groups --------------------------------------------------------------------------------------
// With tiles of its own a wave brings 16 KB (head_dim 128) into LDS for 32 rows x 32 keys, 512 clocks of products: the L2 delivers
// about 50 bytes per clock and CU, so a full chip of such waves waits for tiles (5003 tokens x 32 heads, GQA 4, 250 us; without the
// loads 170).  Here RT row tiles share them, and a wave does not alternate between products and exponentials but always has both:
// 209 us, 1.0 PFLOP/s of the pairs it visits.  Two thirds of a SIMD's time are products then (timing-only builds: no LDS reads -9 %,
// no exponentials -2 %).  64 rows per wave at one wave per SIMD, with the same order of work: 273 us, since a single wave issues an
// instruction in four clocks at best; 64 rows per wave with q in LDS: 290.
template <int D, int KG, int RT> struct WideLds {
  static constexpr int WAVES = KG * RT;
  static constexpr int TILE = 32 * D * 2;
  static constexpr int WAVE_BYTES = 2 * TILE;               // a wave's part in the second pass and in the merge: its fp32 partial [32][D]
  static constexpr int GROUP_BYTES = 4 * TILE > RT * WAVE_BYTES ? 4 * TILE : RT * WAVE_BYTES;   // of a key group: two K and two V tiles
  static constexpr int STATS = 2 * WAVES * 32 * 4;          // (m, l) of every wave
  static constexpr int bytes(int max_blk) { return KG * GROUP_BYTES + STATS + 16 + (4 * RT + 2) * max_blk; }
};

template <typename T, int D, int KG, int RT, bool MERGE>
__global__ void __launch_bounds__(64 * KG * RT, D <= 128 ? 2 : 1)
selattn_direct_wide_kernel(DirectParams p) {
  typedef typename Elem<T>::vec8 vec8;
  typedef WideLds<D, KG, RT> L;
  typedef TileLoads<T, D> Loads;
  constexpr int ROWS = 32 * RT, NKS = D / 16, NDT = D / 32, NT = 64 * L::WAVES;
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
  float* st_m = reinterpret_cast<float*>(smem + KG * L::GROUP_BYTES);   // [wave][32]
  float* st_l = st_m + L::WAVES * 32;
  int* info = reinterpret_cast<int*>(st_l + L::WAVES * 32);     // [0] list length, [1] a list names a block twice, [2] second pass
  uint32_t* sel = reinterpret_cast<uint32_t*>(info + 4);        // [block][row tile]: bit i = the i-th query of the row tile
  uint16_t* list = reinterpret_cast<uint16_t*>(sel + RT * p.max_blk);   // visited blocks

  const int h = blockIdx.x % p.hkv;
  DirectTile t_;
  if (!direct_tile(p.cu, p.batch, (int)p.n_tokens, p.g, ROWS, blockIdx.x / p.hkv, t_)) return;
  const int q0 = t_.q0, len = t_.len, rows = t_.n_q * p.g, row0 = t_.tile * ROWS, bks = p.bk_shift;
  const int q_first = div_group(row0, p.g, p.g_shift), q_last = div_group(min(rows, row0 + ROWS) - 1, p.g, p.g_shift);
  const int n_blk = min((q_last >> bks) + 1, (len + (1 << bks) - 1) >> bks);
  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6), col = lane & 31;
  const int rt = wv % RT, kg = wv / RT;

  AttnRows<T, D> r;
  r.scale_log2 = p.scale_log2;
  {
    const int row = min(row0 + 32 * rt + col, rows - 1);
    r.qpos = div_group(row, p.g, p.g_shift);
    r.load_q(reinterpret_cast<const T*>(p.q) + (int64_t)(q0 + r.qpos) * p.q_sn + (int64_t)(h * p.g + row - r.qpos * p.g) * p.q_sh);
  }
  const int q_tile = div_group(min(row0 + 32 * rt, rows - 1), p.g, p.g_shift), qoff = r.qpos - q_tile;
  const Loads kl(p.k, p.k_sn, p.k_sh, q0, h, len), vl(p.v, p.v_sn, p.v_sh, q0, h, len);
  const uint32_t k_lds = lds_addr(smem + kg * L::GROUP_BYTES), v_lds = k_lds + 2 * L::TILE;
  // This wave's share of a K or V tile of its key group: even waves K, odd ones V, each half a tile where there are four.
  constexpr int PARTS = RT >= 4 && Loads::N >= 2 * Loads::NV ? 2 : 1;
  auto issue_k = [&](int key, int stage) {
    if ((rt & 1) == 0 && rt < 2 * PARTS) kl.template issue<PARTS>(key, k_lds + stage * L::TILE, rt >> 1);
  };
  auto issue_v = [&](int key, int stage) {
    if ((rt & 1) == 1 && rt < 2 * PARTS) vl.template issue<PARTS>(key, v_lds + stage * L::TILE, rt >> 1);
  };

  // ---- which blocks, and which of the queries selected them ----
  const int32_t* ids = p.topk_idx + h * p.i_sh + (int64_t)(q0 + q_first) * p.i_sn;
  const int n_ids = (q_last - q_first + 1) * p.topk;
  constexpr int AHEAD = 512 * RT / NT;   // entries per thread that are requested at once (32 lists of 16 for each row tile)
  int qo[AHEAD], id[AHEAD];
#pragma unroll
  for (int i = 0; i < AHEAD; ++i) {
    const int e = min(tid + i * NT, n_ids - 1);
    qo[i] = (uint32_t)e / (uint32_t)p.topk;
    id[i] = ids[qo[i] * p.i_sn + (e - qo[i] * p.topk)];
  }
  int guess = 32 * kg;   // as in the narrow kernel
  if (guess + 32 <= len) {
    issue_k(guess, 0);
    issue_v(guess, 0);
  } else {
    guess = -1;
  }
  for (int b = tid; b < RT * n_blk; b += NT) sel[b] = 0;
  if (tid < 3) info[tid] = 0;
  __syncthreads();
  auto visit = [&](int q, int b) {   // q: relative to q_first
    if (b < 0 || b >= n_blk || b > (q_first + q) >> bks) return;   // (a block behind the query's own holds no key it may see)
    // the rows of a query may lie in several row tiles
    const int r_lo = max((q_first + q) * p.g - row0, 0), r_hi = min((q_first + q) * p.g + p.g - row0, ROWS) - 1;
    for (int x = r_lo >> 5; x <= r_hi >> 5; ++x) {
      const int off = q_first + q - div_group(row0 + 32 * x, p.g, p.g_shift);
      if (atomicOr(&sel[RT * b + x], 1u << off) >> off & 1) info[1] = 1;
    }
  };
#pragma unroll
  for (int i = 0; i < AHEAD; ++i)
    if (tid + i * NT < n_ids) visit(qo[i], id[i]);
  for (int e = tid + AHEAD * NT; e < n_ids; e += NT) {
    const int q = (uint32_t)e / (uint32_t)p.topk;
    visit(q, ids[q * p.i_sn + (e - q * p.topk)]);
  }
  r.settle_q();
  __syncthreads();
  if (wv == 0) {   // the visited blocks, in order
    int at = 0;
    for (int b0 = 0; b0 < n_blk; b0 += WAVE) {
      const int b = b0 + lane;
      uint32_t any = 0;
      if (b < n_blk)
#pragma unroll
        for (int x = 0; x < RT; ++x) any |= sel[RT * b + x];
      const uint64_t m = __ballot(any != 0);
      if (any) list[at + __popcll(m & ((1ull << lane) - 1))] = (uint16_t)b;
      at += __popcll(m);
    }
    if (lane == 0) info[0] = at;
  }
  __syncthreads();
  const bool twice = __builtin_amdgcn_readfirstlane(info[1]) != 0;
  const int upb_shift = bks - 5;   // log2 of the steps of 32 keys per block
  const int n_units = __builtin_amdgcn_readfirstlane(info[0]) << upb_shift;
  const int n_steps = (n_units + KG - 1) / KG;
  struct Unit {
    int key;         // position of its first key
    uint32_t mask;   // queries of the row tile that selected its block
  };
  auto unit = [&](int t) {   // (the last steps of the key groups behind the end: some tile, selected by nobody)
    const int u = kg + KG * t, v = min(u, n_units - 1);
    const int b = __builtin_amdgcn_readfirstlane(list[v >> upb_shift]);
    Unit x;
    x.key = (b << bks) + (v & ((1 << upb_shift) - 1)) * 32;
    x.mask = (uint32_t)__builtin_amdgcn_readfirstlane((int)sel[RT * b + rt]);
    if (u >= n_units) x.mask = 0;
    return x;
  };
  const TileFrags<D> f;

  auto attend = [&]() {
    r.clear();
    if (n_steps <= 0) {
      vm_wait<0>();
      return;
    }
    Unit cur = unit(0), nx1 = unit(1);
    if (cur.key != guess) {
      vm_wait<0>();   // (what is on its way would land in what comes now)
      issue_k(cur.key, 0);
      issue_v(cur.key, 0);
    }
    issue_k(nx1.key, 1);
    int key2 = unit(2).key, b2 = key2 >> bks;
    vec8 pk[2];
    auto step = [&](f32x16& s, f32x16& next, int t) {   // scores of this step in s, those of the next one into `next`
      const int odd = t & 1;
      tiles_arrived();   // K of the next step, V of this one
      issue_k(key2, odd);
      issue_v(nx1.key, odd ^ 1);
      // asked for here, looked at behind the products: the mask of step t + 2, the block of step t + 3
      const uint32_t mask2 = sel[RT * b2 + rt], u3 = min(kg + KG * (t + 3), n_units - 1), b3 = list[u3 >> upb_shift];
      r.template scores<true>(next, s, r.reference(cur.mask >> qoff & 1), pk, k_lds + (odd ^ 1) * L::TILE, f);
      if (__builtin_expect(nx1.key + 31 > q_first, 0)) r.causal(next, nx1.key);   // some row may see the keys partly
      r.raise(r.values(next, pk, v_lds + odd * L::TILE, f), nx1.mask >> qoff & 1);
      cur = nx1;
      nx1.key = key2;
      nx1.mask = kg + KG * (t + 2) < n_units ? (uint32_t)__builtin_amdgcn_readfirstlane((int)mask2) : 0u;
      b2 = __builtin_amdgcn_readfirstlane((int)b3);
      key2 = (b2 << bks) + (u3 & ((1 << upb_shift) - 1)) * 32;
    };
    f32x16 sa, sb;
    tiles_arrived();
    r.template scores<false>(sa, sb, 0.f, pk, k_lds, f);
    if (cur.key + 31 > q_first) r.causal(sa, cur.key);
    r.raise(r.lane_max(sa), cur.mask >> qoff & 1);
    for (int t = 0;;) {
      step(sa, sb, t);
      if (++t >= n_steps) break;
      step(sb, sa, t);
      if (++t >= n_steps) break;
    }
    vm_wait<0>();
  };
  bool careful = twice;
  if (!careful) {
    attend();
    if (__any(r.has_nan())) info[2] = 1;
    __syncthreads();   // (the last reads from the tiles, too)
    careful = __builtin_amdgcn_readfirstlane(info[2]) != 0;
  }
  unsigned char* own = smem + kg * L::GROUP_BYTES + rt * L::WAVE_BYTES;
  if (careful) {
    vm_wait<0>();
    __syncthreads();
    r.clear();
    for (int t = 0; t < n_steps; ++t) {
      const Unit u = unit(t);
      if (u.mask != 0)
        r.step_carefully(kl, vl, f, lds_addr(own), u.key, u.mask >> qoff & 1, twice ? direct_times(p, h, q0 + r.qpos, u.key >> bks) : 1.f);
    }
  }
  r.l = sum32(r.l);

  // ---- merge of the key groups ----
  r.park(reinterpret_cast<float*>(own), st_m + wv * 32, st_l + wv * 32);
  __syncthreads();
  constexpr int CPR = Loads::CPR;
  for (int wr = tid / CPR; wr < ROWS && row0 + wr < rows; wr += NT / CPR) {
    const int x = wr >> 5;
    direct_store<T, D, MERGE, KG>(p, h, q0, row0 + wr, wr & 31, tid % CPR, smem + x * L::WAVE_BYTES, L::GROUP_BYTES, st_m + x * 32,
                                  st_l + x * 32, RT * 32);
  }
}

template <typename T, int D, int KG, bool MERGE> static int launch_direct_narrow(const DirectParams& p, hipStream_t stream) {
  static LdsAllowed allowed;
  typedef NarrowLds<D, KG> L;
  if (int rc = allow_lds(allowed, (const void*)selattn_direct_narrow_kernel<T, D, KG, MERGE>, L::bytes(DIR_MAX_BLOCKS))) return rc;
  const int64_t tiles = p.n_tokens * p.g / 32 + p.batch + 1;
  ProfScope ps_("selattn_direct_fwd", stream);
  selattn_direct_narrow_kernel<T, D, KG, MERGE><<<(unsigned)(tiles * p.hkv), 64 * KG, L::bytes(p.max_blk), stream>>>(p);
  return 0;
}
template <typename T, int D, int KG, int RT, bool MERGE> static int launch_direct_wide(const DirectParams& p, hipStream_t stream) {
  static LdsAllowed allowed;
  typedef WideLds<D, KG, RT> L;
  if (int rc = allow_lds(allowed, (const void*)selattn_direct_wide_kernel<T, D, KG, RT, MERGE>, L::bytes(DIR_MAX_BLOCKS))) return rc;
  const int64_t tiles = p.n_tokens * p.g / (32 * RT) + p.batch + 1;
  ProfScope ps_("selattn_direct_fwd", stream);
  selattn_direct_wide_kernel<T, D, KG, RT, MERGE><<<(unsigned)(tiles * p.hkv), 64 * KG * RT, L::bytes(p.max_blk), stream>>>(p);
  return 0;
}
// What the kernels take, in us on one chip: a part that grows with rows x keys, a chain of steps through the longest sequence, and
// what does not depend on the size.  Fitted to 3 x 30 sizes (lists of 16 blocks of 64; head_dim 256: 8 of 128; one sequence).
// narrow / wide 2 x 2 / wide 1 x 4 in us, head_dim 128, tokens x heads: 1500 x 4 15.9 / 23.7 / 36.6, 3000 x 4 28 / 40 / 62,
// 1500 x 32 44 / 40 / 41, 3000 x 16 65 / 56 / 66, 3000 x 32 127 / 100 / 97, 5000 x 32 312 / 245 / 222, 8000 x 32 757 / 576 / 503; 64:
// 5000 x 32 165 / 139 / 136; 256: 3000 x 4 48 / 73 / 109, 3000 x 32 314 / 249 / 210.
enum DirectForm { DIRECT_NARROW, DIRECT_WIDE_2X2, DIRECT_WIDE_1X4, DIRECT_FORMS };
static double direct_us(DirectForm form, int d, double rows, double len) {   // rows: of 128 dims
  struct Fit { double per_us, step, fixed; };
  static constexpr Fit fits[3][DIRECT_FORMS] = {{{2.55e6, 0.0036, 6}, {3.3e6, 0.0062, 8.5}, {3.75e6, 0.0145, 7}},
                                                {{2.65e6, 0.0055, 6}, {3.5e6, 0.0095, 9}, {4.3e6, 0.018, 7}},
                                                {{2.2e6, 0.01, 10}, {2.75e6, 0.021, 12}, {3.8e6, 0.0325, 12}}};
  const Fit& f = fits[d <= 64 ? 0 : d <= 128 ? 1 : 2][form];
  return std::hypot(rows * len / f.per_us, f.step * len) + f.fixed;
}
static DirectForm direct_form(int d, double rows, double len) {
  DirectForm best = DIRECT_NARROW;
  for (int i = 1; i < DIRECT_FORMS; ++i)
    if (direct_us((DirectForm)i, d, rows, len) < direct_us(best, d, rows, len)) best = (DirectForm)i;
  return best;
}

template <typename T, int D, bool MERGE> static int launch_direct_fwd(const DirectParams& p, int64_t max_len, hipStream_t stream) {
  switch (direct_form(D, (double)p.n_tokens * p.hkv * p.g * D / 128, (double)max_len)) {
    case DIRECT_WIDE_2X2: return launch_direct_wide<T, D, 2, 2, MERGE>(p, stream);
    case DIRECT_WIDE_1X4: return launch_direct_wide<T, D, 1, 4, MERGE>(p, stream);
    default: return launch_direct_narrow<T, D, 4, MERGE>(p, stream);
  }
}
template <typename T, bool MERGE> static int dispatch_direct_fwd(int d, const DirectParams& p, int64_t max_len, hipStream_t stream) {
  if (d == 128) return launch_direct_fwd<T, 128, MERGE>(p, max_len, stream);
  if (d == 64) return launch_direct_fwd<T, 64, MERGE>(p, max_len, stream);
  return launch_direct_fwd<T, 256, MERGE>(p, max_len, stream);
}

// Whether the forward of `n` tokens in sequences of at most `max_len` takes this path.  Both sides in us on one chip: these
// kernels visit up to half of a sequence for every row; the block-major launches write and read a partial row for every (row,
// block) and work on topk * block keys per row, behind a fixed part and, unless the caller builds it all the same (training), the
// index.  index + block-major / direct in us, blocks of 64 and 16 to a list unless said otherwise, head_dim 128: 3000 x 4 13 + 40 /
// 28, 5000 x 4 17 + 54 / 46, 8000 x 4 23 + 77 / 100, 5000 x 32 27 + 288 / 222, 8000 x 32 33 + 460 / 503, 5000 x 32, 16 blocks of
// 32, 19 + 260 / 199, 8 of 64 14 + 155 / 199, 8 of 128 13 + 196 / 208; 64: 8000 x 4 23 + 49 / 55, 5000 x 32 27 + 171 / 136, 16
// blocks of 32 19 + 148 / 121, 8 of 64 14 + 88 / 119; 256: 3000 x 32 13 + 361 / 203, 16 blocks of 32 14 + 321 / 200, 8 of 64 11 +
// 219 / 202, 8 of 128 12 + 243 / 210; 5000 x 4 17 + 114 / 105, 8 of 64 13 + 78 / 102; lists that do not load four at a time take the
// index longer: 6 of 64, 3000 x 4 of 256, 17 + 51 / 53.  The block-major side is fitted to 4000 measured calls (one in ten of them more
// than 17 to 29 % off), with 2 us for every gap between its launches.  Over 4700 calls the choice takes 1.005 (training) and 1.010
// (inference) of the better form's time.
bool selattn_direct_preferred(int64_t n, int64_t max_len, int hq, int d, int topk, int bk, bool index_needed) {
  if (!(d == 64 || d == 128 || d == 256) || !(bk == 32 || bk == 64 || bk == 128) || topk > 4096 ||
      max_len > (int64_t)bk * DIR_MAX_BLOCKS)
    return false;
  const double rows = (double)n * hq * d / 128, len = (double)max_len;
  const double keys = std::min<double>((double)topk * bk, len);
  struct Fit { double fixed, row, block, key, key_128; };   // per row of 128 dims; key_128: what a key of a block of 128 adds
  static constexpr Fit fits[3] = {{18.4, 1.3e-4, 8.4e-5, 2.7e-7, 6.5e-7}, {19.8, 1.8e-4, 7.7e-5, 2.6e-7, 1.5e-7}, {23.8, 3.2e-4, 8.05e-5, 2.55e-7, 0}};
  const Fit& f = fits[d <= 64 ? 0 : d <= 128 ? 1 : 2];
  const double blocks = std::min<double>(topk, std::ceil(len / bk));
  const double block_major = f.fixed + rows * (f.row + blocks * f.block + keys * (f.key + (bk == 128 ? f.key_128 : 0)));
  const double index = index_needed ? 0 : 13.3 + (topk % 4 ? 4e-4 : 1.2e-4) * (double)n * topk;
  return direct_us(direct_form(d, rows, len), d, rows, len) <= block_major + index;
}

int selattn_direct_fwd(const void* q, const void* k, const void* v, int32_t dtype, int64_t q_stride_n, int64_t q_stride_h,
                       int64_t k_stride_n, int64_t k_stride_h, int64_t v_stride_n, int64_t v_stride_h, const int32_t* topk_idx,
                       int64_t idx_stride_h, int64_t idx_stride_n, const int32_t* cu_seqlens, int32_t batch,
                       int64_t total_tokens, int64_t max_len, int32_t num_q_heads, int32_t num_kv_heads, int32_t head_dim, int32_t topk,
                       int32_t block_size, float softmax_scale, void* o, int64_t o_stride_n, int64_t o_stride_h, float* lse,
                       const MergeEpilogue& merge, hipStream_t stream) {
  FSA_CHECK_ARG(q && k && v && topk_idx && cu_seqlens && ((o && lse) || merge.out), "fsa_selattn_direct_fwd: null pointer");
  FSA_CHECK_ARG(dtype == FSA_BF16 || dtype == FSA_FP16, "fsa_selattn_direct_fwd: dtype must be bf16 or fp16");
  FSA_CHECK_ARG(num_kv_heads >= 1 && num_q_heads % num_kv_heads == 0,
                "fsa_selattn_direct_fwd: num_q_heads must be a multiple of num_kv_heads");
  FSA_CHECK_ARG(batch >= 1 && total_tokens >= 1 && max_len >= 1 && max_len <= total_tokens && topk >= 1 && topk <= 4096,
                "fsa_selattn_direct_fwd: bad sizes");
  FSA_CHECK_ARG((q_stride_n | q_stride_h | k_stride_n | k_stride_h | v_stride_n | v_stride_h | o_stride_n | o_stride_h) % 8 == 0,
                "fsa_selattn_direct_fwd: strides must be multiples of 8 elements (16-byte rows)");
  FSA_CHECK_ARG(((uintptr_t)k | (uintptr_t)v) % 16 == 0, "fsa_selattn_direct_fwd: k and v must be 16-byte aligned");
  FSA_CHECK_ARG(k_stride_n >= head_dim && v_stride_n >= head_dim && total_tokens * 2 * k_stride_n < ((int64_t)1 << 31) &&
                    total_tokens * 2 * v_stride_n < ((int64_t)1 << 31), "fsa_selattn_direct_fwd: k / v strides out of range");
  FSA_CHECK_ARG(block_size >= 1 && max_len <= (int64_t)block_size * DIR_MAX_BLOCKS && total_tokens * num_q_heads < ((int64_t)1 << 31),
                "fsa_selattn_direct_fwd: too many tokens");
  if ((head_dim != 64 && head_dim != 128 && head_dim != 256) || (block_size != 32 && block_size != 64 && block_size != 128)) {
    set_error("selected attention (direct): head_dim=%d with block_size=%d is not supported", head_dim, block_size);
    return FSA_ERR_UNSUPPORTED;
  }
  DirectParams p = {};
  p.q = q; p.k = k; p.v = v;
  p.q_sn = q_stride_n; p.q_sh = q_stride_h;
  p.k_sn = k_stride_n; p.k_sh = k_stride_h;
  p.v_sn = v_stride_n; p.v_sh = v_stride_h;
  p.o_sn = o_stride_n; p.o_sh = o_stride_h;
  p.topk_idx = topk_idx; p.i_sh = idx_stride_h; p.i_sn = idx_stride_n;
  p.cu = cu_seqlens; p.batch = batch; p.hkv = num_kv_heads; p.g = num_q_heads / num_kv_heads; p.g_shift = group_shift(p.g);
  p.bk_shift = block_size == 32 ? 5 : block_size == 64 ? 6 : 7;
  p.topk = topk; p.max_blk = (int)((max_len + block_size - 1) / block_size); p.n_tokens = total_tokens;
  p.scale_log2 = softmax_scale * LOG2E;
  p.o = o; p.lse = lse; p.merge = merge;
  const int rc = merge.out ? (dtype == FSA_BF16 ? dispatch_direct_fwd<__bf16, true>(head_dim, p, max_len, stream)
                                                : dispatch_direct_fwd<_Float16, true>(head_dim, p, max_len, stream))
                           : (dtype == FSA_BF16 ? dispatch_direct_fwd<__bf16, false>(head_dim, p, max_len, stream)
                                                : dispatch_direct_fwd<_Float16, false>(head_dim, p, max_len, stream));
  if (rc) return rc;
  FSA_CHECK_LAUNCH("fsa_selattn_direct_fwd");
  return 0;
}

}  // namespace fsa

using namespace fsa;

extern "C" int fsa_selattn_direct_fwd(const void* q, const void* k, const void* v, int32_t dtype, int64_t q_stride_n,
                                      int64_t q_stride_h, int64_t k_stride_n, int64_t k_stride_h, int64_t v_stride_n,
                                      int64_t v_stride_h, const int32_t* topk_idx, int64_t idx_stride_h, int64_t idx_stride_n,
                                      const int32_t* cu_seqlens, int32_t batch, int64_t total_tokens, int64_t max_len,
                                      int32_t num_q_heads, int32_t num_kv_heads, int32_t head_dim, int32_t topk, int32_t block_size,
                                      float softmax_scale, void* o, int64_t o_stride_n, int64_t o_stride_h, float* lse,
                                      void* stream) {
  return fsa::selattn_direct_fwd(q, k, v, dtype, q_stride_n, q_stride_h, k_stride_n, k_stride_h, v_stride_n, v_stride_h, topk_idx,
                                 idx_stride_h, idx_stride_n, cu_seqlens, batch, total_tokens, max_len, num_q_heads, num_kv_heads,
                                 head_dim, topk, block_size, softmax_scale, o, o_stride_n, o_stride_h, lse, MergeEpilogue(),
                                 (hipStream_t)stream);
}

extern "C" int fsa_selattn_direct_preferred(int64_t total_tokens, int64_t max_len, int32_t num_q_heads, int32_t head_dim,
                                            int32_t topk, int32_t block_size, int32_t index_needed) {
  FSA_CHECK_ARG(total_tokens >= 1 && max_len >= 1 && num_q_heads >= 1 && topk >= 1, "fsa_selattn_direct_preferred: bad sizes");
  return selattn_direct_preferred(total_tokens, max_len, num_q_heads, head_dim, topk, block_size, index_needed != 0);
}
