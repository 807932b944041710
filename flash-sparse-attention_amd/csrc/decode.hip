// One-step decode for gfx950: one new query per request against its caches.
//
//   decode_attn_kernel (compressed mode): the g heads of a kv group attend every
//       visible compressed key of the request; the raw scores of one "scoring"
//       head are kept for the block selection.
//   decode_attn_kernel (selected mode): the g heads attend the cached keys of
//       the T selected blocks.
//   decode_topk_kernel: probabilities -> re-binned block scores -> top-k ids.
//
// Both attention modes are HBM-bound streams of K/V rows (g rows of queries
// only).  The 32-key tiles of all (request, kv head) pairs form one sequence,
// and a persistent grid of single-wave work-groups - as many as are resident
// on the chip at once - cuts it into equal contiguous shares: no work-group is
// dispatched while the kernel runs, every wave streams for the whole launch
// and always has the rows of its next tile in flight while it computes the
// current one.  The rows of a tile arrive row-coalesced (16 B per lane, whole
// 2*D-byte rows per instruction) and pass through a wave-private LDS tile: K
// is read back as 16x16x32 MFMA operands, V transposed.  A wave writes one
// fp32 partial (m, l, O) per pair it touches; a small merge kernel combines
// the partials of a pair in a fixed order.  Where there are few tiles, a pair
// has a number of work-groups of its own and the last of them merges, or one
// work-group, whose waves meet in LDS (dec_launch).  The query heads occupy the first
// g of the 16 MFMA columns; column g carries the scoring head.
//
// Semantics: fsa_preview/ops/compressed_attention_decode.py:361-490 (attention),
// :494-592 (scores), :284-357 (transform), :203-205 (top-k);
// fsa_preview/ops/selected_attention_decode.py:8-42.
#include "fsa_common.h"

#include <algorithm>
#include <atomic>
#include <mutex>
#include <type_traits>

namespace fsa {

constexpr int DEC_MODE_COMPRESSED = 0;
constexpr int DEC_MODE_SELECTED = 1;
constexpr int DEC_TK = 32;            // keys per wave tile
constexpr int DEC_MAX_WAVES = 4096;   // upper bound of the persistent grid (the workspace is sized for it)
// resident waves per SIMD the register budget is set for (head_dim 256 stages twice the rows per tile)
template <int D> struct DecOcc {
  static constexpr int WAVES_PER_SIMD = D >= 256 ? 1 : 2;
  static constexpr int WG_WAVES = 2;  // waves per work-group at most
};

typedef float f32x2 __attribute__((ext_vector_type(2)));

struct DecParams {
  const void* q;   // [B, Hq, D]
  const void* k;   // [total, Hkv, D]
  const void* v;
  int64_t q_sb, q_sh, k_sn, k_sh, v_sn, v_sh;
  const int32_t* cu_k;      // [B+1] rows of k / v per request
  const int32_t* pos;       // compressed mode: position of the query
  const int32_t* topk_idx;  // selected mode: [Hkv, B, T]
  const int32_t* seqlens;   // selected mode, optional: [B] valid rows of each request's slot (null: the whole slot)
  int batch, hq, hkv, g, topk, block_size, kernel_size, kernel_stride;
  // One launch covers the heads [head0, head0 + g) of every GQA group of gq heads (the 16 columns of the MFMA tile
  // hold at most 16 heads): groups of more heads are served by several launches over the same workspace.
  int gq, head0;
  int score_col;            // compressed mode with raw_score: the column whose unscaled scores are kept
  float scale_log2;
  void* o;                  // [B, Hq, D] contiguous
  float* lse;               // [Hq, B]
  float* raw_score;         // compressed mode, optional: [Hkv, B, raw_ld] unscaled q.k of the scoring head
  int64_t raw_ld;
  int score_head_as_written;  // 0: first head of the group, 1: q-head with the kv head's own index
  int max_keys;             // compressed mode: host upper bound of the visible keys of a request (more are ignored)
  // Layer form (one request, caches stored un-rotated and without the new token).  Compressed mode: "request" 0 is the
  // compressed cache, 1 the window over the raw cache; selected mode: request 0 is the raw cache.
  struct Source {
    const void *k, *v;            // rows of the cache
    const void *k_new, *v_new;    // [hkv, D]: row number n_cache, kept apart from the cache
    int64_t k_sn, k_sh, v_sn, v_sh;
    int n_cache, n_keys;          // rows of the cache, visible keys (n_cache or n_cache + 1)
    int pos0, pos_step;           // key row r is rotated for position pos0 + r * pos_step
  } src[2];
  const float* inv_freq;    // [D/2]
  float rope_scale;
  int n_groups;             // groups of hkv waves that share the tile sequence
  float* part;              // [hkv][n_groups + batch][g][4 + D]: base-2 scaled max, sum, 2 unused, unnormalised O
                            // (layer form: [hkv][chunks[0] + chunks[1]][g][4 + D])
                            // (chunked form: [batch][hkv][chunks[0]][g][4 + D])
  int chunks[2];            // layer form: work-groups per kv head of source 0 and 1; chunked form: [0] per (request, kv head)
  int* arrived;             // layer form: [2][hkv] work-groups of (source, kv head) that have left their partial; zero between calls
  uint64_t* stamps;         // chunked form: [batch][hkv][chunks[0]], `call` where the partial is there
  uint64_t call;            // no other call's number
  int32_t* tile_prefix;     // [B+1]: tiles (of one kv head) of the requests before b; batches of more than 64 requests
};

// Loads and stores of what a work-group hands to another one of the same launch: as atomics of the device's scope they go past
// the L2 copies of the XCDs, so that neither side has to write back or invalidate a cache (1.7 us a launch).  SHARED false: plain.
// The hand-over has no release and no acquire, whose cost that is.  It rests on how the chip orders these accesses: a wave's
// s_waitcnt vmcnt(0) covers its stores until they are where all XCDs look (device scope: behind the L2s); a barrier collects
// the waves; only then is the counter or the stamp touched, by an access of the same scope; and what the last work-group loads, it
// loads behind that, past its own L2, in program order that neither the compiler (atomics, volatile statements between them)
// nor the wave (the loads wait for the answer through a branch and a barrier) turns round.  Nobody waits for anybody, so a late
// work-group costs nothing but its own time.  What plain stores leave, o_cmp, o_win and a counter set back to zero, is read by
// later launches only.
template <bool SHARED, typename V> __device__ __forceinline__ V dec_load(const float* p) {
  if constexpr (!SHARED) {
    return *reinterpret_cast<const V*>(p);
  } else if constexpr (sizeof(V) == 4) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  } else {
    typedef uint64_t words __attribute__((ext_vector_type(sizeof(V) / 8)));
    words w;
#pragma unroll
    for (int i = 0; i < (int)(sizeof(V) / 8); ++i)
      w[i] = __hip_atomic_load(reinterpret_cast<const uint64_t*>(p) + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return __builtin_bit_cast(V, w);
  }
}
template <bool SHARED> __device__ __forceinline__ void dec_store(float* p, f32x4 v) {
  if constexpr (!SHARED) {
    *reinterpret_cast<f32x4*>(p) = v;
  } else {
    typedef uint64_t words __attribute__((ext_vector_type(2)));
    const words w = __builtin_bit_cast(words, v);
#pragma unroll
    for (int i = 0; i < 2; ++i)
      __hip_atomic_store(reinterpret_cast<uint64_t*>(p) + i, w[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

template <int D> struct DecLds {
  static constexpr int VS = D + 8;
  static constexpr int BYTES = DEC_TK * VS * 2;  // one wave's tile
};

// number of 32-key tiles of request b per kv head (and, in compressed mode, its visible keys)
template <int MODE>
__device__ __forceinline__ int dec_tiles(const DecParams& p, int b, int len, int& n_keys, int& tpb) {
  n_keys = 0;
  tpb = 1;
  if (MODE == DEC_MODE_COMPRESSED) {
    const int qp = p.pos[b];
    n_keys = qp >= p.kernel_size - 1 ? min(len, (qp - p.kernel_size + 1) / p.kernel_stride + 1) : 0;
    n_keys = min(n_keys, p.max_keys);
    return (n_keys + DEC_TK - 1) / DEC_TK;
  }
  tpb = (p.block_size + DEC_TK - 1) / DEC_TK;
  return p.topk * tpb;
}

__device__ __forceinline__ int wave_inclusive_sum(int x) {
  const int lane = threadIdx.x & (WAVE - 1);
#pragma unroll
  for (int o = 1; o < WAVE; o <<= 1) {
    const int y = __shfl_up(x, o, WAVE);
    if (lane >= o) x += y;
  }
  return x;
}

// tile_prefix[b] = tiles (of one kv head) of the requests before b: batches of more than 64 requests only (one wave)
__global__ void __launch_bounds__(WAVE)
decode_plan_kernel(DecParams p) {
  const int lane = threadIdx.x;
  int carry = 0;
  for (int b0 = 0; b0 < p.batch; b0 += WAVE) {
    const int b = b0 + lane;
    int nt = 0;
    if (b < p.batch) {
      int n_keys, tpb;
      nt = dec_tiles<DEC_MODE_COMPRESSED>(p, b, p.cu_k[b + 1] - p.cu_k[b], n_keys, tpb);
    }
    const int incl = wave_inclusive_sum(nt);
    if (b < p.batch) p.tile_prefix[b] = carry + incl - nt;
    carry += __shfl(incl, WAVE - 1, WAVE);
  }
  if (lane == 0) p.tile_prefix[p.batch] = carry;
}

// The tile sequence of one kv head: the tiles of all requests, one after the other.  Selected mode: every request has
// topk x tiles-per-block tiles, the prefix is a product.  Compressed mode: up to 64 requests are scanned by every wave
// itself (lane b holds request b; a microsecond inside the kernel against a launch of its own), larger batches read
// the prefix that decode_plan_kernel wrote.
template <int MODE> struct DecSeq {
  int per_req = 0, incl = 0, nt = 0, total = 0;
  bool scanned = false;
  __device__ __forceinline__ void init(const DecParams& p) {
    if (MODE == DEC_MODE_SELECTED) {
      per_req = p.topk * ((p.block_size + DEC_TK - 1) / DEC_TK);
      total = p.batch * per_req;
      return;
    }
    scanned = p.batch <= WAVE;
    if (scanned) {
      const int lane = threadIdx.x & (WAVE - 1);
      if (lane < p.batch) {
        int n_keys, tpb;
        nt = dec_tiles<MODE>(p, lane, p.cu_k[lane + 1] - p.cu_k[lane], n_keys, tpb);
      }
      incl = wave_inclusive_sum(nt);
      total = __builtin_amdgcn_readlane(incl, WAVE - 1);
    } else {
      total = p.tile_prefix[p.batch];
    }
  }
  __device__ __forceinline__ int prefix(const DecParams& p, int b) const {   // b uniform
    if (MODE == DEC_MODE_SELECTED) return b * per_req;
    return scanned ? __builtin_amdgcn_readlane(incl - nt, b) : p.tile_prefix[b];
  }
  __device__ __forceinline__ int request_of(const DecParams& p, int x) const {  // x < total
    if (MODE == DEC_MODE_SELECTED) return x / per_req;
    return scanned ? __ffsll((unsigned long long)__ballot(incl > x)) - 1 : upper_seg(p.tile_prefix, p.batch, x);
  }
};

// share of the tile sequence per group of hkv waves for n_groups of them
__device__ __forceinline__ int dec_share(int total, int n_groups) { return max(1, (total + n_groups - 1) / n_groups); }

// Stores four elements of a merged row, and its lse.
template <typename T, int D>
__device__ __forceinline__ void dec_emit(const DecParams& p, int b, int h, int col, int lr, f32x4 o, float lse) {
  const int hq_i = h * p.gq + p.head0 + col;
  typename Elem<T>::vec4 x;
#pragma unroll
  for (int i = 0; i < 4; ++i) x[i] = (T)o[i];
  store8(reinterpret_cast<T*>(p.o) + ((int64_t)b * p.hq + hq_i) * D + lr * 4, x);
  if (lr == 0) p.lse[(int64_t)hq_i * p.batch + b] = lse;
}

// cos / sin of x radians, |x| < 2^18: the turns are formed with the rounding error of the product and the low part of
// 1 / (2 pi), so that the hardware instructions (which take turns) see an argument good to 2^-24.  No contraction: with
// t - rint(t) fused to x * HI - rint(t) the rounding error of t would be added twice, 6e-3 radians at x = 1e5.
__device__ __forceinline__ void sincos_turns(float x, float& sn, float& cs) {
#pragma clang fp contract(off)
  constexpr float HI = 0.15915494f, LO = 6.4206382e-9f;   // HI + LO = 1 / (2 pi)
  const float t = x * HI;
  const float e = __builtin_fmaf(x, HI, -t) + x * LO;
  const float f = (t - rintf(t)) + e;
  sn = __builtin_amdgcn_sinf(f);
  cs = __builtin_amdgcn_cosf(f);
}

// Wave = (group of tiles, kv head): the waves of a group read the same cache rows, one kv head each, at about the same
// time, so that a row (all kv heads, contiguous in memory) is fetched whole instead of in hkv visits of 2 D bytes.
// ONE > 0: a work-group of ONE waves serves one (request, kv head), its waves sharing the tiles and merging their partials
// in LDS; no partial goes through memory and no merge kernel follows.
// CHUNKED: as ONE, but a (request, kv head), or in the LAYER form a (source, kv head), has p.chunks work-groups, each of which
// leaves the partial of its tiles.
template <typename T, int D, int MODE, bool LAYER, int ONE, bool CHUNKED = LAYER>
__device__ __forceinline__ void decode_attn_body(const DecParams& p) {
  typedef typename Elem<T>::vec8 vec8;
  constexpr int VS = DecLds<D>::VS;
  constexpr int NS = D / 32, NDT = D / 16, VCH = DEC_TK * (D / 8) / 64, PS = D + 4;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  T* Vs = reinterpret_cast<T*>(smem + (threadIdx.x / WAVE) * DecLds<D>::BYTES);
  const int lane = threadIdx.x & (WAVE - 1), l16 = lane & 15, kg = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane((int)(blockIdx.x * (blockDim.x / WAVE) + threadIdx.x / WAVE));
  int grp = ONE ? blockIdx.x / p.hkv : w / p.hkv;   // ONE: the request; LAYER: the chunk, from here on of its source
  const int h = (ONE ? blockIdx.x : w) - grp * p.hkv;
  static_assert(!CHUNKED || ONE, "chunks are work-groups");
  // LAYER: the place among the chunks of both sources, then in its source; CHUNKED: the request, the chunk of it
  int chunk = grp;
  const int source = LAYER && grp >= p.chunks[0];
  if (LAYER) {
    grp -= source ? p.chunks[0] : 0;
  } else if (CHUNKED) {
    grp = (uint32_t)grp / (uint32_t)p.chunks[0];
    chunk -= grp * p.chunks[0];
  }
  DecSeq<MODE> seq;
  int x_lo = 0, x_hi = 0;
  if constexpr (!ONE) {
    if (grp >= p.n_groups) return;
    seq.init(p);
    const int per = dec_share(seq.total, p.n_groups);
    x_lo = grp * per;
    x_hi = min(seq.total, x_lo + per);
    if (x_lo >= x_hi) return;
  }

  // position in the tile sequence: request (with its sizes), tile of the request
  struct Req { int b, k0, len, n_keys, tpb, nt, ids; };  // ids: lane t holds the t-th selected block
  auto load_req = [&](Req& r, int b) {
    r.b = b;
    if constexpr (LAYER) {
      const DecParams::Source& c = MODE == DEC_MODE_COMPRESSED && b == 1 ? p.src[1] : p.src[0];
      r.k0 = 0;
      r.len = c.n_keys;
      r.n_keys = c.n_keys;
      r.tpb = MODE == DEC_MODE_SELECTED ? (p.block_size + DEC_TK - 1) / DEC_TK : 1;
      r.nt = MODE == DEC_MODE_SELECTED ? p.topk * r.tpb : (c.n_keys + DEC_TK - 1) / DEC_TK;
      if (MODE == DEC_MODE_SELECTED) r.ids = lane < p.topk ? p.topk_idx[h * p.topk + lane] : -1;
      return;
    }
    r.k0 = p.cu_k[b];
    r.len = p.cu_k[b + 1] - r.k0;
    if (MODE == DEC_MODE_SELECTED && p.seqlens) r.len = max(0, min(r.len, p.seqlens[b]));
    r.nt = dec_tiles<MODE>(p, b, r.len, r.n_keys, r.tpb);
    if (MODE == DEC_MODE_SELECTED) {
      const int32_t* sel = p.topk_idx + ((int64_t)h * p.batch + b) * p.topk;
      r.ids = lane < p.topk ? sel[lane] : -1;
    }
  };
  // first cache row and number of valid keys (0: nothing to do) of a tile
  auto tile_desc = [&](const Req& r, int tt, int& row0, int& n_valid) {
    if (MODE == DEC_MODE_COMPRESSED) {
      row0 = tt * DEC_TK;
      n_valid = min(DEC_TK, r.n_keys - row0);
    } else {
      const int t = tt / r.tpb, sub = tt - t * r.tpb;
      int blk;
      bool dup = false;  // a block that is listed twice counts once
      if (p.topk <= WAVE) {
        blk = __builtin_amdgcn_readlane(r.ids, t);
        dup = (__ballot(r.ids == blk) & ((1ull << t) - 1)) != 0;
      } else {
        const int32_t* sel = p.topk_idx + ((int64_t)h * p.batch + r.b) * p.topk;
        blk = sel[t];
        for (int u = 0; u < t; ++u) dup |= sel[u] == blk;
      }
      row0 = blk * p.block_size + sub * DEC_TK;
      n_valid = (blk < 0 || dup) ? 0 : min(min(DEC_TK, p.block_size - sub * DEC_TK), r.len - row0);
    }
    n_valid = max(n_valid, 0);
    row0 = n_valid > 0 ? row0 : 0;
  };
  // rows of a tile, coalesced (16 B per lane, D/8 lanes per row); rows past n_valid are zero so that
  // 0 * garbage cannot appear
  // (the offsets inside a tile fit 32 bits: uniform base pointer + one offset register per lane)
  auto load_rows = [&](vec8 (&dst)[VCH], const T* base, int64_t sn, int n_valid) {
    constexpr int RPI = 64 / (D / 8);  // rows per load instruction
    const uint32_t off0 = (uint32_t)(lane / (D / 8)) * (uint32_t)sn + (uint32_t)(lane % (D / 8)) * 8u;
    const uint32_t step = (uint32_t)RPI * (uint32_t)sn;
#pragma unroll
    for (int j = 0; j < VCH; ++j) {
      const int row = lane / (D / 8) + RPI * j;
      dst[j] = zero8<T>();
      if (row < n_valid) dst[j] = load16_stream<vec8>(base + (off0 + step * (uint32_t)j));
    }
  };
  auto load_tile = [&](vec8 (&dst)[VCH], const Req& r, bool is_v, int row0, int n_valid) {
    if constexpr (LAYER) {
      const DecParams::Source& c = MODE == DEC_MODE_COMPRESSED && r.b == 1 ? p.src[1] : p.src[0];
      const int64_t sn = is_v ? c.v_sn : c.k_sn;
      load_rows(dst, reinterpret_cast<const T*>(is_v ? c.v : c.k) + (int64_t)row0 * sn + (int64_t)h * (is_v ? c.v_sh : c.k_sh),
                sn, min(n_valid, c.n_cache - row0));
      if (row0 + n_valid > c.n_cache) {  // the last key is the row that is not in the cache yet
        const T* extra = reinterpret_cast<const T*>(is_v ? c.v_new : c.k_new) + h * D + (lane % (D / 8)) * 8;
        constexpr int RPI = 64 / (D / 8);
#pragma unroll
        for (int j = 0; j < VCH; ++j)
          if (lane / (D / 8) + RPI * j == c.n_cache - row0) dst[j] = load16<vec8>(extra);
      }
    } else {
      if (is_v) load_rows(dst, reinterpret_cast<const T*>(p.v) + (int64_t)(r.k0 + row0) * p.v_sn + (int64_t)h * p.v_sh, p.v_sn, n_valid);
      else load_rows(dst, reinterpret_cast<const T*>(p.k) + (int64_t)(r.k0 + row0) * p.k_sn + (int64_t)h * p.k_sh, p.k_sn, n_valid);
    }
  };
  // Layer form: rotation of the K rows of a tile in registers (the caches hold un-rotated rows).  The partner of a
  // lane's eight dims, D/2 further, sits D/16 lanes away and needs the same eight angles: each of the two forms four, packs
  // cosine and sine as two 16-bit numbers, which is what they are rounded to anyway, and they exchange them.  Every angle
  // is fp32 position times fp32 frequency, the product that prefill takes the sine and cosine of.  At position 131072 it
  // may lie 4e-3 from the exact angle, and an angle that does not lie there with it (one formed by the angle sum from
  // another row's) gives other 16-bit entries, 7 % of them in bf16.  (The angle sum for three rows of four is 1.1 us of a
  // step of 54.6 us over 32K tokens.  What the hardware's sine and cosine leave, about 1e-6, changed none of 640 entries
  // near positions 70000 and 131000.)
  constexpr int RPI = 64 / (D / 8);   // rows per load instruction
  auto partner = [&](uint32_t v) -> uint32_t {
    if constexpr (D == 128) return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x128, 0xf, 0xf, false);  // row_ror:8
    return (uint32_t)__shfl_xor((int)v, D / 16, WAVE);
  };
  const bool upper = (lane & (D / 16)) != 0;   // second half of the dims
  float freq[LAYER ? 4 : 1];
  if constexpr (LAYER) {
#pragma unroll
    for (int e = 0; e < 4; ++e) freq[e] = p.inv_freq[(lane % (D / 16)) * 8 + (upper ? 4 : 0) + e];
  }
  auto rotate_tile = [&](vec8 (&x)[VCH], const Req& r, int row0) {
    if constexpr (LAYER) {
      const DecParams::Source& c = MODE == DEC_MODE_COMPRESSED && r.b == 1 ? p.src[1] : p.src[0];
      const float sign = upper ? 1.f : -1.f;   // second half of the dims: x1 sin + x2 cos
#pragma unroll
      for (int j = 0; j < VCH; ++j) {
        const float pos = (float)(c.pos0 + (row0 + lane / (D / 8) + RPI * j) * c.pos_step);
        uint32_t mine[4], theirs[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          float cs, sn;
          sincos_turns(pos * freq[e], sn, cs);
          typedef T pair __attribute__((ext_vector_type(2)));
          mine[e] = __builtin_bit_cast(uint32_t, (pair){(T)(cs * p.rope_scale), (T)(sn * p.rope_scale)});
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) theirs[e] = partner(mine[e]);
        u32x4 own = __builtin_bit_cast(u32x4, x[j]), other;
#pragma unroll
        for (int i = 0; i < 4; ++i) other[i] = partner(own[i]);
        const vec8 y = __builtin_bit_cast(vec8, other);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          typedef T pair __attribute__((ext_vector_type(2)));
          const pair a = __builtin_bit_cast(pair, (e >= 4) == upper ? mine[e % 4] : theirs[e % 4]);
          x[j][e] = (T)((float)x[j][e] * (float)a[0] + sign * ((float)y[e] * (float)a[1]));
        }
      }
    }
  };
  auto park_tile = [&](const vec8 (&src)[VCH]) {
#pragma unroll
    for (int j = 0; j < VCH; ++j) {
      const int c = lane + 64 * j, row = c / (D / 8), cc = c % (D / 8);
      store16(&Vs[row * VS + cc * 8], src[j]);
    }
  };
  // B operand [k = d][n = column]: columns 0..g-1 = heads of the group, column g = scoring head (compressed mode)
  vec8 qreg[NS];
  auto load_q = [&](int b) {
    int hq_i = -1;
    if (l16 < p.g) hq_i = h * p.gq + p.head0 + l16;
    else if (MODE == DEC_MODE_COMPRESSED && p.raw_score && l16 == p.score_col) hq_i = h;  // as written: head h of q
    const T* qrow = reinterpret_cast<const T*>(p.q) + (LAYER ? 0 : (int64_t)b * p.q_sb) + (int64_t)max(hq_i, 0) * p.q_sh + 8 * kg;
#pragma unroll
    for (int s_ = 0; s_ < NS; ++s_) qreg[s_] = hq_i >= 0 ? load16<vec8>(qrow + 32 * s_) : zero8<T>();
  };
  const T* vtr = Vs + (4 * kg + (l16 >> 2)) * VS + 4 * (l16 & 3);

  float m = -INFINITY, l = 0.f;  // of column l16, replicated over the four key groups
  f32x4 oacc[NDT];               // O^T[d = 16 t + 4 kg + i][column l16]
#pragma unroll
  for (int t = 0; t < NDT; ++t) oacc[t] = f32x4{0.f, 0.f, 0.f, 0.f};

  Req rq, rqn;
  load_req(rq, LAYER ? source : ONE ? grp : seq.request_of(p, x_lo));
  rqn = rq;
  if constexpr (ONE) {
    const int wv = w - blockIdx.x * ONE, share = (LAYER ? grp : CHUNKED ? chunk : 0) * ONE + wv, shares = CHUNKED ? p.chunks[source] * ONE : ONE;
    x_lo = (int)((int64_t)rq.nt * share / shares);
    x_hi = (int)((int64_t)rq.nt * (share + 1) / shares);
  }
  int ttn = ONE ? x_lo : x_lo - seq.prefix(p, rq.b);
  int row0 = 0, n_valid = 0;
  if (!ONE || x_lo < x_hi) tile_desc(rq, ttn, row0, n_valid);
  vec8 kst[VCH], vst[VCH];
  load_tile(kst, rq, false, row0, n_valid);
  load_tile(vst, rq, true, row0, n_valid);
  load_q(rq.b);

  for (int x = x_lo; x < x_hi; ++x) {
    const bool has_next = x + 1 < x_hi;
    int row0n = 0, n_validn = 0;
    if (has_next) {  // x + 1 < total: a further tile exists
      if (++ttn == rqn.nt && !ONE) {
        ttn = 0;
        do load_req(rqn, rqn.b + 1); while (rqn.nt == 0);
      }
      tile_desc(rqn, ttn, row0n, n_validn);
    }
    const bool live = n_valid > 0;  // uniform
    // the K rows go through the LDS tile first, V uses it afterwards; the rows of the next tile are requested as
    // soon as the staging registers are free, so that they travel while this tile is computed
    if (live) {
      if (LAYER) rotate_tile(kst, rq, row0);
      park_tile(kst);
    }
    load_tile(kst, rqn, false, row0n, n_validn);
    float alpha = 1.f;
    vec8 pk = zero8<T>();  // contraction index 8 kg + j  <->  key 4 kg + j (j < 4), 16 + 4 kg + j - 4 (j >= 4)
    if (live) {
      __builtin_amdgcn_wave_barrier();
      // S^T[key][column] = K Q^T
      f32x4 acc[2];
#pragma unroll
      for (int a = 0; a < 2; ++a) {
        acc[a] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s_ = 0; s_ < NS; ++s_) {
          vec8 kf = load16<vec8>(&Vs[(a * 16 + l16) * VS + 32 * s_ + 8 * kg]);
          acc[a] = Elem<T>::mfma16(kf, qreg[s_], acc[a]);
        }
      }
      __builtin_amdgcn_wave_barrier();
      if (MODE == DEC_MODE_COMPRESSED && p.raw_score && l16 == p.score_col && (!LAYER || rq.b == 0)) {
        float* rs = p.raw_score + (LAYER ? (int64_t)h : (int64_t)h * p.batch + rq.b) * p.raw_ld + row0;
#pragma unroll
        for (int a = 0; a < 2; ++a) {
          const int key0 = a * 16 + 4 * kg;
          if (row0 + key0 < p.raw_ld) dec_store<LAYER>(rs + key0, acc[a]);
        }
      }
      float mx = m;
#pragma unroll
      for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int key = a * 16 + 4 * kg + i;
          const float sv = key < n_valid ? acc[a][i] : -INFINITY;
          acc[a][i] = sv;
          mx = fmaxf(mx, sv);
        }
      mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
      mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
      const float mref = mx * p.scale_log2;  // n_valid > 0, so mx is finite
      alpha = exp2f(m * p.scale_log2 - mref);
      float lsum = 0.f;
#pragma unroll
      for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float pv = fast_exp2(acc[a][i] * p.scale_log2 - mref);
          lsum += pv;
          pk[a * 4 + i] = (T)pv;
        }
      lsum += __shfl_xor(lsum, 16, 64);
      lsum += __shfl_xor(lsum, 32, 64);
      l = l * alpha + lsum;
      m = mx;
      park_tile(vst);
    }
    load_tile(vst, rqn, true, row0n, n_validn);
    if (live) {
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int t = 0; t < NDT; ++t) {
#pragma unroll
        for (int i = 0; i < 4; ++i) oacc[t][i] *= alpha;
        vec8 vf = lds_read_tr8<T>(vtr + 16 * t, 16 * VS);  // V^T[d = 16 t + l16][keys in the order of pk]
        oacc[t] = Elem<T>::mfma16(vf, pk, oacc[t]);
      }
      __builtin_amdgcn_wave_barrier();
    }
    if (!ONE && (!has_next || rqn.b != rq.b)) {
      // last tile of the request in this wave's share: the partial of (group, request) goes to slot group + request of
      // its kv head, which no other (group, request) can name because the shares are contiguous
      float* out = p.part + (int64_t)(h * (p.n_groups + p.batch) + grp + rq.b) * (p.g * PS);
      if (l16 < p.g) {
        float* oc = out + l16 * PS;
        if (kg == 0) *reinterpret_cast<f32x4*>(oc) = f32x4{m * p.scale_log2, l, 0.f, 0.f};
#pragma unroll
        for (int t = 0; t < NDT; ++t) *reinterpret_cast<f32x4*>(oc + 4 + 16 * t + 4 * kg) = oacc[t];
      }
      m = -INFINITY;
      l = 0.f;
#pragma unroll
      for (int t = 0; t < NDT; ++t) oacc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
      if (has_next) load_q(rqn.b);
    }
    rq = rqn;
    row0 = row0n;
    n_valid = n_validn;
  }
  if constexpr (ONE) {
    // the tile of a wave makes room for its partial
    static_assert(16 * PS * 4 <= DecLds<D>::BYTES, "partial of 16 heads");
    float* mine = reinterpret_cast<float*>(Vs);
    if (l16 < p.g) {
      float* oc = mine + l16 * PS;
      if (kg == 0) *reinterpret_cast<f32x4*>(oc) = f32x4{m * p.scale_log2, l, 0.f, 0.f};
#pragma unroll
      for (int t = 0; t < NDT; ++t) *reinterpret_cast<f32x4*>(oc + 4 + 16 * t + 4 * kg) = oacc[t];
    }
    __syncthreads();
    constexpr int LPR = D / 4, WS = DecLds<D>::BYTES / 4;
    const float* all = reinterpret_cast<const float*>(smem);
    for (int i = threadIdx.x; i < p.g * LPR; i += WAVE * ONE) {
      const int col = i / LPR, lr = i % LPR;
      float mt = -INFINITY, lt = 0.f;
      f32x4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int j = 0; j < ONE; ++j) mt = fmaxf(mt, all[j * WS + col * PS]);
      if (mt > -INFINITY) {
#pragma unroll
        for (int j = 0; j < ONE; ++j) {
          const float* oc = all + j * WS + col * PS;
          const float wgt = exp2f(oc[0] - mt);   // 0 for a wave without a key
          lt += wgt * oc[1];
          o += wgt * *reinterpret_cast<const f32x4*>(oc + 4 + 4 * lr);
        }
      }
      if constexpr (CHUNKED) {
        const int64_t at = LAYER ? (int64_t)h * (p.chunks[0] + p.chunks[1]) + chunk : ((int64_t)grp * p.hkv + h) * p.chunks[0] + chunk;
        float* out = p.part + at * (p.g * PS) + col * PS;
        if (lr == 0) dec_store<true>(out, f32x4{mt, lt, 0.f, 0.f});
        dec_store<true>(out + 4 + 4 * lr, o);
      } else {
        o *= lt > 0.f ? 1.f / lt : 0.f;
        dec_emit<T, D>(p, grp, h, col, lr, o, lt > 0.f ? mt + log2f(lt) : -INFINITY);
      }
    }
  }
}
template <typename T, int D, int MODE, int ONE = 0>
__global__ void __launch_bounds__(ONE ? WAVE * ONE : WAVE * DecOcc<D>::WG_WAVES, ONE ? 1 : DecOcc<D>::WAVES_PER_SIMD)
decode_attn_kernel(DecParams p) {
  decode_attn_body<T, D, MODE, false, ONE>(p);
}

// Whether this work-group is the last of the `n` that count themselves in at `counter`: what the others stored with dec_store
// before has arrived then and is seen by dec_load.  The last one leaves the counter at zero.
__device__ __forceinline__ bool dec_last_to_arrive(int* counter, int n) {
  __shared__ int last;
  vm_wait<0>();      // this wave's stores
  __syncthreads();   // those of all waves
  if (threadIdx.x == 0) {
    last = __hip_atomic_fetch_add(counter, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == n - 1;
    if (last) *counter = 0;
  }
  __syncthreads();
  return last != 0;
}

// The same without a counter that somebody had to clear: every work-group leaves the number of the call beside its partial and
// looks whether all n numbers are there.  Its own store is awaited before it looks, so that at least the last one sees them all;
// if several do, they write the same results.  Numbers are not used twice, and they are cleared once all have been seen: a
// recorded call that is replayed starts without them.
__device__ __forceinline__ bool dec_all_arrived(uint64_t* stamps, int n, int mine, uint64_t call) {
  __shared__ int all;
  vm_wait<0>();
  __syncthreads();
  if (threadIdx.x < WAVE) {
    if (threadIdx.x == 0) __hip_atomic_store(stamps + mine, call, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    vm_wait<0>();
    const bool there =
        (int)threadIdx.x >= n || __hip_atomic_load(stamps + threadIdx.x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == call;
    const bool last = __all(there);
    if (threadIdx.x == 0) all = last;
    if (last && (int)threadIdx.x < n) __hip_atomic_store(stamps + threadIdx.x, (uint64_t)0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  __syncthreads();
  return all != 0;
}

// Partials of a (request, kv head) -> o, lse.  D/4 lanes hold a row of a partial; the row groups of the work-group are
// dealt to the heads of the group and, where there are more of them than heads, to slices of the partials.  All the
// loads of a slice are issued before they are used, slices meet in LDS, everything in a fixed order.  (One thread per
// output element walking through all partials - twice, for the maximum first - took 8 to 25 us of a 50 us step.)
constexpr int DEC_MERGE_THREADS = 512;
// emit(col, lr, o / l as f32x4, lse) is called by the D/4 lanes that hold the merged row of head `col` of the group.
// `part`: the first of ns partials, `slot` floats apart.
template <int D, int THREADS, bool SHARED, typename EMIT>
__device__ __forceinline__ void dec_merge_slots(const DecParams& p, const float* part, int ns, int slot, EMIT emit) {
  constexpr int LPR = D / 4, NG = THREADS / LPR, PS = D + 4;
  __shared__ float part_m[NG], part_l[NG];
  __shared__ f32x4 part_o[NG][LPR];
  const int rg = threadIdx.x / LPR, lr = threadIdx.x % LPR;
  const int n_slice = max(1, NG / p.g);      // slices per head; row groups beyond g * n_slice have none
  const int cols = NG / n_slice;             // heads in flight
  const int slice = rg % n_slice;
  const int chunk = (ns + n_slice - 1) / n_slice, s_lo = slice * chunk, s_hi = min(ns, s_lo + chunk);
  for (int c0 = 0; c0 < p.g; c0 += cols) {
    const int col = c0 + rg / n_slice;
    const bool live = rg / n_slice < cols && col < p.g;
    float m = -INFINITY, l = 0.f;
    f32x4 o = {0.f, 0.f, 0.f, 0.f};
    if (live) {
      const float* pc = part + col * PS;
      constexpr int UB = 8;
      for (int sb = s_lo; sb < s_hi; sb += UB) {
        float ms[UB], ls[UB];
        f32x4 os[UB];
#pragma unroll
        for (int u = 0; u < UB; ++u) {
          const float* ps = pc + (int64_t)min(sb + u, s_hi - 1) * slot;
          const f32x2 ml = dec_load<SHARED, f32x2>(ps);
          ms[u] = sb + u < s_hi ? ml[0] : -INFINITY;
          ls[u] = ml[1];
          os[u] = dec_load<SHARED, f32x4>(ps + 4 + lr * 4);
        }
        float mn = m;
#pragma unroll
        for (int u = 0; u < UB; ++u) mn = fmaxf(mn, ms[u]);
        if (mn > -INFINITY) {
          const float keep = exp2f(m - mn);
          l *= keep;
          o *= keep;
#pragma unroll
          for (int u = 0; u < UB; ++u) {
            const float wgt = exp2f(ms[u] - mn);   // 0 for a partial without a key
            l += wgt * ls[u];
            o += wgt * os[u];
          }
          m = mn;
        }
      }
    }
    if (n_slice > 1) {
      if (c0) __syncthreads();
      if (lr == 0) {
        part_m[rg] = m;
        part_l[rg] = l;
      }
      part_o[rg][lr] = o;
      __syncthreads();
      if (slice == 0 && live) {
        float mt = m;
        for (int j = 1; j < n_slice; ++j) mt = fmaxf(mt, part_m[rg + j]);
        if (mt > -INFINITY) {
          const float keep = exp2f(m - mt);
          l *= keep;
          o *= keep;
          for (int j = 1; j < n_slice; ++j) {
            const float wgt = exp2f(part_m[rg + j] - mt);
            l += wgt * part_l[rg + j];
            o += wgt * part_o[rg + j][lr];
          }
        }
        m = mt;
      }
    }
    if (slice == 0 && live) {
      const float inv_l = l > 0.f ? 1.f / l : 0.f;
      emit(col, lr, o * inv_l, l > 0.f ? m + log2f(l) : -INFINITY);
    }
  }
}

template <typename T, int D, int MODE>
__global__ void __launch_bounds__(DEC_MERGE_THREADS)
decode_merge_kernel(DecParams p) {
  const int b = blockIdx.x, h = blockIdx.y;
  DecSeq<MODE> seq;
  seq.init(p);
  const int per = dec_share(seq.total, p.n_groups);
  const int x0 = seq.prefix(p, b);
  const int nt = (b + 1 < p.batch ? seq.prefix(p, b + 1) : seq.total) - x0;
  const int g0 = x0 / per;
  const int ns = nt > 0 ? (x0 + nt - 1) / per - g0 + 1 : 0;
  const int slot = p.g * (D + 4);
  const float* part = p.part + (int64_t)(h * (p.n_groups + p.batch) + g0 + b) * slot;
  dec_merge_slots<D, DEC_MERGE_THREADS, false>(p, part, ns, slot, [&](int col, int lr, f32x4 o, float lse) {
    dec_emit<T, D>(p, b, h, col, lr, o, lse);
  });
}

// A (request, kv head) in p.chunks[0] work-groups, the last of which merges (dec_all_arrived).
constexpr int DEC_CHUNK_WAVES = 4, DEC_MAX_CHUNKS = WAVE, DEC_CHUNK_SLOTS = 1024;   // work-groups of a launch at most
template <typename T, int D, int MODE>
__global__ void __launch_bounds__(WAVE * DEC_CHUNK_WAVES, DecOcc<D>::WAVES_PER_SIMD)
decode_attn_chunked_kernel(DecParams p) {
  decode_attn_body<T, D, MODE, false, DEC_CHUNK_WAVES, true>(p);
  const int pair = blockIdx.x / p.hkv, h = blockIdx.x - pair * p.hkv, b = (uint32_t)pair / (uint32_t)p.chunks[0], slot = p.g * (D + 4);
  const int64_t first = ((int64_t)b * p.hkv + h) * p.chunks[0];
  if (!dec_all_arrived(p.stamps + first, p.chunks[0], pair - b * p.chunks[0], p.call)) return;
  dec_merge_slots<D, WAVE * DEC_CHUNK_WAVES, true>(p, p.part + first * slot, p.chunks[0], slot, [&](int col, int lr, f32x4 o, float lse) {
    dec_emit<T, D>(p, b, h, col, lr, o, lse);
  });
}

// ------------------------------------------------------------------ top-k ----
struct DecTopkParams {
  const float* raw_score;  // [Hkv, B, raw_ld]
  int64_t raw_ld;
  const float* lse;        // [Hq, B]
  const int32_t* cu_ck;    // [B+1] compressed rows per request
  const int32_t* pos;      // [B]
  const int32_t* seqlens;  // [B] cache length including the new token
  int batch, hkv, g;
  int kernel_size, kernel_stride, block_size, topk, init_blocks, local_blocks;
  int as_written;
  int scores_to_bf16;      // rank the block scores after rounding them to bf16 (what the prefill selection does)
  float scale_log2;
  int32_t* topk_idx;       // [Hkv, B, topk]
  float* block_score;      // optional [Hkv, B, score_ld]
  int64_t score_ld;
};

// One work-group per (request, kv head).  A candidate is a 64-bit key, score bits above and the complement of the block
// id below (scores are >= 0): the larger key is the larger score or, on equal scores, the lower id.  Every wave takes
// the topk best of its quarter of the blocks by itself - the candidates stay in registers, the topk-th largest score is
// found bit by bit, a step being a compare and a ballot per register and scalar counting - and one wave ranks the 4 topk
// finalists.  (topk rounds of a wave maximum instead of the threshold: 8 requests of 8K to
// 16K tokens 6.9 us, this form 5.2.)
constexpr int DEC_TOPK_THREADS = 256;
constexpr int DEC_TOPK_WAVES = DEC_TOPK_THREADS / WAVE;
constexpr int DEC_TOPK_MAX_K = 16;   // finalists of the four waves fill one wave

// NREG: candidates per lane in registers (blocks <= 256 NREG, topk <= DEC_TOPK_MAX_K); 0: any size, scores in LDS
// (nc, qp, len: compressed rows, query position and cache length of request b; lse_r: lse of the scoring head)
// Called by a whole work-group of at least DEC_TOPK_THREADS threads; the threads beyond those only keep the barriers.
// SHARED: the raw scores come from other work-groups of the launch.
template <int NREG, bool SHARED>
__device__ __forceinline__ void dec_topk_block(const DecTopkParams& p, int b, int h, int nc, int qp, int len, float lse_r,
                                               float* bs) {
  __shared__ uint64_t final_key[DEC_TOPK_WAVES * DEC_TOPK_MAX_K];
  const int tid = threadIdx.x, lane = tid & (WAVE - 1), wv = tid / WAVE;
  const bool active = tid < DEC_TOPK_THREADS;
  const int n_vis = qp >= p.kernel_size - 1 ? min(nc, (qp - p.kernel_size + 1) / p.kernel_stride + 1) : 0;
  const int nblk = p.as_written ? (nc + p.block_size - 1) / p.block_size : (len + p.block_size - 1) / p.block_size;
  const int bq = p.as_written ? 0 : (len - 1) / p.block_size;
  const int na = p.kernel_size / p.kernel_stride, ne = p.block_size / p.kernel_stride;
  const int n_off = na + ne - 1, pad = na - 1;
  const float* rs = p.raw_score + ((int64_t)h * p.batch + b) * p.raw_ld;
  auto finish = [&](float acc, int blk) {
    if (blk < p.init_blocks || (bq >= blk && bq < blk + p.local_blocks)) acc = INFINITY;
    if (p.block_score) p.block_score[((int64_t)h * p.batch + b) * p.score_ld + blk] = acc;
    return p.scores_to_bf16 ? (float)(__bf16)acc : acc;
  };
  auto block_score = [&](int blk) {
    float acc = 0.f;
    const int c0 = blk * ne - pad;
    for (int o = 0; o < n_off; ++o) {
      const int c = c0 + o;
      if (c >= 0 && c < n_vis) {
        const int wgt = min(min(o, n_off - 1 - o), min(na, ne) - 1) + 1;
        acc += (float)wgt * fast_exp2(dec_load<SHARED, float>(rs + c) * p.scale_log2 - lse_r);
      }
    }
    return finish(acc, blk);
  };
  auto key_of = [](float score, int blk) { return ((uint64_t)__float_as_uint(score) << 32) | (0xFFFFFFFFu - (uint32_t)blk); };
  if (p.block_score)
    for (int64_t blk = nblk + tid; blk < p.score_ld; blk += DEC_TOPK_THREADS)
      p.block_score[((int64_t)h * p.batch + b) * p.score_ld + blk] = -INFINITY;
  int32_t* out = p.topk_idx + ((int64_t)h * p.batch + b) * p.topk;
  if constexpr (NREG > 0) {
    // score bits + 1; 0: no candidate.  A NaN is a large score; the largest of them is cut to the 31 bits that the search
    // below runs over, a key above every threshold would be taken however many there are.
    uint32_t key[NREG];
    auto key_bits = [](float score) { return min(__float_as_uint(score) & 0x7FFFFFFFu, 0x7FFFFFFEu) + 1u; };
    if (na == 2 && ne == 4) {
      // usual geometry: the scores 4 blk - 1 .. 4 blk + 3 with weights 1 2 2 2 1, all loads of a lane in flight at once
      f32x4 x[NREG];
      float x0[NREG];
      const int last = (int)p.raw_ld - 4;   // raw_ld is a multiple of four; what lies past it is not visible
#pragma unroll
      for (int r = 0; r < NREG; ++r) {
        const int c = 4 * (tid + DEC_TOPK_THREADS * r);
        x[r] = dec_load<SHARED, f32x4>(rs + min(c, last));
        x0[r] = dec_load<SHARED, float>(rs + min(max(c - 1, 0), last));
      }
#pragma unroll
      for (int r = 0; r < NREG; ++r) {
        const int blk = tid + DEC_TOPK_THREADS * r, c = 4 * blk;
        auto pr = [&](float v) { return fast_exp2(v * p.scale_log2 - lse_r); };
        float acc = 0.f;
        if (c >= 1 && c - 1 < n_vis) acc += pr(x0[r]);
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (c + j < n_vis) acc += (j < 3 ? 2.f : 1.f) * pr(x[r][j]);
        key[r] = active && blk < nblk ? key_bits(finish(acc, blk)) : 0u;
      }
    } else {
#pragma unroll
      for (int r = 0; r < NREG; ++r) {
        const int blk = tid + DEC_TOPK_THREADS * r;
        key[r] = active && blk < nblk ? key_bits(block_score(blk)) : 0u;
      }
    }
    if (active) {   // whole waves
      auto count_from = [&](uint32_t t) {
        int c = 0;
#pragma unroll
        for (int r = 0; r < NREG; ++r) c += (int)__popcll(__ballot(key[r] >= t));
        return c;
      };
      // largest threshold that at least topk keys reach (1 where there are fewer); rounded scores have zeros in their low half
      uint32_t thr = 1;
      int at_thr = count_from(1);
      if (at_thr > p.topk) {
        thr = 0;
        for (int bit = 30; bit >= 0 && at_thr != p.topk; --bit) {
          const uint32_t t = thr | (1u << bit);
          const int c = count_from(t);
          if (c >= p.topk) {
            thr = t;
            at_thr = c;
          }
        }
      }
      // of the keys equal to the threshold the lowest ids
      int need = at_thr <= p.topk ? at_thr : p.topk - count_from(thr + 1);
      uint64_t* fin = final_key + wv * DEC_TOPK_MAX_K;
      if (lane < DEC_TOPK_MAX_K) fin[lane] = 0;
      __builtin_amdgcn_wave_barrier();
      int base = 0;
#pragma unroll
      for (int r = 0; r < NREG; ++r) {
        bool take = key[r] >= thr;
        if (at_thr > p.topk) {
          const uint64_t eq = __ballot(key[r] == thr);
          const int rank = __builtin_amdgcn_mbcnt_hi((uint32_t)(eq >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)eq, 0));
          take = key[r] > thr || (key[r] == thr && rank < need);
          need = max(0, need - (int)__popcll(eq));
        }
        const uint64_t m = __ballot(take);
        const int at = base + __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0));
        if (take) fin[at] = key_of(__uint_as_float(key[r] - 1u), tid + DEC_TOPK_THREADS * r);
        base += (int)__popcll(m);
      }
    }
    __syncthreads();
    if (wv == 0) {
      const uint64_t k = final_key[lane];
      int rank = 0, n = 0;
#pragma unroll
      for (int j = 0; j < WAVE; ++j) {
        const uint64_t other = ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(k >> 32), j) << 32) |
                               (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)k, j);
        rank += other > k;
        n += other != 0;
      }
      if (k != 0 && rank < p.topk) out[rank] = (int32_t)(0xFFFFFFFFu - (uint32_t)k);
      if (lane >= n && lane < p.topk) out[lane] = -1;  // fewer than topk blocks exist
    }
    return;
  }
  for (int blk = tid; blk < nblk; blk += DEC_TOPK_THREADS) bs[blk] = block_score(blk);
  __syncthreads();
  for (int t = 0; t < p.topk; ++t) {
    uint64_t best = 0;
    for (int blk = tid; blk < nblk; blk += DEC_TOPK_THREADS) {
      const float vv = bs[blk];
      const uint64_t k = vv < 0.f ? 0ull : key_of(vv, blk);
      best = k > best ? k : best;
    }
    best = wave_max_u64(best);
    if (active && lane == 0) final_key[wv] = best;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < DEC_TOPK_WAVES; ++w) best = final_key[w] > best ? final_key[w] : best;
    const int best_id = (int)(0xFFFFFFFFu - (uint32_t)best);
    if (tid == 0) {
      out[t] = best ? best_id : -1;  // fewer than topk blocks exist
      if (best) bs[best_id] = -1.f;
    }
    __syncthreads();
  }
}

template <int NREG>
__global__ void __launch_bounds__(DEC_TOPK_THREADS)
decode_topk_kernel(DecTopkParams p) {
  extern __shared__ float bs[];
  const int b = blockIdx.x, h = blockIdx.y;
  const int hq_s = p.as_written ? h : h * p.g;
  dec_topk_block<NREG, false>(p, b, h, p.cu_ck[b + 1] - p.cu_ck[b], p.pos[b], p.seqlens[b], p.lse[(int64_t)hq_s * p.batch + b], bs);
}

// ------------------------------------------------------- one token through the layer ----
// Four launches for a token of one request: projections + rotation of q; compressed and window attention with their merge and
// the block selection; selected attention with its merge and the gated sum; output projection.  The caches stay as they are
// (un-rotated, without the new token): keys are rotated in registers on their way into LDS, the new row is read from
// where the projection left it.  Copying and rotating the caches for a step, as a composition of the single operators
// does, moves 32 times the bytes that the step needs (32K tokens: 740 us in 31 launches).
struct DecLayerParams {
  const void* x;
  const void* w[4];        // q, k, v, gate: [rows, hidden] row-major
  const void* w_o;         // [hidden, hq D]
  int hidden, hq, hkv, d, pos;
  const float* inv_freq;
  float rope_scale;
  void *q_rot, *k_new, *v_new;   // [hq, D], [hkv, D], [hkv, D]
  void* gate;                    // [3] sigmoid values
  void *o_cmp, *o_win;           // [hq, D]
  int* arrived;                  // [2][hkv], see DecParams
  void* attn;                    // [hq, D] gated sum
  void* y;                       // [hidden]
};

// Dot products of one wave: two rows of a matrix with x, n elements (a multiple of 8), four 512-element steps of both
// rows in flight.  A row comes in 1 KB pieces; the wave is done after one trip to memory per 2048 elements.
template <typename T>
__device__ __forceinline__ void dot2(const T* __restrict__ x, const T* __restrict__ r0, const T* __restrict__ r1, int n,
                                     float& s0, float& s1) {
  typedef typename Elem<T>::vec8 vec8;
  const int lane = threadIdx.x & (WAVE - 1);
  s0 = s1 = 0.f;
  constexpr int U = 4;
  for (int e0 = lane * 8; e0 < n; e0 += 512 * U) {
    vec8 a[U], b[U], c[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int e = e0 + 512 * u;
      a[u] = b[u] = c[u] = zero8<T>();
      if (e < n) {
        b[u] = load16_stream<vec8>(r0 + e);
        c[u] = load16_stream<vec8>(r1 + e);
        a[u] = load16<vec8>(x + e);
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        s0 += (float)a[u][i] * (float)b[u][i];
        s1 += (float)a[u][i] * (float)c[u][i];
      }
  }
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) {
    s0 += __shfl_xor(s0, o, WAVE);
    s1 += __shfl_xor(s1, o, WAVE);
  }
}

// wave = rows d and d + D/2 of one head of q, k or v (the pair that the rotation mixes), or one row of the gate
template <typename T>
__global__ void __launch_bounds__(256)
decode_project_kernel(DecLayerParams p) {
  if (blockIdx.x == 0)
    for (int i = threadIdx.x; i < 2 * p.hkv; i += 256) p.arrived[i] = 0;
  const int u = blockIdx.x * 4 + threadIdx.x / WAVE, half = p.d / 2;
  const int nq = p.hq * half, nkv = p.hkv * half;
  const int m = u < nq ? 0 : u < nq + nkv ? 1 : u < nq + 2 * nkv ? 2 : 3;   // which matrix (uniform)
  const int v = u - (m == 0 ? 0 : m == 1 ? nq : m == 2 ? nq + nkv : nq + 2 * nkv);
  if (m == 3 && v >= 3) return;
  const int row0 = m == 3 ? v : v / half * p.d + v % half, row1 = m == 3 ? v : row0 + half;
  const T* w = reinterpret_cast<const T*>(p.w[m]);
  float s0, s1;
  dot2<T>(reinterpret_cast<const T*>(p.x), w + (int64_t)row0 * p.hidden, w + (int64_t)row1 * p.hidden, p.hidden, s0, s1);
  if ((threadIdx.x & (WAVE - 1)) != 0) return;
  const T y0 = (T)s0, y1 = (T)s1;
  if (m == 0) {
    float sn, cs;
    sincos_turns((float)p.pos * p.inv_freq[v % half], sn, cs);
    cs = (float)(T)(cs * p.rope_scale);
    sn = (float)(T)(sn * p.rope_scale);
    T* q = reinterpret_cast<T*>(p.q_rot);
    q[row0] = (T)((float)y0 * cs - (float)y1 * sn);
    q[row1] = (T)((float)y0 * sn + (float)y1 * cs);
  } else if (m < 3) {
    T* out = reinterpret_cast<T*>(m == 1 ? p.k_new : p.v_new);
    out[row0] = y0;
    out[row1] = y1;
  } else {
    reinterpret_cast<T*>(p.gate)[v] = (T)(1.f / (1.f + expf(-(float)y0)));
  }
}

// y = w_o attn: wave = two rows
template <typename T>
__global__ void __launch_bounds__(256)
decode_out_kernel(DecLayerParams p) {
  const int r0 = (blockIdx.x * 4 + threadIdx.x / WAVE) * 2;
  if (r0 >= p.hidden) return;
  const int r1 = min(r0 + 1, p.hidden - 1), n = p.hq * p.d;
  const T* w = reinterpret_cast<const T*>(p.w_o);
  float s0, s1;
  dot2<T>(reinterpret_cast<const T*>(p.attn), w + (int64_t)r0 * n, w + (int64_t)r1 * n, n, s0, s1);
  if ((threadIdx.x & (WAVE - 1)) != 0) return;
  T* y = reinterpret_cast<T*>(p.y);
  y[r0] = (T)s0;
  y[r1] = (T)s1;
}

// Compressed and window attention, their merge and the block selection in one launch: the last work-group of a (source, kv head)
// to leave its partial merges them, and, of the compressed branch, selects the blocks of that head.  A launch of its own for
// that took 4 us more, most of them until its first loads had returned.
template <int D> struct DecLayerWaves {
  static constexpr int N = 4;   // DEC_TOPK_THREADS for the selection; more waves per work-group bring more rows into one CU
};
template <typename T, int D, int NREG>
__global__ void __launch_bounds__(WAVE * DecLayerWaves<D>::N, DecOcc<D>::WAVES_PER_SIMD)
decode_layer_select_kernel(DecParams p, DecTopkParams tk, DecLayerParams lp) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  __shared__ float lse_s;
  decode_attn_body<T, D, DEC_MODE_COMPRESSED, true, DecLayerWaves<D>::N>(p);
  const int chunk = blockIdx.x / p.hkv, h = blockIdx.x - chunk * p.hkv, b = chunk >= p.chunks[0], slot = p.g * (D + 4);
  if (!dec_last_to_arrive(p.arrived + b * p.hkv + h, p.chunks[b])) return;
  T* out = reinterpret_cast<T*>(b == 0 ? lp.o_cmp : lp.o_win);
  const float* part = p.part + ((int64_t)h * (p.chunks[0] + p.chunks[1]) + (b ? p.chunks[0] : 0)) * slot;
  dec_merge_slots<D, WAVE * DecLayerWaves<D>::N, true>(p, part, p.chunks[b], slot, [&](int col, int lr, f32x4 o, float lse) {
    typename Elem<T>::vec4 x;
#pragma unroll
    for (int i = 0; i < 4; ++i) x[i] = (T)o[i];
    store8(out + (h * p.g + col) * D + lr * 4, x);
    if (col == 0 && lr == 0) lse_s = lse;
  });
  if (b != 0) return;
  __syncthreads();
  dec_topk_block<NREG, true>(tk, 0, h, p.src[0].n_keys, lp.pos, lp.pos + 1, lse_s, reinterpret_cast<float*>(smem));
}

// Selected attention, its merge and the gated sum of the three branches, in the same way
template <typename T, int D>
__global__ void __launch_bounds__(WAVE * DecLayerWaves<D>::N, DecOcc<D>::WAVES_PER_SIMD)
decode_layer_combine_kernel(DecParams p, DecLayerParams lp) {
  typedef typename Elem<T>::vec4 vec4;
  decode_attn_body<T, D, DEC_MODE_SELECTED, true, DecLayerWaves<D>::N>(p);
  const int h = blockIdx.x % p.hkv, slot = p.g * (D + 4);
  if (!dec_last_to_arrive(p.arrived + h, p.chunks[0])) return;
  const T* gate = reinterpret_cast<const T*>(lp.gate);
  const float g0 = (float)gate[0], g1 = (float)gate[1], g2 = (float)gate[2];
  dec_merge_slots<D, WAVE * DecLayerWaves<D>::N, true>(p, p.part + (int64_t)h * p.chunks[0] * slot, p.chunks[0], slot, [&](int col, int lr, f32x4 o, float) {
    const int at = (h * p.g + col) * D + lr * 4;
    const vec4 a = load8<vec4>(reinterpret_cast<const T*>(lp.o_cmp) + at), c = load8<vec4>(reinterpret_cast<const T*>(lp.o_win) + at);
    vec4 x;
#pragma unroll
    for (int i = 0; i < 4; ++i) x[i] = (T)(g0 * (float)a[i] + g1 * (float)(T)o[i] + g2 * (float)c[i]);
    store8(reinterpret_cast<T*>(lp.attn) + at, x);
  });
}

// One work-group per (request, kv head): a tile takes a wave 3 us from end to end, so its waves may have few of them.  With
// few pairs chunks spread the tiles over more of the chip, and two tiles per wave are the most that the saved exchange
// pays for (one request, two tiles: compressed keys of 6000 tokens 8.1 against 8.8 us); where there are pairs enough to leave
// no chunks, shares would be that long themselves (32 requests x 8 heads, 1024 selected keys, a whole step: 41 -> 37 us).  512
// pairs are resident.
template <int D> struct DecOne {
  static constexpr int WAVES = D >= 256 ? 4 : 8;   // what the registers allow
};
template <typename T, int D, int MODE> static int dec_one_launch(const DecParams& p, int pairs, int dev, hipStream_t stream) {
  constexpr int W = DecOne<D>::WAVES, LDS = W * DecLds<D>::BYTES;
  static LdsAllowed allowed;
  if (int rc_ = allow_lds(allowed, (const void*)decode_attn_kernel<T, D, MODE, W>, LDS, dev)) return rc_;
  decode_attn_kernel<T, D, MODE, W><<<pairs, WAVE * W, LDS, stream>>>(p);
  return 0;
}

// number of waves that are resident at once on the current device, and that device
template <typename T, int D, int MODE>
static int dec_grid_waves(int* n_waves, int* device) {
  static int cached[16] = {0};
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  *device = e == hipSuccess ? dev : -1;
  if (e == hipSuccess && dev >= 0 && dev < 16 && cached[dev] > 0) {
    *n_waves = cached[dev];
    return 0;
  }
  int cus = 0, per_cu = 0;
  if (e == hipSuccess) e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
  if (e == hipSuccess)
    e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, decode_attn_kernel<T, D, MODE>, WAVE, DecLds<D>::BYTES);
  if (e != hipSuccess || cus < 1 || per_cu < 1) {
    set_error("decode: occupancy query failed (%s, %d CUs, %d work-groups per CU)", hipGetErrorString(e), cus, per_cu);
    return e != hipSuccess ? (int)e : FSA_ERR_UNSUPPORTED;
  }
  int n = cus * per_cu;
  if (n > DEC_MAX_WAVES) n = DEC_MAX_WAVES;
  if (dev >= 0 && dev < 16) cached[dev] = n;
  *n_waves = n;
  return 0;
}

// Work-groups per (request, kv head) of the chunked form: a tile per wave while the chip holds them at once, 1 where another form
// is the better one.  Against partials and a merge launch, us, 32 + 8 heads of 128, compressed: one request of 16K 10.7 -> 8.8, 32K
// 12.0 -> 8.8, 128K 21.9 -> 16.8, four of 32K 16.0 -> 12.7, 8 of 16K 14.8 -> 12.6; 16 of 32K 28.5 -> 27.4, with twice the work-groups
// 31.9; 1024 selected keys: one request 9.1 -> 8.6.  What the chip does not hold waits for a place: 128 chunks beside 256 of head_dim
// 256, one to a CU, make 12 pairs of 125 tiles 1.24 times as slow as without chunks, 256 in all 0.75 times.  With more than
// DEC_CHUNK_TILES tiles per wave the shares of the persistent grid are better.
constexpr int DEC_CHUNK_TILES = 4;
template <int D> static int64_t dec_chunks(int64_t req_tiles, int64_t pairs) {
  constexpr int64_t RESIDENT = 256 * DecOcc<D>::WAVES_PER_SIMD;   // a wave on every SIMD of a CU is a work-group
  static_assert(RESIDENT <= DEC_CHUNK_SLOTS, "room for the partials");
  const int64_t most = std::min<int64_t>(DEC_MAX_CHUNKS, RESIDENT / std::max<int64_t>(1, pairs));
  const int64_t n = std::min((req_tiles + DEC_CHUNK_WAVES - 1) / DEC_CHUNK_WAVES, most);
  return n > 1 && req_tiles <= n * DEC_CHUNK_WAVES * DEC_CHUNK_TILES ? n : 1;
}
// Which form.  One work-group for a pair, without an exchange, where its waves have at most two tiles, and four where there are
// pairs enough that the chip is not left idle.  There chunks pay for their exchange only while they cut a pair into four and
// more, and then from the fourth tile on; us, one work-group / chunks, compressed: 128 pairs of 17 tiles of 64 dims 5.8 / 8.3, of 32
// 8.2 / 9.3, of 128 dims 17 tiles 9.9 / 11.3, 32 tiles 17.2 / 16.4, 200 pairs 18.3 / 22.7.
enum DecForm { DEC_FORM_SHARES, DEC_FORM_ONE, DEC_FORM_CHUNKS };
template <int D> static DecForm dec_form(int64_t req_tiles, int64_t pairs, int64_t* chunks) {
  constexpr int W = DecOne<D>::WAVES;
  *chunks = dec_chunks<D>(req_tiles, pairs);
  if (req_tiles <= 2 * W && pairs <= 512) return DEC_FORM_ONE;
  if (pairs >= 96 && req_tiles <= 4 * W && pairs <= 512 && !(D >= 128 && *chunks >= 4 && req_tiles > 3 * W)) return DEC_FORM_ONE;
  return *chunks > 1 && req_tiles > 2 * W ? DEC_FORM_CHUNKS : DEC_FORM_SHARES;
}
static uint64_t dec_call_number() {
  static std::atomic<uint64_t> next{0x5eed0fca115ull};
  const uint64_t x = next.fetch_add(1, std::memory_order_relaxed) * 0x9e3779b97f4a7c15ull;   // odd: no number comes twice
  return x ? x : dec_call_number();
}

// p0.g holds the whole group size on entry.  Scores of the scoring head: with the first head of the group as
// scoring head they are the scores of column 0 of the first launch; with the head that the reference's kernel
// actually reads (q head number h for kv head h) they need a column of their own, so that launch has 15 heads.
template <typename T, int D, int MODE>
static int dec_launch(const DecParams& p0, hipStream_t stream) {
  int n_waves = 0, dev = -1;
  int rc = dec_grid_waves<T, D, MODE>(&n_waves, &dev);
  if (rc) return rc;
  ProfScope ps_(MODE == DEC_MODE_COMPRESSED ? "decode_cmpattn" : "decode_selattn", stream);
  DecParams p = p0;
  p.gq = p0.g;
  // no more waves than there can be tiles
  const int64_t req_tiles = MODE == DEC_MODE_COMPRESSED ? ((int64_t)p.max_keys + DEC_TK - 1) / DEC_TK
                                                        : (int64_t)p.topk * ((p.block_size + DEC_TK - 1) / DEC_TK);
  const int64_t pairs = (int64_t)p.batch * p.hkv;
  int64_t chunks = 0;
  const DecForm form = dec_form<D>(req_tiles, pairs, &chunks);
  const int64_t most = std::max<int64_t>(1, req_tiles * p.batch);
  p.n_groups = (int)std::min<int64_t>(std::max(1, n_waves / p.hkv), most);
  if (MODE == DEC_MODE_COMPRESSED && p.batch > WAVE && form == DEC_FORM_SHARES) decode_plan_kernel<<<1, WAVE, 0, stream>>>(p);
  // two neighbouring kv heads per work-group (64 requests of 32K - 128K: 304 us a step with one, 288 / 291 / 293 with
  // two / four / eight)
  const int wg_waves = std::min(p.hkv, DecOcc<D>::WG_WAVES);
  const int grid = (p.n_groups * p.hkv + wg_waves - 1) / wg_waves;
  for (int head0 = 0; head0 < p0.g;) {
    p.head0 = head0;
    p.raw_score = head0 == 0 ? p0.raw_score : nullptr;
    const bool own_col = MODE == DEC_MODE_COMPRESSED && p.raw_score && p0.score_head_as_written;
    p.g = std::min(p0.g - head0, own_col ? 15 : 16);
    p.score_col = own_col ? p.g : 0;
    if (form == DEC_FORM_ONE) {
      rc = dec_one_launch<T, D, MODE>(p, p.batch * p.hkv, dev, stream);
      if (rc) return rc;
    } else if (form == DEC_FORM_CHUNKS) {
      constexpr int LDS = DEC_CHUNK_WAVES * DecLds<D>::BYTES;
      static LdsAllowed allowed;
      if (int rc_ = allow_lds(allowed, (const void*)decode_attn_chunked_kernel<T, D, MODE>, LDS, dev)) return rc_;
      p.chunks[0] = (int)chunks;
      p.stamps = reinterpret_cast<uint64_t*>(p.part + (int64_t)DEC_CHUNK_SLOTS * p0.g * (D + 4));   // behind the partials
      p.call = dec_call_number();
      decode_attn_chunked_kernel<T, D, MODE><<<(int)(pairs * chunks), WAVE * DEC_CHUNK_WAVES, LDS, stream>>>(p);
    } else {
      decode_attn_kernel<T, D, MODE><<<grid, WAVE * wg_waves, DecLds<D>::BYTES * wg_waves, stream>>>(p);
      decode_merge_kernel<T, D, MODE><<<dim3(p.batch, p.hkv), DEC_MERGE_THREADS, 0, stream>>>(p);
    }
    head0 += p.g;
  }
  return 0;
}

template <int MODE>
static int dec_dispatch(int dtype, int head_dim, const DecParams& p, hipStream_t stream) {
  if (dtype == FSA_BF16) {
    if (head_dim == 64) return dec_launch<__bf16, 64, MODE>(p, stream);
    if (head_dim == 128) return dec_launch<__bf16, 128, MODE>(p, stream);
    if (head_dim == 256) return dec_launch<__bf16, 256, MODE>(p, stream);
  } else {
    if (head_dim == 64) return dec_launch<_Float16, 64, MODE>(p, stream);
    if (head_dim == 128) return dec_launch<_Float16, 128, MODE>(p, stream);
    if (head_dim == 256) return dec_launch<_Float16, 256, MODE>(p, stream);
  }
  set_error("decode: head_dim=%d not supported (64, 128, 256)", head_dim);
  return FSA_ERR_UNSUPPORTED;
}

// workspace: tile prefix of the requests, then one partial slot per (wave, pair) that can occur
static size_t dec_ws_prefix_bytes(int batch) { return align_up((size_t)(batch + 1) * 4, 256); }
static size_t dec_ws_bytes(int batch, int hq, int hkv, int d) {
  return dec_ws_prefix_bytes(batch) + ((size_t)DEC_MAX_WAVES + (size_t)batch * hkv) * (hq / hkv) * (4 + d) * 4;
}

// ---- one token through the layer: host side ----
// work-groups per (source, kv head) at most: one for every CU by all kv heads of a source
constexpr int DEC_LAYER_CHUNKS = 64;
static int dec_layer_chunks(int hkv) { return std::min(DEC_LAYER_CHUNKS, std::max(1, 256 / hkv)); }
struct DecLayerWs {
  size_t q_rot, gate, o_cmp, o_win, attn, idx, raw, part, arrived, total;
  int64_t raw_ld;
  int topk;
};
static DecLayerWs dec_layer_ws(const fsa_decode_layer_args& a) {
  DecLayerWs w;
  size_t at = 0;
  auto take = [&](size_t bytes) {
    const size_t p = at;
    at += align_up(bytes, 256);
    return p;
  };
  const size_t row = (size_t)a.num_q_heads * a.head_dim * 2;
  w.q_rot = take(row);
  w.gate = take(16);
  w.o_cmp = take(row);
  w.o_win = take(row);
  w.attn = take(row);
  w.topk = (int)std::min<int64_t>(a.topk, (a.cache_len + a.block_size) / a.block_size);
  w.idx = take((size_t)a.num_kv_heads * w.topk * 4);
  w.raw_ld = (a.ck_len + 1 + 3) / 4 * 4;
  w.raw = take((size_t)a.num_kv_heads * w.raw_ld * 4);
  w.part = take((size_t)2 * dec_layer_chunks(a.num_kv_heads) * a.num_kv_heads * (a.num_q_heads / a.num_kv_heads) * (4 + a.head_dim) * 4);
  w.arrived = take((size_t)2 * a.num_kv_heads * 4);
  w.total = at;
  return w;
}

static int dec_layer_check(const fsa_decode_layer_args* a, bool attend) {
  FSA_CHECK_ARG(a, "fsa_decode_layer: null pointer");
  FSA_CHECK_ARG(a->x && a->w_q && a->w_k && a->w_v && a->w_gate && a->inv_freq && a->k_new && a->v_new && a->workspace,
                "fsa_decode_layer: null pointer");
  FSA_CHECK_ARG(a->dtype == FSA_BF16 || a->dtype == FSA_FP16, "fsa_decode_layer: dtype must be bf16 or fp16");
  FSA_CHECK_ARG(a->head_dim == 64 || a->head_dim == 128 || a->head_dim == 256,
                "fsa_decode_layer: head_dim=%d not supported (64, 128, 256)", a->head_dim);
  FSA_CHECK_ARG(a->num_kv_heads >= 1 && a->num_q_heads % a->num_kv_heads == 0 && a->num_kv_heads <= 1024 &&
                    a->num_q_heads / a->num_kv_heads <= 16,
                "fsa_decode_layer: at most 16 query heads per kv head");
  FSA_CHECK_ARG(a->hidden >= 8 && a->hidden % 8 == 0, "fsa_decode_layer: hidden must be a multiple of 8");
  FSA_CHECK_ARG(a->cache_len >= 1 && a->cache_len < (1 << 30) && a->ck_len >= 0 && a->ck_len <= a->cache_len,
                "fsa_decode_layer: bad cache lengths");
  FSA_CHECK_ARG(a->kernel_stride >= 1 && a->kernel_size % a->kernel_stride == 0 && a->block_size % a->kernel_stride == 0 &&
                    a->block_size >= 1 && a->topk >= 1 && a->window >= 0,
                "fsa_decode_layer: bad layer configuration");
  const int64_t n_ck = a->ck_len + (a->ck_new ? 1 : 0);
  FSA_CHECK_ARG(!attend || (a->w_o && a->y && a->k_cache && a->v_cache && (a->ck_len == 0 || (a->ck_cache && a->cv_cache)) &&
                            n_ck >= 1 && (!a->ck_new || a->cv_new)),
                "fsa_decode_layer: null pointer or no compressed key");
  FSA_CHECK_ARG((a->cache_len + a->block_size) / a->block_size <= 16384, "fsa_decode_layer: more than 16384 blocks");
  if (a->workspace_bytes < dec_layer_ws(*a).total) {
    set_error("fsa_decode_layer: workspace too small (%zu < %zu)", a->workspace_bytes, dec_layer_ws(*a).total);
    return FSA_ERR_WORKSPACE;
  }
  return 0;
}

static DecLayerParams dec_layer_params(const fsa_decode_layer_args& a, const DecLayerWs& w) {
  char* ws = (char*)a.workspace;
  DecLayerParams p = {};
  p.x = a.x;
  p.w[0] = a.w_q; p.w[1] = a.w_k; p.w[2] = a.w_v; p.w[3] = a.w_gate; p.w_o = a.w_o;
  p.hidden = a.hidden; p.hq = a.num_q_heads; p.hkv = a.num_kv_heads; p.d = a.head_dim; p.pos = (int)a.cache_len;
  p.inv_freq = a.inv_freq; p.rope_scale = a.rope_scale;
  p.q_rot = ws + w.q_rot; p.k_new = a.k_new; p.v_new = a.v_new; p.gate = ws + w.gate;
  p.arrived = (int*)(ws + w.arrived);
  p.o_cmp = ws + w.o_cmp; p.o_win = ws + w.o_win; p.attn = ws + w.attn; p.y = a.y;
  return p;
}

template <typename T, int D>
static int dec_layer_attend(const fsa_decode_layer_args& a, hipStream_t stream) {
  const DecLayerWs w = dec_layer_ws(a);
  const DecLayerParams lp = dec_layer_params(a, w);
  char* ws = (char*)a.workspace;
  const int L = (int)a.cache_len, hkv = a.num_kv_heads;
  DecParams p = {};
  p.q = lp.q_rot; p.q_sh = D;
  p.batch = 2; p.hq = a.num_q_heads; p.hkv = hkv; p.g = p.gq = a.num_q_heads / hkv;
  p.block_size = a.block_size; p.topk = w.topk; p.scale_log2 = a.softmax_scale * LOG2E;
  p.raw_score = (float*)(ws + w.raw); p.raw_ld = w.raw_ld; p.part = (float*)(ws + w.part);
  p.topk_idx = (const int32_t*)(ws + w.idx); p.inv_freq = a.inv_freq; p.rope_scale = a.rope_scale;
  const int n_ck = (int)a.ck_len + (a.ck_new ? 1 : 0);
  const int w0 = std::max(0, L - a.window);
  auto elem = [](const void* base, int64_t off) { return (const void*)((const T*)base + off); };
  p.src[0] = {a.ck_cache, a.cv_cache, a.ck_new, a.cv_new, a.ck_stride_n, a.ck_stride_h, a.cv_stride_n, a.cv_stride_h,
              (int)a.ck_len, std::min(n_ck, L >= a.kernel_size - 1 ? (L - a.kernel_size + 1) / a.kernel_stride + 1 : 0), 0,
              a.kernel_stride};
  p.src[1] = {elem(a.k_cache, w0 * a.k_stride_n), elem(a.v_cache, w0 * a.v_stride_n), a.k_new, a.v_new, a.k_stride_n,
              a.k_stride_h, a.v_stride_n, a.v_stride_h, L - w0, L + 1 - w0, w0, 1};
  // a tile per wave, as long as there are work-groups enough
  constexpr int W = DecLayerWaves<D>::N, LDS = W * DecLds<D>::BYTES;
  auto chunks = [&](int tiles) { return std::max(1, std::min((tiles + W - 1) / W, dec_layer_chunks(hkv))); };
  p.arrived = lp.arrived;
  for (int i = 0; i < 2; ++i) p.chunks[i] = chunks((p.src[i].n_keys + DEC_TK - 1) / DEC_TK);

  DecTopkParams tk = {};
  tk.raw_score = p.raw_score; tk.raw_ld = w.raw_ld; tk.batch = 1; tk.hkv = hkv; tk.g = p.g;
  tk.kernel_size = a.kernel_size; tk.kernel_stride = a.kernel_stride; tk.block_size = a.block_size; tk.topk = w.topk;
  tk.init_blocks = a.init_blocks; tk.local_blocks = a.local_blocks; tk.scores_to_bf16 = 1;
  tk.scale_log2 = p.scale_log2; tk.topk_idx = (int32_t*)(ws + w.idx);
  const int nblk = (L + a.block_size) / a.block_size;
  const int grid = (p.chunks[0] + p.chunks[1]) * hkv;
  auto select = [&](auto nreg, size_t lds) {
    constexpr int NREG = decltype(nreg)::value;
    static LdsAllowed allowed;
    if (int rc_ = allow_lds(allowed, (const void*)decode_layer_select_kernel<T, D, NREG>, std::max(LDS, 64 * 1024))) return rc_;
    decode_layer_select_kernel<T, D, NREG><<<grid, WAVE * W, std::max(lds, (size_t)LDS), stream>>>(p, tk, lp);
    return 0;
  };
  int rc;
  if (w.topk <= DEC_TOPK_MAX_K && nblk <= DEC_TOPK_THREADS) rc = select(std::integral_constant<int, 1>{}, 0);
  else if (w.topk <= DEC_TOPK_MAX_K && nblk <= 4 * DEC_TOPK_THREADS) rc = select(std::integral_constant<int, 4>{}, 0);
  else rc = select(std::integral_constant<int, 0>{}, (size_t)nblk * 4);
  if (rc) return rc;

  p.batch = 1;
  p.src[0] = {a.k_cache, a.v_cache, a.k_new, a.v_new, a.k_stride_n, a.k_stride_h, a.v_stride_n, a.v_stride_h, L, L + 1, 0, 1};
  p.chunks[0] = chunks(w.topk * ((a.block_size + DEC_TK - 1) / DEC_TK));
  p.chunks[1] = 0;
  static LdsAllowed allowed;
  if (int rc_ = allow_lds(allowed, (const void*)decode_layer_combine_kernel<T, D>, LDS)) return rc_;
  decode_layer_combine_kernel<T, D><<<p.chunks[0] * hkv, WAVE * W, LDS, stream>>>(p, lp);
  decode_out_kernel<T><<<(a.hidden + 7) / 8, 256, 0, stream>>>(lp);
  FSA_CHECK_LAUNCH("fsa_decode_layer_attend");
  return 0;
}

// Scratch memory of fsa_decode_selattn_static: lives in the code object, one copy per device that loads it, for
// as long as the process runs.  In host code the array's name is only a handle for hipGetSymbolAddress.
constexpr size_t DEC_STATIC_SCRATCH_BYTES = (size_t)FSA_DECODE_STATIC_SCRATCH_BYTES;
static __device__ __align__(256) unsigned char dec_static_scratch[DEC_STATIC_SCRATCH_BYTES];

// Per-device state of the scratch array: its device address (looked up once), and the stream and completion
// event of the last call that used it.
struct DecStaticState {
  void* ptr = nullptr;
  hipEvent_t done = nullptr;
  hipStream_t last_stream = nullptr;
  bool used = false;
};
constexpr int DEC_STATIC_MAX_DEV = 64;
static DecStaticState dec_static_state[DEC_STATIC_MAX_DEV];
static std::mutex dec_static_mu;

// Set-up for one call on `stream`: the scratch address of the current device, and - the array is shared by every
// call on the device - an ordering edge behind the previous call when that one ran on another stream
// (hipStreamWaitEvent on its completion event; nothing is allocated per call, the event is created once per
// device).  Calls recorded into a graph take no part in this: a capturing stream may neither wait for nor record
// an event of eager work, so captured calls are ordered by the graph's own dependencies.
static int dec_static_begin(hipStream_t stream, void** out, bool* capturing) {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) {
    set_error("fsa_decode_selattn_static: hipGetDevice: %s", hipGetErrorString(e));
    return (int)e;
  }
  if (dev < 0 || dev >= DEC_STATIC_MAX_DEV) {
    set_error("fsa_decode_selattn_static: device %d out of range", dev);
    return FSA_ERR_UNSUPPORTED;
  }
  hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(stream, &cs) != hipSuccess) {
    (void)hipGetLastError();
    cs = hipStreamCaptureStatusNone;
  }
  *capturing = cs != hipStreamCaptureStatusNone;
  std::lock_guard<std::mutex> lock(dec_static_mu);
  DecStaticState& st = dec_static_state[dev];
  if (!st.ptr) {
    void* a = nullptr;
    e = hipGetSymbolAddress(&a, HIP_SYMBOL(dec_static_scratch));
    if (e != hipSuccess || !a) {
      set_error("fsa_decode_selattn_static: hipGetSymbolAddress: %s", hipGetErrorString(e));
      return e != hipSuccess ? (int)e : FSA_ERR_UNSUPPORTED;
    }
    st.ptr = a;
  }
  *out = st.ptr;
  if (*capturing) return 0;
  if (!st.done) {
    e = hipEventCreateWithFlags(&st.done, hipEventDisableTiming);
    if (e != hipSuccess) {
      set_error("fsa_decode_selattn_static: hipEventCreateWithFlags: %s", hipGetErrorString(e));
      return (int)e;
    }
  }
  if (st.used && st.last_stream != stream) {
    e = hipStreamWaitEvent(stream, st.done, 0);
    if (e != hipSuccess) {
      set_error("fsa_decode_selattn_static: hipStreamWaitEvent: %s", hipGetErrorString(e));
      return (int)e;
    }
  }
  return 0;
}

// After the kernels of an eager call are enqueued: remember its stream and mark its end.
static int dec_static_end(hipStream_t stream) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= DEC_STATIC_MAX_DEV) return 0;
  std::lock_guard<std::mutex> lock(dec_static_mu);
  DecStaticState& st = dec_static_state[dev];
  if (!st.done) return 0;
  hipError_t e = hipEventRecord(st.done, stream);
  if (e != hipSuccess) {
    set_error("fsa_decode_selattn_static: hipEventRecord: %s", hipGetErrorString(e));
    return (int)e;
  }
  st.last_stream = stream;
  st.used = true;
  return 0;
}

}  // namespace fsa

using namespace fsa;

extern "C" size_t fsa_decode_workspace_bytes(int32_t batch, int32_t num_q_heads, int32_t num_kv_heads,
                                             int32_t head_dim, int64_t max_keys) {
  if (batch < 1 || num_kv_heads < 1 || num_q_heads % num_kv_heads || max_keys < 0) return 0;
  return dec_ws_bytes(batch, num_q_heads, num_kv_heads, head_dim);
}

extern "C" int fsa_decode_cmpattn(const void* q, const void* ck, const void* cv, int32_t dtype,
                                  int64_t q_stride_b, int64_t q_stride_h, int64_t k_stride_n,
                                  int64_t k_stride_h, int64_t v_stride_n, int64_t v_stride_h,
                                  const int32_t* cu_ck, const int32_t* pos, int32_t batch,
                                  int32_t num_q_heads, int32_t num_kv_heads, int32_t head_dim,
                                  int32_t kernel_size, int32_t kernel_stride, float softmax_scale,
                                  int32_t score_head_as_written, int64_t max_keys, void* o, float* lse,
                                  float* raw_score, int64_t raw_ld, void* workspace, size_t workspace_bytes,
                                  void* stream_) {
  FSA_CHECK_ARG(q && ck && cv && cu_ck && pos && o && lse, "fsa_decode_cmpattn: null pointer");
  FSA_CHECK_ARG(dtype == FSA_BF16 || dtype == FSA_FP16, "fsa_decode_cmpattn: dtype must be bf16 or fp16");
  FSA_CHECK_ARG(num_kv_heads >= 1 && num_q_heads % num_kv_heads == 0,
                "fsa_decode_cmpattn: num_q_heads must be a multiple of num_kv_heads");
  const int g = num_q_heads / num_kv_heads;
  FSA_CHECK_ARG(max_keys >= 0 && max_keys < (1ll << 30), "fsa_decode_cmpattn: bad max_keys");
  FSA_CHECK_ARG(workspace && workspace_bytes >= dec_ws_bytes(batch, num_q_heads, num_kv_heads, head_dim),
                "fsa_decode_cmpattn: workspace too small (see fsa_decode_workspace_bytes)");
  FSA_CHECK_ARG(batch >= 1 && kernel_size >= 1 && kernel_stride >= 1, "fsa_decode_cmpattn: bad sizes");
  FSA_CHECK_ARG(!raw_score || (raw_ld >= 4 && raw_ld % 4 == 0), "fsa_decode_cmpattn: raw_ld must be a multiple of 4");
  FSA_CHECK_ARG(!score_head_as_written || num_kv_heads <= num_q_heads, "fsa_decode_cmpattn: bad scoring head");
  DecParams p = {};
  p.q = q; p.k = ck; p.v = cv; p.q_sb = q_stride_b; p.q_sh = q_stride_h;
  p.k_sn = k_stride_n; p.k_sh = k_stride_h; p.v_sn = v_stride_n; p.v_sh = v_stride_h;
  p.cu_k = cu_ck; p.pos = pos; p.batch = batch; p.hq = num_q_heads; p.hkv = num_kv_heads; p.g = g;
  p.kernel_size = kernel_size; p.kernel_stride = kernel_stride; p.scale_log2 = softmax_scale * LOG2E;
  p.o = o; p.lse = lse; p.raw_score = raw_score; p.raw_ld = raw_ld;
  p.score_head_as_written = score_head_as_written;
  p.tile_prefix = (int32_t*)workspace; p.part = (float*)((char*)workspace + dec_ws_prefix_bytes(batch));
  p.max_keys = (int)max_keys;
  int rc = dec_dispatch<DEC_MODE_COMPRESSED>(dtype, head_dim, p, (hipStream_t)stream_);
  if (rc) return rc;
  FSA_CHECK_LAUNCH("fsa_decode_cmpattn");
  return 0;
}

extern "C" int fsa_decode_topk(const float* raw_score, int64_t raw_ld, const float* lse,
                               const int32_t* cu_ck, const int32_t* pos, const int32_t* seqlens,
                               int32_t batch, int32_t num_q_heads, int32_t num_kv_heads,
                               int32_t kernel_size, int32_t kernel_stride, int32_t block_size,
                               int32_t topk, int32_t init_blocks, int32_t local_blocks,
                               int32_t as_written, int32_t scores_to_bf16, float softmax_scale,
                               int64_t max_blocks, int32_t* topk_idx, float* block_score, void* stream_) {
  hipStream_t stream = (hipStream_t)stream_;
  FSA_CHECK_ARG(raw_score && lse && cu_ck && pos && seqlens && topk_idx, "fsa_decode_topk: null pointer");
  FSA_CHECK_ARG(batch >= 1 && topk >= 1 && num_kv_heads >= 1 && num_q_heads % num_kv_heads == 0,
                "fsa_decode_topk: bad sizes");
  FSA_CHECK_ARG(kernel_stride >= 1 && kernel_size % kernel_stride == 0 && block_size % kernel_stride == 0,
                "fsa_decode_topk: kernel_size and block_size must be multiples of kernel_stride");
  FSA_CHECK_ARG(max_blocks >= 1 && max_blocks * 4 <= 64 * 1024,
                "fsa_decode_topk: max_blocks must be in [1, 16384]");
  DecTopkParams p = {};
  p.raw_score = raw_score; p.raw_ld = raw_ld; p.lse = lse; p.cu_ck = cu_ck; p.pos = pos; p.seqlens = seqlens;
  p.batch = batch; p.hkv = num_kv_heads; p.g = num_q_heads / num_kv_heads;
  p.kernel_size = kernel_size; p.kernel_stride = kernel_stride; p.block_size = block_size; p.topk = topk;
  p.init_blocks = init_blocks; p.local_blocks = local_blocks; p.as_written = as_written;
  p.scores_to_bf16 = scores_to_bf16;
  p.scale_log2 = softmax_scale * LOG2E; p.topk_idx = topk_idx; p.block_score = block_score;
  p.score_ld = max_blocks;
  {
    ProfScope ps_("decode_topk", stream);
    const dim3 grid(batch, num_kv_heads);
    if (topk <= DEC_TOPK_MAX_K && max_blocks <= 1 * DEC_TOPK_THREADS) decode_topk_kernel<1><<<grid, DEC_TOPK_THREADS, 0, stream>>>(p);
    else if (topk <= DEC_TOPK_MAX_K && max_blocks <= 4 * DEC_TOPK_THREADS) decode_topk_kernel<4><<<grid, DEC_TOPK_THREADS, 0, stream>>>(p);
    else if (topk <= DEC_TOPK_MAX_K && max_blocks <= 8 * DEC_TOPK_THREADS) decode_topk_kernel<8><<<grid, DEC_TOPK_THREADS, 0, stream>>>(p);
    else decode_topk_kernel<0><<<grid, DEC_TOPK_THREADS, (size_t)max_blocks * 4, stream>>>(p);
  }
  FSA_CHECK_LAUNCH("fsa_decode_topk");
  return 0;
}

extern "C" int fsa_decode_selattn(const void* q, const void* k_cache, const void* v_cache, int32_t dtype,
                                  int64_t q_stride_b, int64_t q_stride_h, int64_t k_stride_n,
                                  int64_t k_stride_h, int64_t v_stride_n, int64_t v_stride_h,
                                  const int32_t* cu_k, const int32_t* seqlens, const int32_t* topk_idx,
                                  int32_t batch, int32_t num_q_heads, int32_t num_kv_heads, int32_t head_dim,
                                  int32_t topk, int32_t block_size, float softmax_scale, void* o,
                                  float* lse, void* workspace, size_t workspace_bytes, void* stream_) {
  FSA_CHECK_ARG(q && k_cache && v_cache && cu_k && topk_idx && o && lse, "fsa_decode_selattn: null pointer");
  FSA_CHECK_ARG(dtype == FSA_BF16 || dtype == FSA_FP16, "fsa_decode_selattn: dtype must be bf16 or fp16");
  FSA_CHECK_ARG(num_kv_heads >= 1 && num_q_heads % num_kv_heads == 0,
                "fsa_decode_selattn: num_q_heads must be a multiple of num_kv_heads");
  FSA_CHECK_ARG(batch >= 1 && topk >= 1 && block_size >= 1, "fsa_decode_selattn: bad sizes");
  FSA_CHECK_ARG(workspace && workspace_bytes >= dec_ws_bytes(batch, num_q_heads, num_kv_heads, head_dim),
                "fsa_decode_selattn: workspace too small (see fsa_decode_workspace_bytes)");
  DecParams p = {};
  p.q = q; p.k = k_cache; p.v = v_cache; p.q_sb = q_stride_b; p.q_sh = q_stride_h;
  p.k_sn = k_stride_n; p.k_sh = k_stride_h; p.v_sn = v_stride_n; p.v_sh = v_stride_h;
  p.cu_k = cu_k; p.seqlens = seqlens; p.topk_idx = topk_idx; p.batch = batch; p.hq = num_q_heads;
  p.hkv = num_kv_heads; p.g = num_q_heads / num_kv_heads; p.topk = topk; p.block_size = block_size;
  p.scale_log2 = softmax_scale * LOG2E; p.o = o; p.lse = lse;
  p.tile_prefix = (int32_t*)workspace; p.part = (float*)((char*)workspace + dec_ws_prefix_bytes(batch));
  int rc = dec_dispatch<DEC_MODE_SELECTED>(dtype, head_dim, p, (hipStream_t)stream_);
  if (rc) return rc;
  FSA_CHECK_LAUNCH("fsa_decode_selattn");
  return 0;
}

extern "C" int fsa_decode_selattn_static(const void* q, const void* k_cache, const void* v_cache, int32_t dtype,
                                         int64_t q_stride_b, int64_t q_stride_h, int64_t k_stride_n,
                                         int64_t k_stride_h, int64_t v_stride_n, int64_t v_stride_h,
                                         const int32_t* cu_k, const int32_t* seqlens, const int32_t* topk_idx,
                                         int32_t batch, int32_t num_q_heads, int32_t num_kv_heads, int32_t head_dim,
                                         int32_t topk, int32_t block_size, float softmax_scale, void* o,
                                         float* lse, void* stream_) {
  FSA_CHECK_ARG(batch >= 1 && num_kv_heads >= 1 && num_q_heads >= 1 && num_q_heads % num_kv_heads == 0 &&
                    head_dim >= 1,
                "fsa_decode_selattn_static: bad sizes");
  const size_t need = dec_ws_bytes(batch, num_q_heads, num_kv_heads, head_dim);
  if (need > DEC_STATIC_SCRATCH_BYTES) {
    set_error("fsa_decode_selattn_static: batch %d x %d kv heads x %d heads per group x head_dim %d needs %zu bytes "
              "of scratch, the built-in buffer holds %zu; use fsa_decode_selattn with a caller workspace",
              batch, num_kv_heads, num_q_heads / num_kv_heads, head_dim, need, DEC_STATIC_SCRATCH_BYTES);
    return FSA_ERR_WORKSPACE;
  }
  void* scratch = nullptr;
  bool capturing = false;
  int rc = dec_static_begin((hipStream_t)stream_, &scratch, &capturing);
  if (rc) return rc;
  // every partial slot that the merge reads is written by the attention kernel of the same call: nothing in the
  // buffer has to start at zero
  rc = fsa_decode_selattn(q, k_cache, v_cache, dtype, q_stride_b, q_stride_h, k_stride_n, k_stride_h, v_stride_n,
                          v_stride_h, cu_k, seqlens, topk_idx, batch, num_q_heads, num_kv_heads, head_dim, topk, block_size,
                          softmax_scale, o, lse, scratch, DEC_STATIC_SCRATCH_BYTES, stream_);
  if (rc || capturing) return rc;
  return dec_static_end((hipStream_t)stream_);
}

extern "C" size_t fsa_decode_layer_workspace_bytes(const fsa_decode_layer_args* args) {
  if (!args || args->num_kv_heads < 1 || args->block_size < 1) return 0;
  return dec_layer_ws(*args).total;
}

extern "C" int fsa_decode_layer_project(const fsa_decode_layer_args* args, void* stream_) {
  hipStream_t stream = (hipStream_t)stream_;
  if (int rc = dec_layer_check(args, false)) return rc;
  const DecLayerParams p = dec_layer_params(*args, dec_layer_ws(*args));
  const int units = (args->num_q_heads + 2 * args->num_kv_heads) * (args->head_dim / 2) + 3;
  ProfScope ps_("decode_layer_project", stream);
  if (args->dtype == FSA_BF16) decode_project_kernel<__bf16><<<(units + 3) / 4, 256, 0, stream>>>(p);
  else decode_project_kernel<_Float16><<<(units + 3) / 4, 256, 0, stream>>>(p);
  FSA_CHECK_LAUNCH("fsa_decode_layer_project");
  return 0;
}

extern "C" int fsa_decode_layer_attend(const fsa_decode_layer_args* args, void* stream_) {
  hipStream_t stream = (hipStream_t)stream_;
  if (int rc = dec_layer_check(args, true)) return rc;
  ProfScope ps_("decode_layer_attend", stream);
  const bool bf = args->dtype == FSA_BF16;
  if (args->head_dim == 64) return bf ? dec_layer_attend<__bf16, 64>(*args, stream) : dec_layer_attend<_Float16, 64>(*args, stream);
  if (args->head_dim == 128) return bf ? dec_layer_attend<__bf16, 128>(*args, stream) : dec_layer_attend<_Float16, 128>(*args, stream);
  return bf ? dec_layer_attend<__bf16, 256>(*args, stream) : dec_layer_attend<_Float16, 256>(*args, stream);
}
