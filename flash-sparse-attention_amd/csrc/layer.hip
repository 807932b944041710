// The attention core of the layer as two calls (gfx950): everything between the projections of q, k, v and the output
// projection, forward and backward.
//
//   layer_prep        : cu_seqlens of the compressed keys, cos / sin table of all positions, gates sigmoid(x w_gate^T)
//   rope_segments     : rotation of q, k and the compressed keys in one launch, angles from the table
//   merge_stats       : backward of the gated sum without its outputs (below)
//   gate_bwd          : d w_gate and the gate's share of dx
//   kv_combine        : dk / dv of the branches added, dk rotated back
//
// The backward needs no gradient tensor per branch: with out = sum_i g_i o_i, branch i sees dO_i = g_i d_out, hence
// dS_i = g_i P_i (d_out V^T - delta_i) with delta_i = d_out . o_i, and g_i P_i is the probability taken relative to
// lse_i - log2 g_i.  So every branch runs its unchanged backward kernels on d_out itself with the pairs
// (lse_i - log2 g_i, delta_i): three tensors are neither written nor read, and the delta kernels are gone, because
// delta_i is what the gate's own gradient sums up.  (32K tokens x 32 heads of 128: 650 us of launches before.)
//
// Semantics: fsa/module/fsa.py:92-173.
#include "fsa_common.h"

#include <algorithm>

namespace fsa {

// ------------------------------------------------- tables and gates ----
// gate[n, i] = sigmoid(x[n] . w[i]), i < 3.  A wave takes four tokens, so that the three weight rows are fetched once for
// them; bound by the bytes of x.  (The product as a GEMM with three output columns runs at a third of that rate.)
constexpr int GATE_TOK = 4;
template <typename T>
__device__ __forceinline__ void gate_fwd(const T* __restrict__ x, const T* __restrict__ w, T* __restrict__ gate, int64_t n,
                                         int hidden, int64_t block) {
  typedef typename Elem<T>::vec8 vec8;
  const int lane = threadIdx.x & (WAVE - 1);
  const int64_t t0 = (block * 4 + threadIdx.x / WAVE) * GATE_TOK;
  if (t0 >= n) return;
  float s[GATE_TOK][3] = {};
  for (int e = lane * 8; e < hidden; e += 512) {
    vec8 a[GATE_TOK], b[3];
#pragma unroll
    for (int t = 0; t < GATE_TOK; ++t) a[t] = load16<vec8>(x + min(t0 + t, n - 1) * hidden + e);
#pragma unroll
    for (int i = 0; i < 3; ++i) b[i] = load16<vec8>(w + (int64_t)i * hidden + e);
#pragma unroll
    for (int t = 0; t < GATE_TOK; ++t)
#pragma unroll
      for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 8; ++j) s[t][i] += (float)a[t][j] * (float)b[i][j];
  }
#pragma unroll
  for (int t = 0; t < GATE_TOK; ++t)
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      float v = s[t][i];
#pragma unroll
      for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o, WAVE);
      if (lane == 0 && t0 + t < n) gate[(t0 + t) * 3 + i] = (T)(1.f / (1.f + expf(-(float)(T)v)));
    }
}

// What needs nothing but the arguments, in one launch: cu_ck (work-group 0), the gates, and
// table[pos][D/2] = (cos, sin) of pos * inv_freq, scaled, in the tensor's type.
template <typename T>
__global__ void __launch_bounds__(256)
layer_prep_kernel(const int32_t* __restrict__ cu, int batch, int ks, int stride, int32_t* __restrict__ cu_ck,
                  const float* __restrict__ inv_freq, float scale, int half, int64_t n_pairs, T* __restrict__ table,
                  const T* __restrict__ x, const T* __restrict__ w_gate, T* __restrict__ gate, int64_t n, int hidden) {
  const int64_t gate_blocks = (n + 4 * GATE_TOK - 1) / (4 * GATE_TOK);
  if (blockIdx.x == 0) {
    __shared__ int wave_total[4];
    const int tid = threadIdx.x, lane = tid & (WAVE - 1), w = tid / WAVE;
    int base = 0;
    for (int s0 = 0; s0 < batch; s0 += 256) {
      const int s = s0 + tid, len = s < batch ? cu[s + 1] - cu[s] : 0;
      int inc = len >= ks ? (len - ks) / stride + 1 : 0;
#pragma unroll
      for (int o = 1; o < WAVE; o <<= 1) {
        const int x_ = __shfl_up(inc, o, WAVE);
        if (lane >= o) inc += x_;
      }
      if (lane == WAVE - 1) wave_total[w] = inc;
      __syncthreads();
      int total = 0;
      for (int ww = 0; ww < 4; ++ww) {
        if (ww == w) inc += total;
        total += wave_total[ww];
      }
      if (s < batch) cu_ck[s + 1] = base + inc;
      base += total;
      __syncthreads();
    }
    if (tid == 0) cu_ck[0] = 0;
    return;
  }
  if (blockIdx.x <= gate_blocks) return gate_fwd<T>(x, w_gate, gate, n, hidden, blockIdx.x - 1);
  const int64_t i = (int64_t)(blockIdx.x - 1 - gate_blocks) * 256 + threadIdx.x;
  if (i >= n_pairs) return;
  const int pos = (int)(i / half), d = (int)(i - (int64_t)pos * half);
  float sn, cs;
  sincosf((float)pos * inv_freq[d], &sn, &cs);
  table[2 * i] = (T)(cs * scale);
  table[2 * i + 1] = (T)(sn * scale);
}

struct RopeSegment {
  const void* x;
  void* out;
  const int32_t* cu;
  int64_t n;         // tokens
  int heads, step;   // token j of a sequence sits at position j * step
};
struct RopeSegments {
  RopeSegment seg[3];
  int batch;
};

// One wave per token: D/16 lanes cover a head (8 dims of the first half and their partners), all tensors [n, heads, D]
// contiguous.  Bound by the bytes of x and out.
template <typename T, int D>
__global__ void __launch_bounds__(256)
rope_segments_kernel(RopeSegments p, const T* __restrict__ table, int inverse) {
  typedef typename Elem<T>::vec8 vec8;
  constexpr int LPR = D / 16, HPW = WAVE / LPR;
  int64_t tok = (int64_t)blockIdx.x * 4 + threadIdx.x / WAVE;
  int k = 0;
  while (k < 2 && tok >= (p.seg[k].n + 3) / 4 * 4) {   // segments start at multiples of four tokens: uniform per work-group
    tok -= (p.seg[k].n + 3) / 4 * 4;
    ++k;
  }
  const RopeSegment g = p.seg[k];
  if (tok >= g.n) return;
  const int lane = threadIdx.x & (WAVE - 1), sub = lane % LPR, hl = lane / LPR;
  const int s = upper_seg(g.cu, p.batch, (int)tok);
  const int64_t pos = (tok - g.cu[s]) * g.step;
  const T* cs = table + pos * D + sub * 16;
  const vec8 c0 = load16<vec8>(cs), c1 = load16<vec8>(cs + 8);
  float c[8], sn[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    c[e] = (float)(e < 4 ? c0[2 * e] : c1[2 * e - 8]);
    sn[e] = (float)(e < 4 ? c0[2 * e + 1] : c1[2 * e - 7]);
    if (inverse) sn[e] = -sn[e];
  }
  const T* x = reinterpret_cast<const T*>(g.x) + tok * g.heads * D + sub * 8;
  T* out = reinterpret_cast<T*>(g.out) + tok * g.heads * D + sub * 8;
#pragma unroll 4
  for (int head = hl; head < g.heads; head += HPW) {
    const vec8 a = load16<vec8>(x + head * D), b = load16<vec8>(x + head * D + D / 2);
    vec8 oa, ob;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float x1 = (float)a[e], x2 = (float)b[e];
      oa[e] = (T)(x1 * c[e] - x2 * sn[e]);
      ob[e] = (T)(x1 * sn[e] + x2 * c[e]);
    }
    store16(out + head * D, oa);
    store16(out + head * D + D / 2, ob);
  }
}

// ------------------------------------------------------------------ gate ----
// d w[i] = sum_n dl[n, i] x[n] (partial per chunk of tokens, fp32) and dx[n] = sum_i dl[n, i] w[i] in one pass over x.
// A thread owns eight columns for all tokens of the chunk.  Bound by reading x and writing dx.
constexpr int GATE_COLS = 2048;   // columns per work-group
template <typename T>
__global__ void __launch_bounds__(256)
gate_bwd_kernel(const T* __restrict__ x, const T* __restrict__ w, const T* __restrict__ dl, T* __restrict__ dx,
                float* __restrict__ part, int64_t n, int hidden, int chunk) {
  typedef typename Elem<T>::vec8 vec8;
  extern __shared__ float dls[];   // [chunk][3]
  const int64_t t0 = (int64_t)blockIdx.x * chunk;
  const int nt = (int)min((int64_t)chunk, n - t0);
  for (int i = threadIdx.x; i < nt * 3; i += 256) dls[i] = (float)dl[t0 * 3 + i];
  __syncthreads();
  const int col = blockIdx.y * GATE_COLS + threadIdx.x * 8;
  if (col >= hidden) return;
  float wf[3][8], acc[3][8];
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    const vec8 v = load16<vec8>(w + (int64_t)i * hidden + col);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      wf[i][j] = (float)v[j];
      acc[i][j] = 0.f;
    }
  }
  const T* xp = x + t0 * hidden + col;
  constexpr int U = 4;
  for (int tb = 0; tb < nt; tb += U) {
    vec8 xs[U];
#pragma unroll
    for (int u = 0; u < U; ++u) xs[u] = load16<vec8>(xp + (int64_t)min(tb + u, nt - 1) * hidden);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (tb + u < nt) {
        const float d0 = dls[(tb + u) * 3], d1 = dls[(tb + u) * 3 + 1], d2 = dls[(tb + u) * 3 + 2];
        vec8 o;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const float xf = (float)xs[u][j];
          acc[0][j] += d0 * xf;
          acc[1][j] += d1 * xf;
          acc[2][j] += d2 * xf;
          o[j] = (T)(d0 * wf[0][j] + d1 * wf[1][j] + d2 * wf[2][j]);
        }
        if (dx) store16(dx + (t0 + tb + u) * hidden + col, o);
      }
    }
  }
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    float* pp = part + ((int64_t)blockIdx.x * 3 + i) * hidden + col;
    *reinterpret_cast<f32x4*>(pp) = f32x4{acc[i][0], acc[i][1], acc[i][2], acc[i][3]};
    *reinterpret_cast<f32x4*>(pp + 4) = f32x4{acc[i][4], acc[i][5], acc[i][6], acc[i][7]};
  }
}

// dw = sum of the chunks' partials: 64 columns per work-group, the chunks shared out over its four waves, fixed order
template <typename T>
__global__ void __launch_bounds__(256)
gate_dw_kernel(const float* __restrict__ part, T* __restrict__ dw, int64_t cols, int chunks) {
  __shared__ float quarter[3][WAVE];
  const int lane = threadIdx.x & (WAVE - 1), wv = threadIdx.x / WAVE;
  const int64_t c = (int64_t)blockIdx.x * WAVE + lane;
  const int per = (chunks + 3) / 4, lo = wv * per, hi = min(chunks, lo + per);
  float s = 0.f;
  if (c < cols) {
#pragma unroll 8
    for (int i = lo; i < hi; ++i) s += part[(int64_t)i * cols + c];
  }
  if (wv > 0) quarter[wv - 1][lane] = s;
  __syncthreads();
  if (wv == 0 && c < cols) dw[c] = (T)(((s + quarter[0][lane]) + quarter[1][lane]) + quarter[2][lane]);
}

// ------------------------------------------------------------ merge, backward ----
struct MergeStats {
  const void *d_out, *o[3];      // [N, Hq, D]
  const void* gate;              // [N, 3]
  const float* lse[3];           // [Hq, N]
  float2* stat[3];               // [N, Hq] (lse - log2 gate, delta); lse +inf where the row has no probability at all
  void* dl;                      // [N, 3] gradient of the gate's logits
  int64_t n;
  int hq;
};
// One wave per token, D/8 lanes per head; bound by reading the four tensors.
template <typename T, int D>
__global__ void __launch_bounds__(256)
merge_stats_kernel(MergeStats p) {
  typedef typename Elem<T>::vec8 vec8;
  constexpr int LPR = D / 8, HPS = WAVE / LPR;   // heads per 512-element step
  const int64_t n = (int64_t)blockIdx.x * 4 + threadIdx.x / WAVE;
  if (n >= p.n) return;
  const int lane = threadIdx.x & (WAVE - 1), sub = lane % LPR, hl = lane / LPR;
  const int64_t base = n * p.hq * D + sub * 8;
  float g[3], lg[3], dg[3] = {0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    g[i] = (float)reinterpret_cast<const T*>(p.gate)[n * 3 + i];
    lg[i] = log2f(g[i]);
  }
  for (int h0 = 0; h0 < p.hq; h0 += HPS) {
    const int h = h0 + hl;
    const bool live = h < p.hq;
    const int hc = live ? h : p.hq - 1;
    const vec8 d = load16_stream<vec8>(reinterpret_cast<const T*>(p.d_out) + base + hc * D);
    vec8 o[3];
#pragma unroll
    for (int i = 0; i < 3; ++i) o[i] = load16_stream<vec8>(reinterpret_cast<const T*>(p.o[i]) + base + hc * D);
    float s[3] = {0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < 3; ++i) {
#pragma unroll
      for (int e = 0; e < 8; ++e) s[i] += (float)d[e] * (float)o[i][e];
#pragma unroll
      for (int off = LPR / 2; off >= 1; off >>= 1) s[i] += __shfl_xor(s[i], off, LPR);
      if (live) dg[i] += s[i];
    }
    if (live && sub < 3) {   // three lanes of the head store one pair each
      const float delta = sub == 0 ? s[0] : sub == 1 ? s[1] : s[2];
      const float* lse = sub == 0 ? p.lse[0] : sub == 1 ? p.lse[1] : p.lse[2];
      const float l = sub == 0 ? lg[0] : sub == 1 ? lg[1] : lg[2];
      float2* st = sub == 0 ? p.stat[0] : sub == 1 ? p.stat[1] : p.stat[2];
      // No visible key (lse -inf) or a gate that is zero (l -inf): +inf, every probability 0.  The difference of the two
      // where both hold would be NaN.
      const float lse_h = lse[(int64_t)h * p.n + n];
      st[n * p.hq + h] = make_float2(lse_h == -INFINITY || l == -INFINITY ? INFINITY : lse_h - l, delta);
    }
  }
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    // every lane of a head holds the head's sum: add over the head groups only
#pragma unroll
    for (int off = 32; off >= LPR; off >>= 1) dg[i] += __shfl_xor(dg[i], off, WAVE);
    if (lane == 0) reinterpret_cast<T*>(p.dl)[n * 3 + i] = (T)((float)(T)dg[i] * (1.f - g[i]) * g[i]);
  }
}

// dk = R^-1 (dk_a + dk_b) + dk_c and dv = dv_a + dv_b + dv_c, D/8 lanes per row
struct KvCombine {
  const void *dk[3], *dv[3];
  void *dk_out, *dv_out;
  const void* table;
  const int32_t* cu;
  int batch, heads;
  int64_t n;
};
template <typename T, int D>
__global__ void __launch_bounds__(256)
kv_combine_kernel(KvCombine p) {
  typedef typename Elem<T>::vec8 vec8;
  constexpr int LPR = D / 8, RPB = 256 / LPR;
  const int64_t R = (int64_t)blockIdx.x * RPB + threadIdx.x / LPR;
  if (R >= p.n * p.heads) return;
  const int sub = threadIdx.x % LPR;
  const int64_t tok = R / p.heads, at = R * D + sub * 8;
  auto ld = [&](const void* x) { return load16_stream<vec8>(reinterpret_cast<const T*>(x) + at); };
  const vec8 a = ld(p.dk[0]), b = ld(p.dk[1]), c = ld(p.dk[2]), x = ld(p.dv[0]), y = ld(p.dv[1]), z = ld(p.dv[2]);
  const int s = upper_seg(p.cu, p.batch, (int)tok);
  const T* cs = reinterpret_cast<const T*>(p.table) + (tok - p.cu[s]) * D + (sub % (LPR / 2)) * 16;
  const vec8 c0 = load16<vec8>(cs), c1 = load16<vec8>(cs + 8);
  const float sign = sub < LPR / 2 ? 1.f : -1.f;
  vec8 k, v;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const float own = (float)a[e] + (float)b[e];
    const float other = __shfl_xor(own, LPR / 2, LPR);
    const float cc = (float)(e < 4 ? c0[2 * e] : c1[2 * e - 8]), sn = (float)(e < 4 ? c0[2 * e + 1] : c1[2 * e - 7]);
    k[e] = (T)(own * cc + sign * (other * sn) + (float)c[e]);
    v[e] = (T)((float)x[e] + (float)y[e] + (float)z[e]);
  }
  store16(reinterpret_cast<T*>(p.dk_out) + at, k);
  store16(reinterpret_cast<T*>(p.dv_out) + at, v);
}

// `chunks` times eight 16-bit elements from an address that is aligned to one element only
__global__ void __launch_bounds__(256) copy_aligned_kernel(const uint16_t* __restrict__ src, void* __restrict__ dst, int64_t chunks) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= chunks) return;
  uint32_t x[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) x[e] = src[8 * i + 2 * e] | (uint32_t)src[8 * i + 2 * e + 1] << 16;
  reinterpret_cast<uint4*>(dst)[i] = make_uint4(x[0], x[1], x[2], x[3]);
}

// -------------------------------------------------------------- host side ----
struct Bump {
  size_t at = 0;
  size_t take(size_t bytes) {
    const size_t p = at;
    at += align_up(bytes, 256);
    return p;
  }
};

// What the forward keeps for the backward.
struct LayerSaved {
  size_t cu_ck, table, gates, q, k, ck, cv, o[3], lse[3], cu_blocks, counts, starts, sel, slot, tiles_fwd, tiles_bwd, total;
  int64_t max_blocks;
  int t_out;
  bool direct, index;   // selected forward from the block lists; whether the inverted index is built
};
static LayerSaved layer_saved(const fsa_layer_args& a) {
  LayerSaved s;
  Bump b;
  const size_t e = 2, n = a.total_tokens, d = a.head_dim, hq = a.num_q_heads, hkv = a.num_kv_heads;
  s.t_out = (int)std::min<int64_t>(a.topk, (a.max_len + a.block_size - 1) / a.block_size);
  s.max_blocks = (a.total_tokens + a.block_size - 1) / a.block_size + a.batch;
  // sequences of unknown lengths are priced as in the operator: three quarters of the batch as one
  const int64_t len = a.batch > 1 && a.max_len == a.total_tokens ? a.max_len - a.max_len / 4 : a.max_len;
  s.direct = a.total_tokens * a.num_kv_heads * a.head_dim < (int64_t)1 << 30 && a.max_len <= (int64_t)a.block_size * DIR_MAX_BLOCKS &&
             selattn_direct_preferred(a.total_tokens, len, a.num_q_heads, a.head_dim, s.t_out, a.block_size, !a.inference);
  s.index = !s.direct || !a.inference;
  s.cu_ck = b.take((a.batch + 1) * 4);
  s.table = b.take((size_t)a.max_len * d * e);
  s.gates = b.take(n * 3 * e);
  s.q = b.take(n * hq * d * e);
  s.k = b.take(n * hkv * d * e);
  s.ck = b.take((size_t)a.total_ck * hkv * d * e);
  s.cv = b.take((size_t)a.total_ck * hkv * d * e);
  // (inference: the selected branch goes into the gated sum without being stored, and nothing asks for the backward's tiles)
  for (int i = 0; i < 3; ++i) s.o[i] = b.take(a.inference && i == 1 ? 0 : n * hq * d * e);
  for (int i = 0; i < 3; ++i) s.lse[i] = b.take(a.inference && i == 1 ? 0 : n * hq * 4);
  s.cu_blocks = b.take((a.batch + 1) * 4);
  s.counts = b.take(!s.index ? 0 : hkv * s.max_blocks * 4);
  s.starts = b.take(!s.index ? 0 : hkv * (s.max_blocks + 1) * 4);
  s.sel = b.take(!s.index ? 0 : hkv * n * s.t_out * 4);
  s.slot = b.take(!s.index ? 0 : hkv * n * s.t_out * 4);
  s.tiles_fwd = b.take(s.direct ? 0 : fsa_selattn_tiles_bytes(0, n, hq, hkv, d, s.t_out, a.block_size, s.max_blocks));
  s.tiles_bwd = b.take(a.inference ? 0 : fsa_selattn_tiles_bytes(1, n, hq, hkv, d, s.t_out, a.block_size, s.max_blocks));
  s.total = b.at;
  return s;
}

// Forward workspace: the stages run one after the other and share it, beside the un-rotated compressed keys.
struct LayerFwdWs {
  size_t ck_raw, stage, total, topk_bytes, index_bytes, sel_bytes, kv_bytes;
};
static LayerFwdWs layer_fwd_ws(const fsa_layer_args& a, const LayerSaved& s) {
  LayerFwdWs w;
  Bump b;
  w.ck_raw = b.take((size_t)a.total_ck * a.num_kv_heads * a.head_dim * 2);
  w.stage = b.at;
  const bool rebin = a.kernel_size == 2 * a.kernel_stride && a.block_size == 4 * a.kernel_stride;
  w.topk_bytes = fsa_cmp_topk_workspace_bytes(a.total_tokens, a.num_kv_heads, rebin ? a.max_ck / 4 + 1 : a.max_ck);
  w.index_bytes = !s.index ? 0 : fsa_index_workspace_bytes(a.total_tokens, s.t_out, a.num_kv_heads, s.max_blocks);
  w.sel_bytes = s.direct ? 0 : fsa_selattn_fwd_workspace_bytes(a.total_tokens, a.num_q_heads, a.num_kv_heads, a.head_dim, s.t_out, s.max_blocks);
  w.kv_bytes = align_up((size_t)a.total_tokens * a.num_kv_heads * a.head_dim * 2, 256);
  w.total = w.stage + align_up(std::max({w.topk_bytes, w.index_bytes, w.sel_bytes, s.direct ? 2 * w.kv_bytes + 16 : 0}), 256);
  return w;
}

struct LayerBwdWs {
  size_t stat[3], dl, gate_part, dq_cmp, dq_win, dk_sel, dv_sel, dk_win, dv_win, dck, dcv, dck_raw, dk_lc, dv_lc, dbias, stage,
      total, sel_bytes;
  int chunk, chunks;
};
static LayerBwdWs layer_bwd_ws(const fsa_layer_args& a, const LayerSaved& s) {
  LayerBwdWs w;
  Bump b;
  const size_t e = 2, n = a.total_tokens, d = a.head_dim, hq = a.num_q_heads, hkv = a.num_kv_heads;
  const size_t kv = n * hkv * d * e, ck = (size_t)a.total_ck * hkv * d * e;
  for (int i = 0; i < 3; ++i) w.stat[i] = b.take(n * hq * 8);
  w.dl = b.take(n * 3 * e);
  // two work-groups per CU for the pass over x, at least 8 tokens each and no more than LDS holds without asking (48 KB)
  const int64_t col_groups = (a.hidden + GATE_COLS - 1) / GATE_COLS;
  w.chunk = (int)std::min<int64_t>(4096, std::max<int64_t>(8, (a.total_tokens * col_groups + 511) / 512));
  w.chunks = (int)((a.total_tokens + w.chunk - 1) / w.chunk);
  w.gate_part = b.take((size_t)w.chunks * 3 * a.hidden * 4);
  w.dq_cmp = b.take(n * hq * d * e);
  w.dq_win = b.take(n * hq * d * e);
  for (size_t* x : {&w.dk_sel, &w.dv_sel, &w.dk_win, &w.dv_win, &w.dk_lc, &w.dv_lc}) *x = b.take(kv);
  for (size_t* x : {&w.dck, &w.dcv, &w.dck_raw}) *x = b.take(ck);
  w.dbias = b.take(hkv * d * 4);
  w.stage = b.at;
  w.sel_bytes = fsa_selattn_bwd_workspace_bytes(n, hq, hkv, d, s.t_out, a.block_size, s.max_blocks);
  const size_t dense_bytes = layer_attn_bwd_workspace_bytes(n, a.total_ck, a.max_len, a.window, a.batch, hq, hkv, d);
  w.total = w.stage + align_up(std::max(w.sel_bytes, dense_bytes), 256);
  return w;
}

static LayerAttn layer_attn(const fsa_layer_args& a, const LayerSaved& s) {
  char* sv = (char*)a.saved;
  LayerAttn l = {};
  l.dtype = a.dtype; l.hq = a.num_q_heads; l.hkv = a.num_kv_heads; l.head_dim = a.head_dim; l.batch = a.batch;
  l.kernel_size = a.kernel_size; l.kernel_stride = a.kernel_stride; l.window = a.window;
  l.n = a.total_tokens; l.total_ck = a.total_ck; l.max_len = a.max_len; l.scale = a.softmax_scale;
  l.cu = a.cu_seqlens; l.cu_ck = (const int32_t*)(sv + s.cu_ck);
  l.q = sv + s.q; l.k = sv + s.k; l.v = a.v; l.ck = sv + s.ck; l.cv = sv + s.cv;
  l.o_cmp = sv + s.o[0]; l.o_win = sv + s.o[2];
  l.lse_cmp = (float*)(sv + s.lse[0]); l.lse_win = (float*)(sv + s.lse[2]);
  return l;
}

static int layer_check(const fsa_layer_args* a) {
  FSA_CHECK_ARG(a, "fsa_layer: null pointer");
  FSA_CHECK_ARG(a->x && a->w_gate && a->q && a->k && a->v && a->w_ck && a->w_cv && a->pe && a->cu_seqlens && a->inv_freq &&
                    a->saved && a->workspace, "fsa_layer: null pointer");
  FSA_CHECK_ARG(a->dtype == FSA_BF16 || a->dtype == FSA_FP16, "fsa_layer: dtype must be bf16 or fp16");
  FSA_CHECK_ARG(a->head_dim == 64 || a->head_dim == 128 || a->head_dim == 256, "fsa_layer: head_dim=%d not supported", a->head_dim);
  FSA_CHECK_ARG(a->num_kv_heads >= 1 && a->num_q_heads % a->num_kv_heads == 0, "fsa_layer: bad head counts");
  FSA_CHECK_ARG(a->batch >= 1 && a->total_tokens >= 1 && a->total_ck >= 1 && a->max_ck >= 1 && a->max_len >= 1 &&
                    a->max_len <= a->total_tokens, "fsa_layer: bad sizes");
  FSA_CHECK_ARG(a->hidden >= 8 && a->hidden % 8 == 0, "fsa_layer: hidden must be a multiple of 8");
  FSA_CHECK_ARG(a->topk >= 1 && a->block_size >= 1 && a->window >= 0, "fsa_layer: bad configuration");
  return 0;
}

#define FSA_LAYER_D(CALL)                            \
  do {                                               \
    if (a.head_dim == 64) { CALL(64); }              \
    else if (a.head_dim == 128) { CALL(128); }       \
    else { CALL(256); }                              \
  } while (0)

template <typename T>
static int launch_rope(const fsa_layer_args& a, const RopeSegments& segs, const void* table, bool inverse, hipStream_t stream) {
  int64_t groups = 0;
  for (const RopeSegment& s : segs.seg) groups += (s.n + 3) / 4;
  ProfScope ps_("rope", stream);
#define FSA_CALL(DD) rope_segments_kernel<T, DD><<<(unsigned)groups, 256, 0, stream>>>(segs, (const T*)table, inverse)
  FSA_LAYER_D(FSA_CALL);
#undef FSA_CALL
  FSA_CHECK_LAUNCH("fsa_layer rope");
  return 0;
}

template <typename T>
static int layer_forward(const fsa_layer_args& a, void* out, int32_t* topk_idx, hipStream_t stream) {
  const LayerSaved s = layer_saved(a);
  const LayerFwdWs w = layer_fwd_ws(a, s);
  char *sv = (char*)a.saved, *ws = (char*)a.workspace;
  const int64_t n = a.total_tokens, d = a.head_dim, qs = a.num_q_heads * d, ks_ = a.num_kv_heads * d;
  int32_t* cu_ck = (int32_t*)(sv + s.cu_ck);
  {
    ProfScope ps_("layer_prep", stream);
    const int64_t pairs = a.max_len * (d / 2);
    const int64_t gate_blocks = (n + 4 * GATE_TOK - 1) / (4 * GATE_TOK);
    layer_prep_kernel<T><<<(unsigned)(1 + gate_blocks + (pairs + 255) / 256), 256, 0, stream>>>(
        a.cu_seqlens, a.batch, a.kernel_size, a.kernel_stride, cu_ck, a.inv_freq, a.rope_scale, (int)d / 2, pairs, (T*)(sv + s.table),
        (const T*)a.x, (const T*)a.w_gate, (T*)(sv + s.gates), n, a.hidden);
    FSA_CHECK_LAUNCH("fsa_layer prep");
  }
#define FSA_RUN(call) \
  if (int rc_ = (call)) return rc_
  LcTensors lc[2] = {};
  lc[0].x = a.k; lc[0].w = a.w_ck; lc[0].pe = a.pe; lc[0].y = ws + w.ck_raw;
  lc[1].x = a.v; lc[1].w = a.w_cv; lc[1].y = sv + s.cv;
  for (LcTensors& t : lc) {
    t.x_sn = ks_;
    t.x_sh = d;
  }
  FSA_RUN(linear_compress_fwd(lc, 2, a.dtype, a.cu_seqlens, cu_ck, a.batch, a.max_ck, a.num_kv_heads, a.head_dim, a.kernel_size,
                              a.kernel_stride, stream));
  RopeSegments segs = {};
  segs.batch = a.batch;
  segs.seg[0] = {a.q, sv + s.q, a.cu_seqlens, n, a.num_q_heads, 1};
  segs.seg[1] = {a.k, sv + s.k, a.cu_seqlens, n, a.num_kv_heads, 1};
  segs.seg[2] = {ws + w.ck_raw, sv + s.ck, cu_ck, a.total_ck, a.num_kv_heads, a.kernel_stride};
  FSA_RUN(launch_rope<T>(a, segs, sv + s.table, false, stream));
  const void *q = sv + s.q, *k = sv + s.k, *ck = sv + s.ck;
  float* lse0 = (float*)(sv + s.lse[0]);
  FSA_RUN(layer_attn_fwd(layer_attn(a, s), stream));
  FSA_RUN(fsa_cmp_topk(q, ck, lse0, a.dtype, qs, d, ks_, d, a.cu_seqlens, cu_ck, a.batch, n, a.max_len, a.max_ck, a.num_q_heads,
                       a.num_kv_heads, a.head_dim, a.kernel_size, a.kernel_stride, a.block_size, a.topk, a.init_blocks,
                       a.local_blocks, 1, 0, a.softmax_scale, topk_idx, nullptr, ws + w.stage, w.topk_bytes, stream));
  int32_t *cu_blocks = (int32_t*)(sv + s.cu_blocks), *counts = (int32_t*)(sv + s.counts), *starts = (int32_t*)(sv + s.starts),
          *sel = (int32_t*)(sv + s.sel), *slot = (int32_t*)(sv + s.slot), *tf = s.direct ? nullptr : (int32_t*)(sv + s.tiles_fwd), *tb = a.inference ? nullptr : (int32_t*)(sv + s.tiles_bwd);
  if (s.index)
    FSA_RUN(fsa_build_index_tiles(topk_idx, n * s.t_out, s.t_out, a.cu_seqlens, a.batch, n, a.num_kv_heads, s.t_out, a.block_size,
                                s.max_blocks, cu_blocks, counts, starts, sel, slot, a.num_q_heads, a.head_dim, tf, tb,
                                ws + w.stage, w.index_bytes, stream));
  MergeEpilogue merge;
  merge.a = sv + s.o[0];
  merge.c = sv + s.o[2];
  merge.gate = sv + s.gates;
  merge.out = out;
  if (s.direct) {
    // its K and V go to LDS by 16-byte loads, which want aligned rows; the other kernels do without
    const void* kv[2] = {k, a.v};
    char* copies = (char*)align_up((uintptr_t)(ws + w.stage), 16);
    for (int i = 0; i < 2; ++i) {
      if ((uintptr_t)kv[i] % 16 == 0) continue;
      ProfScope ps_("copy_aligned", stream);
      const int64_t chunks = n * ks_ / 8;
      copy_aligned_kernel<<<(unsigned)((chunks + 255) / 256), 256, 0, stream>>>((const uint16_t*)kv[i], copies + i * w.kv_bytes, chunks);
      FSA_CHECK_LAUNCH("fsa_layer copy");
      kv[i] = copies + i * w.kv_bytes;
    }
    FSA_RUN(selattn_direct_fwd(q, kv[0], kv[1], a.dtype, qs, d, ks_, d, ks_, d, topk_idx, n * s.t_out, s.t_out, a.cu_seqlens, a.batch, n,
                               a.max_len, a.num_q_heads, a.num_kv_heads, a.head_dim, s.t_out, a.block_size, a.softmax_scale,
                               a.inference ? nullptr : sv + s.o[1], qs, d, a.inference ? nullptr : (float*)(sv + s.lse[1]), merge,
                               stream));
    return 0;
  }
  FSA_RUN(selattn_fwd(q, k, a.v, a.dtype, qs, d, ks_, d, ks_, d, a.cu_seqlens, a.batch, n, a.num_q_heads, a.num_kv_heads, a.head_dim,
                      s.t_out, a.block_size, s.max_blocks, a.softmax_scale, cu_blocks, counts, starts, sel, slot, tf,
                      a.inference ? nullptr : sv + s.o[1], qs, d, a.inference ? nullptr : (float*)(sv + s.lse[1]), ws + w.stage, w.sel_bytes, merge, stream));
  return 0;
}

template <typename T>
static int layer_backward(const fsa_layer_args& a, const fsa_layer_grads& g, hipStream_t stream) {
  const LayerSaved s = layer_saved(a);
  const LayerBwdWs w = layer_bwd_ws(a, s);
  char *sv = (char*)a.saved, *ws = (char*)a.workspace;
  const int64_t n = a.total_tokens, d = a.head_dim, qs = a.num_q_heads * d, ks_ = a.num_kv_heads * d;
  const int32_t* cu_ck = (const int32_t*)(sv + s.cu_ck);
  MergeStats m = {};
  m.d_out = g.d_out;
  m.gate = sv + s.gates;
  m.dl = ws + w.dl;
  m.n = n;
  m.hq = a.num_q_heads;
  for (int i = 0; i < 3; ++i) {
    m.o[i] = sv + s.o[i];
    m.lse[i] = (const float*)(sv + s.lse[i]);
    m.stat[i] = (float2*)(ws + w.stat[i]);
  }
  {
    ProfScope ps_("merge_stats", stream);
#define FSA_CALL(DD) merge_stats_kernel<T, DD><<<(unsigned)((n + 3) / 4), 256, 0, stream>>>(m)
    FSA_LAYER_D(FSA_CALL);
#undef FSA_CALL
    FSA_CHECK_LAUNCH("fsa_layer merge backward");
  }
  {
    ProfScope ps_("gate_bwd", stream);
    const dim3 grid(w.chunks, (a.hidden + GATE_COLS - 1) / GATE_COLS);
    gate_bwd_kernel<T><<<grid, 256, (size_t)w.chunk * 12, stream>>>((const T*)a.x, (const T*)a.w_gate, (const T*)(ws + w.dl), (T*)g.dx,
                                                                    (float*)(ws + w.gate_part), n, a.hidden, w.chunk);
    const int64_t cols = (int64_t)3 * a.hidden;
    gate_dw_kernel<T><<<(unsigned)((cols + WAVE - 1) / WAVE), 256, 0, stream>>>((const float*)(ws + w.gate_part), (T*)g.dw_gate, cols, w.chunks);
    FSA_CHECK_LAUNCH("fsa_layer gate backward");
  }
  const void *q = sv + s.q, *k = sv + s.k;
  void* stage = ws + w.stage;
  LayerAttn dense = layer_attn(a, s);
  dense.d_out = g.d_out;
  dense.stat_cmp = m.stat[0]; dense.stat_win = m.stat[2];
  dense.dq_cmp = ws + w.dq_cmp; dense.dq_win = ws + w.dq_win;
  dense.dck = ws + w.dck; dense.dcv = ws + w.dcv; dense.dk_win = ws + w.dk_win; dense.dv_win = ws + w.dv_win;
  FSA_RUN(layer_attn_bwd(dense, stage, stream));
  DqEpilogue epi;
  epi.add0 = ws + w.dq_cmp;
  epi.add1 = ws + w.dq_win;
  epi.rope = sv + s.table;
  epi.cu = a.cu_seqlens;
  epi.batch = a.batch;
  FSA_RUN(selattn_bwd(q, k, a.v, nullptr, g.d_out, nullptr, a.dtype, qs, d, ks_, d, ks_, d, qs, d, qs, d, a.cu_seqlens, a.batch, n,
                      a.num_q_heads, a.num_kv_heads, a.head_dim, s.t_out, a.block_size, s.max_blocks, a.softmax_scale,
                      (const int32_t*)(sv + s.cu_blocks), (const int32_t*)(sv + s.counts), (const int32_t*)(sv + s.starts),
                      (const int32_t*)(sv + s.sel), (const int32_t*)(sv + s.slot), (const int32_t*)(sv + s.tiles_bwd), g.dq,
                      ws + w.dk_sel, ws + w.dv_sel, stage, w.sel_bytes, m.stat[1], epi, stream));
  RopeSegments segs = {};
  segs.batch = a.batch;
  segs.seg[0] = {ws + w.dck, ws + w.dck_raw, cu_ck, a.total_ck, a.num_kv_heads, a.kernel_stride};
  FSA_RUN(launch_rope<T>(a, segs, sv + s.table, true, stream));
  LcTensors lc[2] = {};
  lc[0].x = a.k; lc[0].w = a.w_ck; lc[0].pe = a.pe; lc[0].dy = ws + w.dck_raw; lc[0].dx = ws + w.dk_lc; lc[0].dw = g.dw_ck;
  lc[0].dpe = g.dpe; lc[0].dbias = (float*)(ws + w.dbias);
  lc[1].x = a.v; lc[1].w = a.w_cv; lc[1].dy = ws + w.dcv; lc[1].dx = ws + w.dv_lc; lc[1].dw = g.dw_cv;
  for (LcTensors& t : lc) {
    t.x_sn = ks_;
    t.x_sh = d;
  }
  FSA_RUN(linear_compress_bwd(lc, 2, a.dtype, a.cu_seqlens, cu_ck, a.batch, a.max_len, a.num_kv_heads, a.head_dim, a.kernel_size,
                              a.kernel_stride, stream));
  KvCombine c = {};
  c.dk[0] = ws + w.dk_sel; c.dk[1] = ws + w.dk_win; c.dk[2] = ws + w.dk_lc;
  c.dv[0] = ws + w.dv_sel; c.dv[1] = ws + w.dv_win; c.dv[2] = ws + w.dv_lc;
  c.dk_out = g.dk; c.dv_out = g.dv;
  c.table = sv + s.table; c.cu = a.cu_seqlens; c.batch = a.batch; c.heads = a.num_kv_heads; c.n = n;
  ProfScope ps_("kv_combine", stream);
#define FSA_CALL(DD)                                                                                                      \
  kv_combine_kernel<T, DD><<<(unsigned)((n * a.num_kv_heads + 256 / (DD / 8) - 1) / (256 / (DD / 8))), 256, 0, stream>>>(c)
  FSA_LAYER_D(FSA_CALL);
#undef FSA_CALL
#undef FSA_RUN
  FSA_CHECK_LAUNCH("fsa_layer kv gradients");
  return 0;
}

}  // namespace fsa

using namespace fsa;

extern "C" size_t fsa_layer_saved_bytes(const fsa_layer_args* args) {
  if (!args || args->block_size < 1 || args->num_kv_heads < 1) return 0;
  return layer_saved(*args).total;
}

extern "C" size_t fsa_layer_workspace_bytes(const fsa_layer_args* args, int32_t backward) {
  if (!args || args->block_size < 1 || args->num_kv_heads < 1) return 0;
  const LayerSaved s = layer_saved(*args);
  return backward ? layer_bwd_ws(*args, s).total : layer_fwd_ws(*args, s).total;
}

extern "C" int fsa_layer_forward(const fsa_layer_args* args, void* out, int32_t* topk_idx, void* stream_) {
  if (int rc = layer_check(args)) return rc;
  FSA_CHECK_ARG(out && topk_idx, "fsa_layer_forward: null pointer");
  if (args->saved_bytes < fsa_layer_saved_bytes(args) || args->workspace_bytes < fsa_layer_workspace_bytes(args, 0)) {
    set_error("fsa_layer_forward: workspace too small");
    return FSA_ERR_WORKSPACE;
  }
  return args->dtype == FSA_BF16 ? layer_forward<__bf16>(*args, out, topk_idx, (hipStream_t)stream_)
                                 : layer_forward<_Float16>(*args, out, topk_idx, (hipStream_t)stream_);
}

extern "C" int fsa_layer_backward(const fsa_layer_args* args, const fsa_layer_grads* grads, void* stream_) {
  if (int rc = layer_check(args)) return rc;
  FSA_CHECK_ARG(grads && grads->d_out && grads->dq && grads->dk && grads->dv && grads->dw_gate && grads->dw_ck && grads->dw_cv &&
                    grads->dpe, "fsa_layer_backward: null pointer");
  FSA_CHECK_ARG(!args->inference, "fsa_layer_backward: the forward ran for inference and kept nothing for a backward");
  if (args->saved_bytes < fsa_layer_saved_bytes(args) || args->workspace_bytes < fsa_layer_workspace_bytes(args, 1)) {
    set_error("fsa_layer_backward: workspace too small");
    return FSA_ERR_WORKSPACE;
  }
  return args->dtype == FSA_BF16 ? layer_backward<__bf16>(*args, *grads, (hipStream_t)stream_)
                                 : layer_backward<_Float16>(*args, *grads, (hipStream_t)stream_);
}
