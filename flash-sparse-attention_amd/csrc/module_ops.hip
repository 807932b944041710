// Kernels the attention layer needs around the hot path (gfx950):
//   rope          : rotary embedding on packed sequences (forward, and its inverse
//                   rotation = backward), positions start + j*stride per sequence
//   lc_fwd        : linear compression y[n,h,:] = sum_k x[n*stride+k,h,:] W[h,k] (+ bias)
//                   as a strided-window GEMM: Y^T = W^T X^T on 32x32x16 MFMA, W tiles
//                   through LDS with transposing reads, X rows straight from memory
//   lc_dx / lc_dw : its backward without atomics: dX^T = sum_r W[h,k_r] dY[n_r]^T per
//                   token phase, and dW[h,k] = X_k^T dY with both operands read
//                   transposed from LDS tiles
//
// Semantics: nsa_ref/module/rope.py:64-134, nsa_ref/ops/linear_compress.py:28-131
// (forward), :135-292 (backward, fp32 atomics there), :474-502 (positional bias).
#include "fsa_common.h"

namespace fsa {

// ------------------------------------------------------------------- rope ----
// One wave per token.  d/16 lanes cover a head (each lane 8 dims of the first half and their partners in the second
// half), so a load instruction of the wave covers the half-rows of 64 / (d/16) neighbouring heads: the token's row
// is read and written in contiguous 2*d-byte pieces.  The angles depend on the position and the dim only; every lane
// evaluates the cos / sin of its 8 dims once and reuses them for all the heads it visits.  For the usual head dims
// (LPR = d/16 a compile-time power of two) the lanes that share the same dims split the eight evaluations among
// themselves and exchange the results, so a lane evaluates one or two angles instead of eight.
template <typename T, int LPR>
__global__ void __launch_bounds__(256)
rope_kernel(const T* __restrict__ x, int64_t x_sn, int64_t x_sh, T* __restrict__ out, int64_t o_sn,
            int64_t o_sh, const int32_t* __restrict__ cu, int batch, int64_t n, int h, int d,
            const float* __restrict__ inv_freq, float attn_scale, int start, int stride, int conj) {
  typedef typename Elem<T>::vec8 vec8;
  const int lpr = LPR > 0 ? LPR : d / 16, hpw = WAVE / lpr;
  const int lane = threadIdx.x & (WAVE - 1);
  const int64_t tok = (int64_t)blockIdx.x * (256 / WAVE) + (threadIdx.x / WAVE);
  if (tok >= n) return;
  const int sub = lane % lpr, hl = lane / lpr;
  if (hl >= hpw) return;  // lanes left over where d/16 does not divide the wave
  const int s = upper_seg(cu, batch, (int)tok);
  const float pos = (float)(start + ((int)tok - cu[s]) * stride);
  // the tables are rounded to the tensor's dtype before use, as in the reference
  auto table = [&](int e, float& cv_out, float& sv_out) {
    float sv, cv;
    sincosf(pos * inv_freq[sub * 8 + e], &sv, &cv);
    cv_out = (float)(T)(cv * attn_scale);
    sv_out = (float)(T)(sv * attn_scale);
    if (conj) sv_out = -sv_out;
  };
  float c[8], sn[8];
  if constexpr (LPR > 0) {
    constexpr int HPW = WAVE / LPR;                  // lanes that hold the same dims
    constexpr int PER = HPW >= 8 ? 1 : 8 / HPW;      // evaluations per lane
    float cl[PER], sl[PER];
#pragma unroll
    for (int i = 0; i < PER; ++i) table((hl + i * HPW) % 8, cl[i], sl[i]);
#pragma unroll
    for (int e = 0; e < 8; ++e) {  // dim e was evaluated by the lane with hl = e % HPW in its turn e / HPW
      const int src = (e % HPW) * LPR + sub;
      c[e] = __shfl(cl[HPW >= 8 ? 0 : e / HPW], src, WAVE);
      sn[e] = __shfl(sl[HPW >= 8 ? 0 : e / HPW], src, WAVE);
    }
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e) table(e, c[e], sn[e]);
  }
#pragma unroll 4
  for (int head = hl; head < h; head += hpw) {
    const T* xr = x + tok * x_sn + (int64_t)head * x_sh + sub * 8;
    vec8 a = load16<vec8>(xr), b = load16<vec8>(xr + d / 2);
    vec8 oa, ob;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float x1 = (float)a[e], x2 = (float)b[e];
      oa[e] = (T)(x1 * c[e] - x2 * sn[e]);
      ob[e] = (T)(x1 * sn[e] + x2 * c[e]);
    }
    T* orow = out + tok * o_sn + (int64_t)head * o_sh + sub * 8;
    store16(orow, oa);
    store16(orow + d / 2, ob);
  }
}

// ------------------------------------------------------- linear compress ----
constexpr int LC_KC = 64;     // contraction chunk staged per step
constexpr int LC_ROWS = 128;  // compressed tokens (or tokens) per work-group

struct LcPair {
  LcTensors t[2];
};

// Forward: a work-group owns 32 rows (compressed tokens) and DN output columns of one head; its four waves split the window
// offsets k (wave w takes k = w, w + 4, ...), each with a private W tile in LDS and no work-group barrier inside the loop,
// and the partial Y^T tiles are summed through LDS at the end.  (Few compressed tokens exist - a 16th of the sequence - so
// the work is spread over the offsets as well to fill the chip.)  The bias of a head, the same product with the positional
// rows in place of the window, is one more row of every tile: it costs 1 of 32 rows instead of a pass of its own over W.
// With DEPTH steps of loads in flight the kernel is bound by the address side of the loads: a fragment of x is 32 rows, a
// line each.  8 heads of 128, keys and values, bias included, 5003 tokens: 33 us; one step at a time, a launch for each
// tensor and one for the bias took 71.
constexpr int LCF_WAVES = 4;
constexpr int LCF_ROWS = 32;

template <int D, int DN> struct LcFwdLds {
  static constexpr int KC = 32;                            // rows of W staged per step and wave
  static constexpr int DEPTH = DN > 128 ? 1 : DN > 64 ? 2 : 4;  // steps whose loads are in flight
  static constexpr int WS = DN + 16;                       // W tile row stride (32 B pad for the transposing reads)
  static constexpr int RS = DN + 4;                        // row stride of the fp32 reduction tiles
  static constexpr int TILE_BYTES = LCF_WAVES * KC * WS * 2;
  static constexpr int RED_BYTES = LCF_WAVES * LCF_ROWS * RS * 4;
  static constexpr int BYTES = TILE_BYTES > RED_BYTES ? TILE_BYTES : RED_BYTES;
};

template <typename T, int D, int DN>
__global__ void __launch_bounds__(64 * LCF_WAVES)
lc_fwd_kernel(LcPair p, const int32_t* __restrict__ cu_x, const int32_t* __restrict__ cu_y, int nheads, int ks, int stride) {
  typedef typename Elem<T>::vec8 vec8;
  typedef typename Elem<T>::vec4 vec4;
  typedef LcFwdLds<D, DN> L;
  constexpr int KC = L::KC, WS = L::WS, RS = L::RS, NT = DN / 32, ND = D / KC, NC = D / DN;
  constexpr int NLD = KC * (DN / 8) / 64;  // 16-byte chunks of a W tile per lane
  extern __shared__ __attribute__((aligned(16))) unsigned char lc_smem[];
  const int s = blockIdx.y, dn_lo = blockIdx.z % NC * DN, hz = blockIdx.z / NC, h = hz % nheads;
  const LcTensors& tp = p.t[hz / nheads];
  const bool has_pe = tp.pe != nullptr;
  const int rows = has_pe ? LCF_ROWS - 1 : LCF_ROWS;   // the last row is the bias
  const int y0 = cu_y[s], ny = cu_y[s + 1] - y0, x0 = cu_x[s];
  const int n_lo = blockIdx.x * rows;
  if (n_lo >= ny) return;
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int col = lane & 31, hh = lane >> 5;
  T* Wt = reinterpret_cast<T*>(lc_smem) + wv * (KC * WS);
  const int n = n_lo + col;
  const bool is_pe = has_pe && col == rows;   // (rows past the end repeat the first one and are not stored)
  const T* xrow0 = is_pe ? reinterpret_cast<const T*>(tp.pe) + (int64_t)h * ks * D
                         : reinterpret_cast<const T*>(tp.x) + (int64_t)(x0 + (col < rows && n < ny ? n : 0) * stride) * tp.x_sn + (int64_t)h * tp.x_sh;
  xrow0 += 8 * hh;
  const int64_t x_sn = is_pe ? D : tp.x_sn;
  const T* wh = reinterpret_cast<const T*>(tp.w) + (int64_t)h * ks * D * D + dn_lo;
  const int tr_row = (lane & 15) >> 2, tr_col = 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
  f32x16 acc[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[t][i] = 0.f;
  constexpr int DEPTH = L::DEPTH;
  vec8 wreg[DEPTH][NLD], xf[DEPTH][KC / 16];
  const int steps = wv < ks ? (ks - wv + 3) / 4 * ND : 0;
  const uint32_t w_lane = (lane / (DN / 8)) * D + lane % (DN / 8) * 8;
  // Behind the end: the last step once more, unused.  Always loads, so that the number of loads in flight is known at every
  // point and none is waited for early.
  auto load_step = [&](int i, vec8 (&wr)[NLD], vec8 (&xr)[KC / 16]) {
    i = max(0, min(i, steps - 1));
    const int k = min(wv + 4 * (i / ND), ks - 1), dc = i % ND * KC;
    const T* wt = wh + ((int64_t)k * D + dc) * D;
#pragma unroll
    for (int j = 0; j < NLD; ++j) wr[j] = load16<vec8>(wt + w_lane + j * (64 / (DN / 8)) * D);
    const T* xr0 = xrow0 + k * x_sn + dc;
#pragma unroll
    for (int kk = 0; kk < KC / 16; ++kk) xr[kk] = load16<vec8>(xr0 + 16 * kk);
  };
  auto step = [&](const vec8 (&wr)[NLD], const vec8 (&xr)[KC / 16]) {
    __builtin_amdgcn_wave_barrier();  // the previous tile has been consumed
#pragma unroll
    for (int j = 0; j < NLD; ++j) {
      const int c = lane + 64 * j;
      store16(&Wt[c / (DN / 8) * WS + c % (DN / 8) * 8], wr[j]);
    }
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int kk = 0; kk < KC / 16; ++kk)
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        vec8 wf = lds_tr8_rows<T>(&Wt[(16 * kk + 8 * hh + tr_row) * WS + t * 32 + tr_col], WS);
        acc[t] = Elem<T>::mfma32(wf, xr[kk], acc[t]);
      }
  };
#pragma unroll
  for (int i = 0; i < DEPTH; ++i) load_step(i, wreg[i], xf[i]);
  // (whole turns in a loop without exits inside: a load's age is the same on every way to the place that waits for it)
  int i = 0;
  for (; i + DEPTH <= steps; i += DEPTH) {
#pragma unroll
    for (int u = 0; u < DEPTH; ++u) {
      step(wreg[u], xf[u]);
      load_step(i + u + DEPTH, wreg[u], xf[u]);
    }
  }
#pragma unroll
  for (int u = 0; u < DEPTH - 1; ++u)
    if (i + u < steps) step(wreg[u], xf[u]);
  // sum of the waves' tiles: red[wave][row][dout] fp32
  float* red = reinterpret_cast<float*>(lc_smem);
  __syncthreads();
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int qd = 0; qd < 4; ++qd)
      *reinterpret_cast<f32x4*>(&red[(wv * LCF_ROWS + col) * RS + t * 32 + 8 * qd + 4 * hh]) =
          f32x4{acc[t][4 * qd], acc[t][4 * qd + 1], acc[t][4 * qd + 2], acc[t][4 * qd + 3]};
  __syncthreads();
  auto total = [&](int row, int d4) {
    f32x4 sum = *reinterpret_cast<const f32x4*>(&red[row * RS + d4]);
#pragma unroll
    for (int ww = 1; ww < 4; ++ww) sum += *reinterpret_cast<const f32x4*>(&red[(ww * LCF_ROWS + row) * RS + d4]);
    return sum;
  };
  for (int e = tid; e < rows * (DN / 4); e += 64 * LCF_WAVES) {
    const int row = e / (DN / 4), d4 = (e % (DN / 4)) * 4;
    if (n_lo + row >= ny) continue;
    const f32x4 sum = total(row, d4);
    vec4 out;
#pragma unroll
    for (int i = 0; i < 4; ++i) out[i] = (T)sum[i];
    if (has_pe) {
      const f32x4 bias = total(rows, d4);
#pragma unroll
      for (int i = 0; i < 4; ++i) out[i] = (T)((float)out[i] + (float)(T)bias[i]);
    }
    store8(reinterpret_cast<T*>(tp.y) + ((int64_t)(y0 + n_lo + row) * nheads + h) * D + dn_lo + d4, out);
  }
}

// dbias[h, dout] = sum_n dY[n, h, dout]  (fp32) for 32 columns, by one work-group: four lanes read a 64-byte piece of a row,
// 64 rows at a time with several steps in flight, and the 64 row slices meet in LDS in a fixed order.
constexpr int LCB_COLS = 32;
template <typename T>
__device__ __forceinline__ void lc_dbias(const LcTensors& tp, const int32_t* cu_y, int batch, int nheads, int d, int h, int group,
                                         float* part /* [64][LCB_COLS + 1] */) {
  typedef typename Elem<T>::vec8 vec8;
  constexpr int P = LCB_COLS + 1;
  const int tid = threadIdx.x, c = (tid & 3) * 8, slice = tid >> 2;
  const int ny = cu_y[batch];
  const T* yp = reinterpret_cast<const T*>(tp.dy) + (int64_t)h * d + group * LCB_COLS + c;
  float s[8] = {};
  constexpr int U = 8;
  for (int i0 = slice; i0 < ny; i0 += 64 * U) {
    vec8 x[U];
#pragma unroll
    for (int u = 0; u < U; ++u) x[u] = load16<vec8>(yp + (int64_t)min(i0 + 64 * u, ny - 1) * nheads * d);
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int e = 0; e < 8; ++e) s[e] += i0 + 64 * u < ny ? (float)x[u][e] : 0.f;
  }
#pragma unroll
  for (int e = 0; e < 8; ++e) part[slice * P + c + e] = s[e];
  for (int o = 32; o >= 1; o >>= 1) {
    __syncthreads();
    for (int i = tid; i < o * LCB_COLS; i += 256) part[i / LCB_COLS * P + i % LCB_COLS] += part[(i / LCB_COLS + o) * P + i % LCB_COLS];
  }
  __syncthreads();
  if (tid < LCB_COLS) tp.dbias[h * d + group * LCB_COLS + tid] = part[tid];
}

// dpe[h, k, d] = sum_dout W[h,k,d,dout] dbias[h,dout]: D/8 lanes per row of W; LC_DPE_WGS work-groups per head share the rows
constexpr int LC_DPE_WGS = 16;
template <typename T> __device__ __forceinline__ void lc_dpe(const LcTensors& tp, int kd, int d, int h, int wg) {
  typedef typename Elem<T>::vec8 vec8;
  const int lpr = d / 8, rows = 256 / lpr, sub = threadIdx.x % lpr;   // lpr: 8, 16 or 32
  float b[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) b[e] = tp.dbias[h * d + sub * 8 + e];
  const T* w = reinterpret_cast<const T*>(tp.w) + (int64_t)h * kd * d + sub * 8;
  constexpr int U = 4;
  for (int i0 = wg * rows + threadIdx.x / lpr; i0 - (int)threadIdx.x / lpr < kd; i0 += LC_DPE_WGS * rows * U) {   // uniform
    vec8 x[U];
#pragma unroll
    for (int u = 0; u < U; ++u) x[u] = load16<vec8>(w + (int64_t)min(i0 + u * LC_DPE_WGS * rows, kd - 1) * d);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int i = i0 + u * LC_DPE_WGS * rows;
      float s = 0.f;
#pragma unroll
      for (int e = 0; e < 8; ++e) s += (float)x[u][e] * b[e];
      for (int o = lpr / 2; o >= 1; o >>= 1) s += __shfl_xor(s, o, WAVE);
      if (sub == 0 && i < kd) reinterpret_cast<T*>(tp.dpe)[(int64_t)h * kd + i] = (T)s;
    }
  }
}

// dX: one wave = 32 tokens of one phase (t % stride), so that the window offsets k_r are wave-uniform
template <int D> struct LcDxLds {
  static constexpr int WS = D + 8;                          // W of a step, rows 16 bytes apart in the banks
  static constexpr int ROWS_BYTES = LC_ROWS * D * 2;        // the results of the four waves, in place of it (head_dim 64: the larger)
  static constexpr int SUMS_BYTES = 64 * (LCB_COLS + 1) * 4;   // lc_dbias
  static constexpr int BYTES = std::max({D * WS * 2, ROWS_BYTES, SUMS_BYTES});
};
template <typename T, int D>
__global__ void __launch_bounds__(256)
lc_dx_kernel(LcPair p, const int32_t* __restrict__ cu_x, const int32_t* __restrict__ cu_y, int nheads, int ks, int stride) {
  typedef typename Elem<T>::vec8 vec8;
  typedef typename Elem<T>::vec4 vec4;
  constexpr int NT = D / 32;
  const int s = blockIdx.y, h = blockIdx.z % nheads;
  const LcTensors& tp = p.t[blockIdx.z / nheads];
  extern __shared__ __attribute__((aligned(16))) unsigned char lc_smem[];
  if ((int)blockIdx.x < D / LCB_COLS) {   // the column sums of dY, for dpe and dW
    if (s == 0 && tp.pe) lc_dbias<T>(tp, cu_y, gridDim.y, nheads, D, h, blockIdx.x, reinterpret_cast<float*>(lc_smem));
    return;
  }
  const int tile = blockIdx.x - D / LCB_COLS;
  const T *dy = reinterpret_cast<const T*>(tp.dy), *w = reinterpret_cast<const T*>(tp.w);
  T* dx = reinterpret_cast<T*>(tp.dx);
  const int x0 = cu_x[s], len = cu_x[s + 1] - x0, y0 = cu_y[s], ny = cu_y[s + 1] - y0;
  const int m_per_phase = (len + stride - 1) / stride;
  const int tiles_per_phase = (m_per_phase + LC_ROWS - 1) / LC_ROWS;
  const int phase = tile / tiles_per_phase, mt = tile % tiles_per_phase;
  if (phase >= stride || len == 0) return;
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int col = lane & 31, hh = lane >> 5;
  const int m = mt * LC_ROWS + wv * 32 + col;
  const int t = phase + stride * m;
  const bool valid = t < len;
  const int nrep = ks / stride;
  f32x16 acc[NT];
#pragma unroll
  for (int i_ = 0; i_ < NT; ++i_)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[i_][i] = 0.f;
  // W[h, k] ([d][dout], 2 D^2 bytes) of the step is staged in LDS: as the A operand every lane reads a different
  // row of it, which straight from global memory is 64 cache lines per load instruction
  constexpr int WS = LcDxLds<D>::WS;
  T* Ws = reinterpret_cast<T*>(lc_smem);
  for (int r = 0; r < nrep; ++r) {
    const int nwin = m - r, k = phase + r * stride;
    const bool ok = valid && nwin >= 0 && nwin < ny;
    const T* dyrow = dy + ((int64_t)(y0 + (ok ? nwin : 0)) * nheads + h) * D + 8 * hh;
    const T* wk = w + ((int64_t)h * ks + k) * D * D;
    vec8 yf[D / 16];
#pragma unroll
    for (int kk = 0; kk < D / 16; ++kk) {
      yf[kk] = zero8<T>();
      if (ok) yf[kk] = load16<vec8>(dyrow + 16 * kk);
    }
    if (r) __syncthreads();
    for (int c = tid; c < D * (D / 8); c += 256) {
      const int row = c / (D / 8), cc = c % (D / 8);
      store16(&Ws[row * WS + cc * 8], load16<vec8>(wk + (int64_t)row * D + cc * 8));
    }
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < D / 16; ++kk)
#pragma unroll
      for (int i_ = 0; i_ < NT; ++i_) {
        vec8 wf = load16<vec8>(&Ws[(i_ * 32 + col) * WS + 16 * kk + 8 * hh]);  // A[m = d][k = dout]
        acc[i_] = Elem<T>::mfma32(wf, yf[kk], acc[i_]);
      }
  }
  // Whole rows, by way of LDS (chunk c of row r in the place of chunk c ^ chunk_swizzle(r)).  Against pieces of 8 bytes of 32 rows,
  // us: 4 x 8192 tokens x 8 heads of 128 105 -> 92, 5003 x 8 26.7 -> 23.4, 6000 x 8 of 64 15.8 -> 12.3.
  __syncthreads();
  static_assert(256 / WAVE * 32 * D * (int)sizeof(T) <= LcDxLds<D>::BYTES, "a tile of 32 rows for every wave");
  T* own = Ws + wv * (32 * D);
#pragma unroll
  for (int i_ = 0; i_ < NT; ++i_)
#pragma unroll
    for (int qd = 0; qd < 4; ++qd) {
      vec4 v;
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = (T)acc[i_][4 * qd + e];
      store8(&own[col * D + ((4 * i_ + qd) ^ chunk_swizzle<D>(col)) * 8 + 4 * hh], v);
    }
  __builtin_amdgcn_wave_barrier();
  constexpr int CPR = D / 8, RPI = 64 / CPR;
#pragma unroll
  for (int j = 0; j < 32 / RPI; ++j) {
    const int r = j * RPI + lane / CPR, c = lane % CPR, tr = phase + stride * (mt * LC_ROWS + wv * 32 + r);
    const vec8 v = load16<vec8>(&own[r * D + (c ^ chunk_swizzle<D>(r)) * 8]);
    if (tr < len) store16(dx + ((int64_t)(x0 + tr) * nheads + h) * D + c * 8, v);
  }
}

// dW[h, k, d, dout] = sum_n x[tok(n) + k, h, d] dY[n, h, dout] (+ pe[h,k,d] dbias[h,dout])
// One work-group per (offset k, head, 128 input dims; at head_dim 64: two neighbouring offsets): few work-groups, each a long loop over all compressed
// tokens, so a step covers many tokens (LCW_KC) to keep enough rows in flight.  (Cutting the output dims over more
// work-groups was measured and is slower: the strided X rows, 256 bytes every kernel_stride tokens, are what the
// kernel waits for, and every cut reads them again.)
constexpr int LCW_KC = 128;
template <int D> struct LcDwLds { static constexpr int BYTES = LCW_KC * ((128 + 16) + (D + 16)) * 2; };

template <typename T, int D>
__global__ void __launch_bounds__(256)
lc_dw_kernel(LcPair p, const int32_t* __restrict__ cu_x, const int32_t* __restrict__ cu_y, int batch, int nheads, int ks,
             int stride) {
  typedef typename Elem<T>::vec8 vec8;
  constexpr int LCW_DOUT = D;  // output dims per work-group
  constexpr int XS = 128 + 16, YS = LCW_DOUT + 16, NT = LCW_DOUT / 32;  // 32 B pads: conflict-free transposing reads
  constexpr int LC_KC = LCW_KC;  // compressed tokens per step of this kernel
  constexpr int YC = LCW_DOUT / 8;  // 16-byte chunks of a dY row slice
  extern __shared__ __attribute__((aligned(16))) unsigned char lcw_smem[];
  T* Xs = reinterpret_cast<T*>(lcw_smem);
  T* Ys = Xs + LC_KC * XS;
  constexpr int KPW = D < 128 ? 128 / D : 1;   // window offsets per work-group: the X tile holds 128 (offset, dim) columns
  const int h = blockIdx.y % nheads;
  const LcTensors& tp = p.t[blockIdx.y / nheads];
  if ((int)blockIdx.x < LC_DPE_WGS) {
    if (tp.pe && blockIdx.z == 0) lc_dpe<T>(tp, ks * D, D, h, blockIdx.x);
    return;
  }
  const int k = (blockIdx.x - LC_DPE_WGS) * KPW;
  const T *x = reinterpret_cast<const T*>(tp.x), *dy = reinterpret_cast<const T*>(tp.dy), *pe = reinterpret_cast<const T*>(tp.pe);
  const float* dbias = tp.dbias;
  const int64_t x_sn = tp.x_sn, x_sh = tp.x_sh;
  T* dw = reinterpret_cast<T*>(tp.dw);
  const int dz = (blockIdx.z / (D / LCW_DOUT)) * 128, dout0 = (blockIdx.z % (D / LCW_DOUT)) * LCW_DOUT;
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int col = lane & 31, hh = lane >> 5;
  const int ny_total = cu_y[batch];
  const int tr_row = (lane & 15) >> 2, tr_col = 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
  f32x16 acc[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[t][i] = 0.f;
  // the rows of the next step travel while the current one is multiplied
  constexpr int NX = LC_KC * 16 / 256, NY = LC_KC * YC / 256;
  static_assert(LC_KC * YC % 256 == 0, "dY slice must divide over the threads");
  vec8 xr[NX], yr[NY];
  // Token of compressed row n at window offset k (-1 past the end): looked up by one thread per row of a step (a
  // search through cu_y, a chain of dependent loads) two steps ahead and handed to the 16 threads that load the
  // row through a small double-buffered LDS table, so the search is neither repeated per chunk nor part of the
  // latency of a step.
  __shared__ int tok_l[2][LC_KC];
  auto find_tokens = [&](int n0, int buf) {
    if (tid < LC_KC) {
      const int n = n0 + tid;
      int tok = -1;
      if (n < ny_total) {
        const int s = upper_seg(cu_y, batch, n);
        tok = cu_x[s] + (n - cu_y[s]) * stride + k;
      }
      tok_l[buf][tid] = tok;
    }
  };
  auto load_step = [&](int n0, int buf) {
#pragma unroll
    for (int j = 0; j < NY; ++j) {
      const int c = tid + 256 * j, r = c / YC, cc = c % YC;
      const int n = n0 + r;
      yr[j] = zero8<T>();
      if (n < ny_total) yr[j] = load16<vec8>(dy + ((int64_t)n * nheads + h) * D + dout0 + cc * 8);
    }
#pragma unroll
    for (int j = 0; j < NX; ++j) {  // X rows: 128 dims = 16 chunks
      const int c = tid + 256 * j, cc = c % 16;
      const int tok = tok_l[buf][c / 16];
      xr[j] = zero8<T>();
      if (tok >= 0) xr[j] = load16<vec8>(x + (int64_t)(tok + cc * 8 / D) * x_sn + (int64_t)h * x_sh + dz + cc * 8 % D);
    }
  };
  find_tokens(0, 0);
  find_tokens(LC_KC, 1);
  __syncthreads();
  load_step(0, 0);
  // step i uses table i & 1; the table of step i + 2 is written after the barriers of step i, i.e. after every
  // thread has read the same buffer for step i's rows (in the previous iteration)
  int buf = 0;
  for (int n0 = 0; n0 < ny_total; n0 += LC_KC, buf ^= 1) {
    __syncthreads();
#pragma unroll
    for (int j = 0; j < NX; ++j) {
      const int c = tid + 256 * j;
      store16(&Xs[(c / 16) * XS + (c % 16) * 8], xr[j]);
    }
#pragma unroll
    for (int j = 0; j < NY; ++j) {
      const int c = tid + 256 * j;
      store16(&Ys[(c / YC) * YS + (c % YC) * 8], yr[j]);
    }
    __syncthreads();
    if (n0 + LC_KC < ny_total) {
      load_step(n0 + LC_KC, buf ^ 1);
      find_tokens(n0 + 2 * LC_KC, buf);
    }
#pragma unroll
    for (int kk = 0; kk < LC_KC / 16; ++kk) {
      vec8 xf = lds_tr8_rows<T>(&Xs[(16 * kk + 8 * hh + tr_row) * XS + wv * 32 + tr_col], XS);  // A[m = d][k = n]
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        vec8 yf = lds_tr8_rows<T>(&Ys[(16 * kk + 8 * hh + tr_row) * YS + t * 32 + tr_col], YS);  // B[k = n][dout]
        acc[t] = Elem<T>::mfma32(xf, yf, acc[t]);
      }
    }
  }
  // C layout: lane column = dout within the tile, registers = d rows
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int dk = dz + wv * 32 + 8 * (i >> 2) + 4 * hh + (i & 3);   // column of the X tile
      const int dd = dk % D, kk = k + (KPW > 1 ? dk / D : 0);
      const int dout = dout0 + t * 32 + col;
      float v = acc[t][i];
      if (pe) v += (float)pe[((int64_t)h * ks + kk) * D + dd] * dbias[h * D + dout];
      dw[(((int64_t)h * ks + kk) * D + dd) * D + dout] = (T)v;
    }
}

// -------------------------------------------------------------- gate merge ----
// out[n, :] = g[n,0] a[n, :] + g[n,1] b[n, :] + g[n,2] c[n, :]  (one wave per token row, 16-byte chunks,
// fp32 sum rounded once); backward: d_a = g0 d_out (same for b, c) and d_g[n,i] = <d_out[n, :], x_i[n, :]>.
template <typename T>
__global__ void __launch_bounds__(256)
gate_merge_fwd_kernel(const T* __restrict__ a, const T* __restrict__ b, const T* __restrict__ c,
                      const T* __restrict__ gate, T* __restrict__ out, int64_t n_tokens, int row) {
  typedef typename Elem<T>::vec8 vec8;
  const int64_t n = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (n >= n_tokens) return;
  const int lane = threadIdx.x & 63;
  const float g0 = (float)gate[n * 3], g1 = (float)gate[n * 3 + 1], g2 = (float)gate[n * 3 + 2];
  const int64_t base = n * row;
  for (int e = lane * 8; e < row; e += 512) {
    const vec8 x = load16_stream<vec8>(a + base + e), y = load16_stream<vec8>(b + base + e), z = load16_stream<vec8>(c + base + e);
    vec8 r;
#pragma unroll
    for (int i = 0; i < 8; ++i) r[i] = (T)(g0 * (float)x[i] + g1 * (float)y[i] + g2 * (float)z[i]);
    store16(out + base + e, r);
  }
}

template <typename T>
__global__ void __launch_bounds__(256)
gate_merge_bwd_kernel(const T* __restrict__ d_out, const T* __restrict__ a, const T* __restrict__ b,
                      const T* __restrict__ c, const T* __restrict__ gate, T* __restrict__ d_a,
                      T* __restrict__ d_b, T* __restrict__ d_c, T* __restrict__ d_gate, int64_t n_tokens,
                      int row) {
  typedef typename Elem<T>::vec8 vec8;
  const int64_t n = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (n >= n_tokens) return;
  const int lane = threadIdx.x & 63;
  const float g0 = (float)gate[n * 3], g1 = (float)gate[n * 3 + 1], g2 = (float)gate[n * 3 + 2];
  const int64_t base = n * row;
  float s0 = 0.f, s1 = 0.f, s2 = 0.f;
  for (int e = lane * 8; e < row; e += 512) {
    const vec8 w = load16_stream<vec8>(d_out + base + e);
    const vec8 x = load16_stream<vec8>(a + base + e), y = load16_stream<vec8>(b + base + e), z = load16_stream<vec8>(c + base + e);
    vec8 ra, rb, rc;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float wf = (float)w[i];
      s0 += wf * (float)x[i];
      s1 += wf * (float)y[i];
      s2 += wf * (float)z[i];
      ra[i] = (T)(g0 * wf);
      rb[i] = (T)(g1 * wf);
      rc[i] = (T)(g2 * wf);
    }
    store16(d_a + base + e, ra);
    store16(d_b + base + e, rb);
    store16(d_c + base + e, rc);
  }
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) {
    s0 += __shfl_xor(s0, o, 64);
    s1 += __shfl_xor(s1, o, 64);
    s2 += __shfl_xor(s2, o, 64);
  }
  if (lane == 0) {
    d_gate[n * 3] = (T)s0;
    d_gate[n * 3 + 1] = (T)s1;
    d_gate[n * 3 + 2] = (T)s2;
  }
}

}  // namespace fsa

using namespace fsa;

extern "C" int fsa_rope(const void* x, void* out, int32_t dtype, int64_t x_stride_n, int64_t x_stride_h,
                        int64_t o_stride_n, int64_t o_stride_h, const int32_t* cu_seqlens, int32_t batch,
                        int64_t total_tokens, int32_t num_heads, int32_t head_dim, const float* inv_freq,
                        float attention_scaling, int32_t start, int32_t stride, int32_t inverse,
                        void* stream_) {
  hipStream_t stream = (hipStream_t)stream_;
  FSA_CHECK_ARG(x && out && cu_seqlens && inv_freq, "fsa_rope: null pointer");
  FSA_CHECK_ARG(dtype == FSA_BF16 || dtype == FSA_FP16, "fsa_rope: dtype must be bf16 or fp16");
  FSA_CHECK_ARG(head_dim >= 16 && head_dim % 16 == 0 && head_dim <= 1024,
                "fsa_rope: head_dim must be a multiple of 16, at most 1024");
  FSA_CHECK_ARG(batch >= 1 && num_heads >= 1, "fsa_rope: bad sizes");
  if (total_tokens == 0) return 0;
  const unsigned grid = (unsigned)((total_tokens + 3) / 4);  // one wave per token
  ProfScope ps_("rope", stream);
#define FSA_ROPE(TT, LPR)                                                                                      \
  rope_kernel<TT, LPR><<<grid, 256, 0, stream>>>((const TT*)x, x_stride_n, x_stride_h, (TT*)out, o_stride_n,   \
                                                 o_stride_h, cu_seqlens, batch, total_tokens, num_heads,      \
                                                 head_dim, inv_freq, attention_scaling, start, stride, inverse)
#define FSA_ROPE_D(TT)                      \
  if (head_dim == 64) FSA_ROPE(TT, 4);      \
  else if (head_dim == 128) FSA_ROPE(TT, 8);  \
  else if (head_dim == 256) FSA_ROPE(TT, 16); \
  else FSA_ROPE(TT, 0)
  if (dtype == FSA_BF16) {
    FSA_ROPE_D(__bf16);
  } else {
    FSA_ROPE_D(_Float16);
  }
#undef FSA_ROPE_D
#undef FSA_ROPE
  FSA_CHECK_LAUNCH("fsa_rope");
  return 0;
}

template <typename T, int D, int DN>
static int launch_lc_fwd(const LcPair& p, dim3 grid, const int32_t* cu_x, const int32_t* cu_y, int h, int ks, int stride,
                         hipStream_t stream) {
  constexpr int BYTES = LcFwdLds<D, DN>::BYTES;
  static LdsAllowed lds;
  if (int rc_ = allow_lds(lds, (const void*)lc_fwd_kernel<T, D, DN>, BYTES)) return rc_;
  grid.z *= D / DN;
  ProfScope ps_("linear_compress_fwd", stream);
  lc_fwd_kernel<T, D, DN><<<grid, 64 * LCF_WAVES, BYTES, stream>>>(p, cu_x, cu_y, h, ks, stride);
  return 0;
}
// 64 output columns per work-group where the row tiles alone are less than one for every other CU: more work-groups and
// shorter steps against reading the rows of x once per column group.  (One tensor, bias included: 700 tokens x 8 heads
// 19.0 -> 14.4 us, 2000 x 16 25.1 -> 20.6, 5003 x 16 (176 tiles) 32.6 -> 42.2.  Steps of 64 or 128 rows and deeper
// prefetch were no faster.)
template <typename T, int D>
static int lc_fwd_t(const LcPair& p, int n, const int32_t* cu_x, const int32_t* cu_y, int batch, int64_t max_y, int h, int ks,
                    int stride, hipStream_t stream) {
  bool pe = false;
  for (int i = 0; i < n; ++i) pe |= p.t[i].pe != nullptr;
  const int rows = pe ? LCF_ROWS - 1 : LCF_ROWS;
  const dim3 grid((unsigned)((max_y + rows - 1) / rows), batch, n * h);
  if (D > 64 && (int64_t)grid.x * batch * n * h < 128) return launch_lc_fwd<T, D, 64>(p, grid, cu_x, cu_y, h, ks, stride, stream);
  return launch_lc_fwd<T, D, D>(p, grid, cu_x, cu_y, h, ks, stride, stream);
}

template <typename T, int D>
static int lc_bwd_t(const LcPair& p, int n, const int32_t* cu_x, const int32_t* cu_y, int batch, int64_t max_x, int h, int ks,
                    int stride, hipStream_t stream) {
  static LdsAllowed lds1;
  if (int rc_ = allow_lds(lds1, (const void*)lc_dx_kernel<T, D>, LcDxLds<D>::BYTES)) return rc_;
  static LdsAllowed lds2;
  if (int rc_ = allow_lds(lds2, (const void*)lc_dw_kernel<T, D>, LcDwLds<D>::BYTES)) return rc_;
  {
    ProfScope ps_("linear_compress_dx", stream);
    const int64_t m_per_phase = (max_x + stride - 1) / stride;
    // the grid is sized for the longest sequence; shorter sequences recompute their own tiling inside
    const dim3 grid((unsigned)(D / LCB_COLS + stride * ((m_per_phase + LC_ROWS - 1) / LC_ROWS)), batch, n * h);
    lc_dx_kernel<T, D><<<grid, 256, LcDxLds<D>::BYTES, stream>>>(p, cu_x, cu_y, h, ks, stride);
  }
  ProfScope ps_("linear_compress_dw", stream);
  const dim3 grid(LC_DPE_WGS + (D == 64 ? ks / 2 : ks), n * h, D == 64 ? 1 : D / 128);
  lc_dw_kernel<T, D><<<grid, 256, LcDwLds<D>::BYTES, stream>>>(p, cu_x, cu_y, batch, h, ks, stride);
  return 0;
}

#define FSA_LC_DISPATCH(FN, ...)                                             \
  (dtype == FSA_BF16 ? (d == 64    ? FN<__bf16, 64>(__VA_ARGS__)             \
                        : d == 128 ? FN<__bf16, 128>(__VA_ARGS__)            \
                                   : FN<__bf16, 256>(__VA_ARGS__))           \
                     : (d == 64    ? FN<_Float16, 64>(__VA_ARGS__)           \
                        : d == 128 ? FN<_Float16, 128>(__VA_ARGS__)          \
                                   : FN<_Float16, 256>(__VA_ARGS__)))

int fsa::linear_compress_fwd(const LcTensors* t, int n, int dtype, const int32_t* cu_x, const int32_t* cu_y, int batch,
                             int64_t max_y, int h, int d, int ks, int stride, hipStream_t stream) {
  LcPair p = {};
  for (int i = 0; i < n; ++i) p.t[i] = t[i];
  const int rc = FSA_LC_DISPATCH(lc_fwd_t, p, n, cu_x, cu_y, batch, max_y, h, ks, stride, stream);
  if (rc) return rc;
  FSA_CHECK_LAUNCH("fsa_linear_compress_fwd");
  return 0;
}

int fsa::linear_compress_bwd(const LcTensors* t, int n, int dtype, const int32_t* cu_x, const int32_t* cu_y, int batch,
                             int64_t max_x, int h, int d, int ks, int stride, hipStream_t stream) {
  LcPair p = {};
  for (int i = 0; i < n; ++i) p.t[i] = t[i];
  const int rc = FSA_LC_DISPATCH(lc_bwd_t, p, n, cu_x, cu_y, batch, max_x, h, ks, stride, stream);
  if (rc) return rc;
  FSA_CHECK_LAUNCH("fsa_linear_compress_bwd");
  return 0;
}

extern "C" int fsa_linear_compress_fwd(const void* x, const void* w, const void* pe, int32_t dtype,
                                       int64_t x_stride_n, int64_t x_stride_h, const int32_t* cu_seqlens_x,
                                       const int32_t* cu_seqlens_y, int32_t batch, int64_t max_seqlen_y,
                                       int32_t num_heads, int32_t head_dim, int32_t kernel_size,
                                       int32_t kernel_stride, void* y, void* /*bias_scratch*/, void* stream_) {
  FSA_CHECK_ARG(x && w && y && cu_seqlens_x && cu_seqlens_y, "fsa_linear_compress_fwd: null pointer");
  FSA_CHECK_ARG(dtype == FSA_BF16 || dtype == FSA_FP16, "fsa_linear_compress_fwd: dtype must be bf16 or fp16");
  FSA_CHECK_ARG(head_dim == 64 || head_dim == 128 || head_dim == 256,
                "fsa_linear_compress_fwd: head_dim=%d not supported (64, 128, 256)", head_dim);
  FSA_CHECK_ARG(kernel_stride >= 1 && kernel_size % kernel_stride == 0,
                "fsa_linear_compress_fwd: kernel_size must be a multiple of kernel_stride");
  FSA_CHECK_ARG((uintptr_t)pe % 16 == 0, "fsa_linear_compress_fwd: pe must be 16-byte aligned");
  if (max_seqlen_y <= 0) return 0;
  LcTensors t = {};
  t.x = x; t.w = w; t.pe = pe; t.x_sn = x_stride_n; t.x_sh = x_stride_h; t.y = y;
  return linear_compress_fwd(&t, 1, dtype, cu_seqlens_x, cu_seqlens_y, batch, max_seqlen_y, num_heads, head_dim, kernel_size,
                             kernel_stride, (hipStream_t)stream_);
}

extern "C" int fsa_linear_compress_bwd(const void* x, const void* w, const void* pe, const void* dy,
                                       int32_t dtype, int64_t x_stride_n, int64_t x_stride_h,
                                       const int32_t* cu_seqlens_x, const int32_t* cu_seqlens_y,
                                       int32_t batch, int64_t max_seqlen_x, int64_t total_y,
                                       int32_t num_heads, int32_t head_dim, int32_t kernel_size,
                                       int32_t kernel_stride, void* dx, void* dw, void* dpe,
                                       float* dbias_scratch, void* stream_) {
  FSA_CHECK_ARG(x && w && dy && dx && dw && cu_seqlens_x && cu_seqlens_y, "fsa_linear_compress_bwd: null pointer");
  FSA_CHECK_ARG(dtype == FSA_BF16 || dtype == FSA_FP16, "fsa_linear_compress_bwd: dtype must be bf16 or fp16");
  FSA_CHECK_ARG(head_dim == 64 || head_dim == 128 || head_dim == 256,
                "fsa_linear_compress_bwd: head_dim=%d not supported (64, 128, 256)", head_dim);
  FSA_CHECK_ARG(head_dim != 64 || kernel_size % 2 == 0, "fsa_linear_compress_bwd: head_dim 64 needs an even kernel_size");
  FSA_CHECK_ARG(kernel_stride >= 1 && kernel_size % kernel_stride == 0,
                "fsa_linear_compress_bwd: kernel_size must be a multiple of kernel_stride");
  FSA_CHECK_ARG(!pe || (dpe && dbias_scratch), "fsa_linear_compress_bwd: dpe and dbias scratch needed with pe");
  FSA_CHECK_ARG(max_seqlen_x >= 1, "fsa_linear_compress_bwd: bad max_seqlen_x");
  LcTensors t = {};
  t.x = x; t.w = w; t.pe = pe; t.dy = dy; t.x_sn = x_stride_n; t.x_sh = x_stride_h; t.dx = dx; t.dw = dw; t.dpe = dpe;
  t.dbias = dbias_scratch;
  return linear_compress_bwd(&t, 1, dtype, cu_seqlens_x, cu_seqlens_y, batch, max_seqlen_x, num_heads, head_dim, kernel_size,
                             kernel_stride, (hipStream_t)stream_);
}

extern "C" int fsa_gate_merge_fwd(const void* a, const void* b, const void* c, const void* gate, int32_t dtype,
                                  int64_t total_tokens, int32_t row_elems, void* out, void* stream_) {
  hipStream_t stream = (hipStream_t)stream_;
  FSA_CHECK_ARG(a && b && c && gate && out, "fsa_gate_merge_fwd: null pointer");
  FSA_CHECK_ARG(dtype == FSA_BF16 || dtype == FSA_FP16, "fsa_gate_merge_fwd: dtype must be bf16 or fp16");
  FSA_CHECK_ARG(row_elems >= 8 && row_elems % 8 == 0, "fsa_gate_merge_fwd: row_elems must be a multiple of 8");
  if (total_tokens <= 0) return 0;
  const unsigned grid = (unsigned)((total_tokens + 3) / 4);
  ProfScope ps_("gate_merge_fwd", stream);
  if (dtype == FSA_BF16)
    gate_merge_fwd_kernel<__bf16><<<grid, 256, 0, stream>>>((const __bf16*)a, (const __bf16*)b, (const __bf16*)c,
                                                            (const __bf16*)gate, (__bf16*)out, total_tokens, row_elems);
  else
    gate_merge_fwd_kernel<_Float16><<<grid, 256, 0, stream>>>((const _Float16*)a, (const _Float16*)b,
                                                              (const _Float16*)c, (const _Float16*)gate,
                                                              (_Float16*)out, total_tokens, row_elems);
  FSA_CHECK_LAUNCH("fsa_gate_merge_fwd");
  return 0;
}

extern "C" int fsa_gate_merge_bwd(const void* d_out, const void* a, const void* b, const void* c,
                                  const void* gate, int32_t dtype, int64_t total_tokens, int32_t row_elems,
                                  void* d_a, void* d_b, void* d_c, void* d_gate, void* stream_) {
  hipStream_t stream = (hipStream_t)stream_;
  FSA_CHECK_ARG(d_out && a && b && c && gate && d_a && d_b && d_c && d_gate, "fsa_gate_merge_bwd: null pointer");
  FSA_CHECK_ARG(dtype == FSA_BF16 || dtype == FSA_FP16, "fsa_gate_merge_bwd: dtype must be bf16 or fp16");
  FSA_CHECK_ARG(row_elems >= 8 && row_elems % 8 == 0, "fsa_gate_merge_bwd: row_elems must be a multiple of 8");
  if (total_tokens <= 0) return 0;
  const unsigned grid = (unsigned)((total_tokens + 3) / 4);
  ProfScope ps_("gate_merge_bwd", stream);
  if (dtype == FSA_BF16)
    gate_merge_bwd_kernel<__bf16><<<grid, 256, 0, stream>>>(
        (const __bf16*)d_out, (const __bf16*)a, (const __bf16*)b, (const __bf16*)c, (const __bf16*)gate,
        (__bf16*)d_a, (__bf16*)d_b, (__bf16*)d_c, (__bf16*)d_gate, total_tokens, row_elems);
  else
    gate_merge_bwd_kernel<_Float16><<<grid, 256, 0, stream>>>(
        (const _Float16*)d_out, (const _Float16*)a, (const _Float16*)b, (const _Float16*)c, (const _Float16*)gate,
        (_Float16*)d_a, (_Float16*)d_b, (_Float16*)d_c, (_Float16*)d_gate, total_tokens, row_elems);
  FSA_CHECK_LAUNCH("fsa_gate_merge_bwd");
  return 0;
}
