// Selected attention of short sequences, straight from the block lists: no inverted index, no partial rows.
//
// Where a sequence has few blocks, the rows (query, head-in-group) of a query tile together select nearly every block they
// may see, and a query-major kernel that visits the union of their blocks does little more arithmetic than the block-major
// pair (selattn_fwd_main / _reduce) while it reads q once and writes o once.
//
// A work-group takes 32 rows; its KG waves share out the visited keys, 32 at a time, each with all 32 rows and K / V buffers of
// its own that it fills by itself (buffer loads straight into LDS), so there is no barrier between the first step and the merge
// of the partial results in LDS.
#include "fsa_common.h"

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
  int64_t n_tokens;
  float scale_log2;
  void* o;
  float* lse;
  MergeEpilogue merge;
};


constexpr int DIR_ROWS = 32;         // rows per work-group
constexpr int DIR_MAX_BLOCKS = 1024; // of a sequence: size of the tables in LDS
constexpr uint32_t DIR_BUFFER = 1u << 31;  // bytes of the K / V buffer descriptors (host: a head's rows span less)

template <int D, int KG> struct DirectLds {
  static constexpr int TILE = 32 * D * 2;                   // 32 K or V rows, bytes
  static constexpr int WAVE_BYTES = 2 * TILE;               // K and V of a wave; at the end its fp32 partial [32][D]
  static constexpr int STATS = 2 * KG * DIR_ROWS * 4;       // (m, l) of every wave
  static constexpr int bytes(int max_blk) { return KG * WAVE_BYTES + STATS + 16 + 6 * max_blk; }
};

// Four KB of a tile, global memory to LDS: lane l's 16 bytes at voff[j](l) + soff + 1024 j of the buffer land at LDS byte
// `lds` + 1024 j + 16 l (the instruction's offset moves both addresses).
__device__ __forceinline__ void lds_dma4(__amdgpu_buffer_rsrc_t rsrc, const uint32_t* voff, uint32_t soff, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %6\n\ts_nop 0\n\t"
               "buffer_load_dwordx4 %0, %4, %5 offen lds\n\t"
               "buffer_load_dwordx4 %1, %4, %5 offen offset:1024 lds\n\t"
               "buffer_load_dwordx4 %2, %4, %5 offen offset:2048 lds\n\t"
               "buffer_load_dwordx4 %3, %4, %5 offen offset:3072 lds"
               :: "v"(voff[0]), "v"(voff[1]), "v"(voff[2]), "v"(voff[3]), "s"(rsrc), "s"(soff), "s"(lds) : "memory");
}
// A row tile.  The rows of the whole buffer are dealt out, so that none of o and lse stays unwritten where the sequences do not
// fill it: segment i runs from cu[i - 1] to cu[i], with the start of the buffer in front and its end behind.  Segment 0, in
// front of the first sequence, has no keys; the last one holds the last sequence and, as queries at the positions behind it,
// the tokens that follow it, which is where the inverted index counts them too.
struct DirectTile {
  int q0, n_q, len;   // first token, queries and keys of its segment
  int tile;           // of the segment
};
// Row tile of work-group `id`; false: past the last tile.  The late tiles of a segment, which see the most blocks, come first.
__device__ __forceinline__ bool direct_tile(const int32_t* __restrict__ cu, int batch, int n_tokens, int g, int id, DirectTile& t) {
  const int lane = threadIdx.x & (WAVE - 1);
  for (int s0 = 0; s0 <= batch; s0 += WAVE) {
    const int si = s0 + lane;
    const int a = cu[min(max(si - 1, 0), batch)], b = cu[min(si, batch)];
    const int q0 = si > 0 ? a : 0, n_q = (si < batch ? b : n_tokens) - q0;
    const int n = si <= batch ? (int)(((int64_t)n_q * g + DIR_ROWS - 1) / DIR_ROWS) : 0;
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

template <typename T, int D, int BK, int KG, bool MERGE>
__global__ void __launch_bounds__(64 * KG, D <= 128 ? 2 : 1)
selattn_direct_fwd_kernel(DirectParams p) {
  typedef typename Elem<T>::vec8 vec8;
  typedef DirectLds<D, KG> L;
  constexpr int NKS = D / 16, NDT = D / 32, NT = 64 * KG;
  constexpr int CPR = D / 8, RPI = 64 / CPR, NLD = 32 / RPI;   // 16-byte chunks per row, rows and number of loads of a tile
  constexpr int UPB = BK / 32;                                 // steps of 32 keys per block
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
  float* st_m = reinterpret_cast<float*>(smem + KG * L::WAVE_BYTES);   // [wave][row]
  float* st_l = st_m + KG * DIR_ROWS;
  int* info = reinterpret_cast<int*>(st_l + KG * DIR_ROWS);     // [0] list length, [1] a list names a block twice
  uint32_t* sel = reinterpret_cast<uint32_t*>(info + 4);        // [block]: bit i = query q_first + i
  uint16_t* list = reinterpret_cast<uint16_t*>(sel + p.max_blk);   // visited blocks

  const int h = blockIdx.x % p.hkv;
  DirectTile t;
  if (!direct_tile(p.cu, p.batch, (int)p.n_tokens, p.g, blockIdx.x / p.hkv, t)) return;
  const int q0 = t.q0, len = t.len, rows = t.n_q * p.g, row0 = t.tile * DIR_ROWS;
  const int q_first = div_group(row0, p.g, p.g_shift), q_last = div_group(min(rows, row0 + DIR_ROWS) - 1, p.g, p.g_shift);
  const int n_blk = min(q_last / BK + 1, (len + BK - 1) / BK);
  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 31, hh = lane >> 5;

  // q fragments: dims hh D/2 + 8 ks .. + 7
  const int row = min(row0 + col, rows - 1);
  const int qpos = div_group(row, p.g, p.g_shift), qoff = qpos - q_first;
  vec8 qreg[NKS];
  {
    const T* qrow = reinterpret_cast<const T*>(p.q) + (int64_t)(q0 + qpos) * p.q_sn + (int64_t)(h * p.g + row - qpos * p.g) * p.q_sh +
                    hh * (D / 2);
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) qreg[ks] = load16<vec8>(qrow + ks * 8);
  }

  // ---- K / V tiles ----
  const uint32_t k_row = (uint32_t)p.k_sn * 2, v_row = (uint32_t)p.v_sn * 2;   // bytes (host: a head's rows span < 2^31)
  const __amdgpu_buffer_rsrc_t k_rsrc = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<T*>(reinterpret_cast<const T*>(p.k) + (int64_t)q0 * p.k_sn + (int64_t)h * p.k_sh), 0, (int)DIR_BUFFER, 0x00020000);
  const __amdgpu_buffer_rsrc_t v_rsrc = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<T*>(reinterpret_cast<const T*>(p.v) + (int64_t)q0 * p.v_sn + (int64_t)h * p.v_sh), 0, (int)DIR_BUFFER, 0x00020000);
  const uint32_t k_lds = lds_addr(smem + wv * L::WAVE_BYTES), v_lds = k_lds + L::TILE;
  // (the loading lane picks its source so that the chunks land where chunk_swizzle wants them)
  const int ld_row = lane / CPR, ld_chunk = lane % CPR;
  uint32_t k_voff[NLD], v_voff[NLD];
#pragma unroll
  for (int j = 0; j < NLD; ++j) {   // (host: rows are at least 2 D bytes apart, so the difference is not negative)
    const int r = j * RPI + ld_row;
    k_voff[j] = r * k_row + (ld_chunk ^ chunk_swizzle<D>(r)) * 16 - (j & 3) * 1024;
    v_voff[j] = r * v_row + (ld_chunk ^ chunk_swizzle<D>(r)) * 16 - (j & 3) * 1024;
  }
  auto issue = [&](__amdgpu_buffer_rsrc_t rsrc, uint32_t row_bytes, const uint32_t* voff, uint32_t to, int key) {
    if (key + 32 <= len) {
#pragma unroll
      for (int j = 0; j < NLD; j += 4) lds_dma4(rsrc, &voff[j], (uint32_t)key * row_bytes, to + j * 1024);
    } else {
      // A tile that reaches behind the end: zeros there (an offset behind the end of the buffer).  No query of the sequence
      // sees them; one at a position behind it does, with score 0, as in the block-major kernels.
#pragma unroll 1
      for (int j = 0; j < NLD; ++j) {
        const int r = j * RPI + ld_row;
        const uint32_t off =
            key + r < len ? (uint32_t)(key + r) * row_bytes + (ld_chunk ^ chunk_swizzle<D>(r)) * 16 : DIR_BUFFER;
        asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %1, 0 offen lds"
                     :: "v"(off), "s"(rsrc), "s"(to + j * 1024) : "memory");
      }
    }
  };
  auto issue_k = [&](int key) { issue(k_rsrc, k_row, k_voff, k_lds, key); };
  auto issue_v = [&](int key) { issue(v_rsrc, v_row, v_voff, v_lds, key); };
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
  int guess = wv / UPB * BK + wv % UPB * 32;
  if (guess + 32 <= len) {
    issue_k(guess);
    issue_v(guess);
  } else {
    guess = -1;
  }
  for (int b = tid; b < n_blk; b += NT) sel[b] = 0;
  if (tid < 2) info[tid] = 0;
  __syncthreads();
  auto visit = [&](int q, int b) {
    if (b < 0 || b >= n_blk || b > (q_first + q) / BK) return;   // (a block behind the query's own holds no key it may see)
    if (atomicOr(&sel[b], 1u << q) >> q & 1) info[1] = 1;
  };
#pragma unroll
  for (int i = 0; i < AHEAD; ++i)
    if (tid + i * NT < n_ids) visit(qo[i], id[i]);
  for (int e = tid + AHEAD * NT; e < n_ids; e += NT) {
    const int q = (uint32_t)e / (uint32_t)p.topk;
    visit(q, ids[q * p.i_sn + (e - q * p.topk)]);
  }
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
  const int n_units = __builtin_amdgcn_readfirstlane(info[0]) * UPB;
  const int n_steps = (n_units - wv + KG - 1) / KG;   // of this wave
  struct Unit {
    int key;         // position of its first key
    uint32_t mask;   // queries that selected its block
  };
  auto unit = [&](int t) {
    const int u = wv + KG * t;
    const int b = __builtin_amdgcn_readfirstlane(list[u / UPB]);
    return Unit{b * BK + u % UPB * 32, (uint32_t)__builtin_amdgcn_readfirstlane((int)sel[b])};
  };

  // lane addresses of the fragments
  const uint32_t kf_addr = k_lds + col * (D * 2) + (((hh * (D / 16)) ^ chunk_swizzle<D>(col)) << 4);   // k-step ks: ^ 16 ks
  const int vr = 4 * hh + ((lane & 15) >> 2);
  const uint32_t vf_addr = v_lds + vr * (D * 2) + (((2 * ((lane >> 4) & 1) + ((lane & 3) >> 1)) ^ chunk_swizzle<D>(vr)) << 4) + (lane & 1) * 8;
  auto k_frag = [&](int ks) { return load16<vec8>(lds_ptr<T>(kf_addr ^ (16u * ks))); };
  auto v_frag = [&](int j, int dt) { return swizzled_tr_frag<T, D>(vf_addr ^ (64u * dt), j); };   // keys 16 j .., dims 32 dt ..

  float m = -INFINITY, mref = 0.f, l = 0.f;   // reference maximum (raw scores), the same scaled (0 while there is none)
  f32x16 oacc[NDT];
  // CAREFUL: a block that a query did not select must not reach it at all (a key or value of it that is infinite or NaN makes
  // 0 * x NaN in the products), and a block that a list names several times counts as often.
  // At head_dim 128 this pass is 16 registers short: it puts them into scratch (68 bytes) in front of its loop, which the other
  // pass does not touch.
  auto attend = [&](auto careful_, int loaded) {   // loaded: the key of the tiles that are in LDS or on their way there, or -1
    constexpr bool CAREFUL = decltype(careful_)::value;
    m = -INFINITY;
    mref = l = 0.f;
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
      for (int i = 0; i < 16; ++i) oacc[dt][i] = 0.f;
    if (n_steps <= 0 || unit(0).key != loaded) vm_wait<0>();   // (what is on its way would land in what comes now)
    if (n_steps <= 0) return;
    Unit cur = unit(0);
    if (cur.key != loaded) {
      issue_k(cur.key);
      issue_v(cur.key);
    }
    // The counts of vm_wait leave the tile that was requested last on its way, and at head_dim 64 that is what runs.  At 128
    // and 256 the compiler settles qreg, ordinary loads whose first use is in this loop, by waits of its own between the
    // products of S: they run in every step, down to no operation outstanding, so that K of the next step and V of this one
    // are awaited there in full and a step takes the latency of a tile (about 1 us at head_dim 128).
    for (int t = 0;; ++t) {
      const bool more = t + 1 < n_steps;
      const Unit nxt = unit(more ? t + 1 : t);
      vm_wait<NLD>();   // K of this step, not its V
      vec8 kf[NKS];
#pragma unroll
      for (int ks = 0; ks < NKS; ++ks) kf[ks] = k_frag(ks);
      lds_reads_done();
      if (more) issue_k(nxt.key);
      f32x16 acc;
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[i] = 0.f;
#pragma unroll
      for (int ks = 0; ks < NKS; ++ks) acc = Elem<T>::mfma32(kf[ks], qreg[ks], acc);
      const bool on = (cur.mask >> qoff) & 1;
      float times = 1.f;
      if (CAREFUL) {
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[i] = on ? acc[i] : -INFINITY;
        if (twice) {
          const int32_t* ids = p.topk_idx + h * p.i_sh + (int64_t)(q0 + qpos) * p.i_sn;
          int c = 0;
          for (int i = 0; i < p.topk; ++i) c += ids[i] == cur.key / BK;
          times = (float)c;
        }
      }
      if (cur.key + 31 > q_first) {   // some row may see the keys partly
        const int limit = qpos - cur.key;
#pragma unroll
        for (int i = 0; i < 16; ++i)
          if (8 * (i >> 2) + 4 * hh + (i & 3) > limit) acc[i] = -INFINITY;
      }
      float mx = acc[0];
#pragma unroll
      for (int i = 1; i < 16; ++i) mx = fmaxf(mx, acc[i]);
      mx = max32(mx);
      asm volatile("" : "+v"(mx));   // (a select, not a branch over what was computed above)
      mx = fmaxf(m, on ? mx : -INFINITY);
      // a row that has seen no key yet takes its first maximum as it is: there is nothing to rescale
      const bool first = m == -INFINITY;
      mref = first ? (mx == -INFINITY ? 0.f : mx * p.scale_log2) : mref;
      m = first ? mx : m;
      // as in the dense kernels: the reference maximum moves only when some row outgrows it by more than 2^8
      if (__any((mx - m) * p.scale_log2 > 8.f)) {   // (a row without a key: NaN)
        const float alpha = mx == -INFINITY ? 1.f : exp2f((m - mx) * p.scale_log2);
        l *= alpha;
#pragma unroll
        for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
          for (int i = 0; i < 16; ++i) oacc[dt][i] *= alpha;
        m = mx;
        mref = mx == -INFINITY ? 0.f : mx * p.scale_log2;
      }
      const float ref = on ? mref : INFINITY;   // 2^(s - inf) = 0
      float sum = 0.f;
      vec8 pk[2];
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        float pv = fast_exp2(acc[i] * p.scale_log2 - ref);
        if (CAREFUL) pv = on ? pv * times : 0.f;
        sum += pv;
        pk[i >> 3][i & 7] = (T)pv;
      }
      l += sum;   // the lane's own keys: the two lanes of a row are added behind the loop
      if (more) vm_wait<NLD>();   // V of this step, not K of the next (but see above)
      else vm_wait<0>();
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int dt = 0; dt < NDT; ++dt) {
          const f32x16 x = Elem<T>::mfma32(v_frag(j, dt), pk[j], oacc[dt]);
#pragma unroll
          for (int i = 0; i < 16; ++i) oacc[dt][i] = !CAREFUL || on ? x[i] : oacc[dt][i];
        }
      lds_reads_done();
      if (!more) break;
      issue_v(nxt.key);
      cur = nxt;
    }
    l = sum32(l);
  };
  bool careful = twice;
  if (!careful) {
    attend(std::false_type{}, guess);
    float x = 0.f;   // NaN if any accumulator is
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
      for (int i = 0; i < 16; ++i) x += oacc[dt][i];
    careful = __any(x != x || l != l);
  }
  if (careful) attend(std::true_type{}, twice ? guess : -1);

  // ---- merge of the waves ----
  float* part = reinterpret_cast<float*>(smem + wv * L::WAVE_BYTES);   // [32][D], 16-byte chunk c of row r at c ^ r
  constexpr int XM = D / 4 - 1 < 31 ? D / 4 - 1 : 31;
#pragma unroll
  for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
    for (int qd = 0; qd < 4; ++qd) {
      const int c = (dt * 8 + 2 * qd + hh) ^ (col & XM);
      *reinterpret_cast<f32x4*>(part + col * D + c * 4) =
          f32x4{oacc[dt][4 * qd], oacc[dt][4 * qd + 1], oacc[dt][4 * qd + 2], oacc[dt][4 * qd + 3]};
    }
  if (hh == 0) {
    st_m[wv * DIR_ROWS + col] = m == -INFINITY ? -INFINITY : mref;
    st_l[wv * DIR_ROWS + col] = l;
  }
  __syncthreads();
  constexpr int RPP = NT / CPR;   // rows per pass
#pragma unroll
  for (int r0 = 0; r0 < DIR_ROWS; r0 += RPP) {
    const int r = r0 + tid / CPR, sub = tid % CPR;
    if (r >= DIR_ROWS || row0 + r >= rows) break;
    float mw[KG], mx = -INFINITY;
#pragma unroll
    for (int w = 0; w < KG; ++w) {
      mw[w] = st_m[w * DIR_ROWS + r];
      mx = fmaxf(mx, mw[w]);
    }
    float sum = 0.f;
#pragma unroll
    for (int w = 0; w < KG; ++w) {
      mw[w] = mx == -INFINITY ? 0.f : fast_exp2(mw[w] - mx);
      sum += mw[w] * st_l[w * DIR_ROWS + r];
    }
    const float inv = sum == 0.f ? 0.f : 1.f / sum;   // (a sum that is NaN, from a NaN in q or a key, makes the row NaN)
    float out[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) out[e] = 0.f;
#pragma unroll
    for (int w = 0; w < KG; ++w) {
      const float* pw = reinterpret_cast<const float*>(smem + w * L::WAVE_BYTES) + r * D;
      const f32x4 x0 = *reinterpret_cast<const f32x4*>(pw + ((2 * sub) ^ (r & XM)) * 4);
      const f32x4 x1 = *reinterpret_cast<const f32x4*>(pw + ((2 * sub + 1) ^ (r & XM)) * 4);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        out[e] += mw[w] * x0[e];
        out[4 + e] += mw[w] * x1[e];
      }
    }
    vec8 x;
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e] = (T)(out[e] * inv);
    const int qi = div_group(row0 + r, p.g, p.g_shift), hq_i = h * p.g + row0 + r - qi * p.g;
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
      if (!p.o) continue;
    }
    store16(reinterpret_cast<T*>(p.o) + tok * p.o_sn + (int64_t)hq_i * p.o_sh + sub * 8, x);
    if (sub == 0) p.lse[(int64_t)hq_i * p.n_tokens + tok] = sum == 0.f ? -INFINITY : mx + log2f(sum);
  }
}

template <typename T, int D, int BK, int KG, bool MERGE>
static int launch_direct_fwd(const DirectParams& p, int64_t tiles, hipStream_t stream) {
  static LdsAllowed allowed;
  if (int rc = allow_lds(allowed, (const void*)selattn_direct_fwd_kernel<T, D, BK, KG, MERGE>,
                         DirectLds<D, KG>::bytes(DIR_MAX_BLOCKS)))
    return rc;
  ProfScope ps_("selattn_direct_fwd", stream);
  selattn_direct_fwd_kernel<T, D, BK, KG, MERGE>
      <<<(unsigned)((tiles + 1) * p.hkv), 64 * KG, DirectLds<D, KG>::bytes(p.max_blk), stream>>>(p);
  return 0;
}
// Two waves per work-group where there are enough of them to fill the chip: less to merge, and more work-groups in different
// stages on a CU.  (us with four / two waves: 4096 tokens x 4 heads of 128, 512 work-groups, 42 / 65; 4096 x 16, 2048, 115 /
// 114; 2000 x 32, 2000, 71 / 61; 4096 x 32 209 / 197.)
template <typename T, bool MERGE> static int dispatch_direct_fwd(int d, int bk, const DirectParams& p, hipStream_t stream) {
  const int64_t tiles = p.n_tokens * p.g / DIR_ROWS + p.batch;
  const bool two = tiles * p.hkv > 1536;
#define FSA_CASE(DD, BB)                                                                        \
  if (d == DD && bk == BB) {                                                                    \
    if (two) return launch_direct_fwd<T, DD, BB, 2, MERGE>(p, tiles, stream);                   \
    return launch_direct_fwd<T, DD, BB, 4, MERGE>(p, tiles, stream);                            \
  }
  FSA_CASE(128, 32)
  FSA_CASE(128, 64)
  FSA_CASE(128, 128)
  FSA_CASE(64, 32)
  FSA_CASE(64, 64)
  FSA_CASE(64, 128)
  FSA_CASE(256, 32)
  FSA_CASE(256, 64)
  FSA_CASE(256, 128)
#undef FSA_CASE
  set_error("selected attention (direct): head_dim=%d with block_size=%d is not supported", d, bk);
  return FSA_ERR_UNSUPPORTED;
}

// Whether the forward of `n` tokens in sequences of at most `max_len` takes this path.  Both sides in us on one chip, fitted to
// the times below: this kernel visits up to half of a sequence for every row, and its longest work-group works through a whole
// one; the block-major launches work on topk * block keys per row, behind 33 us that do not depend on the size (index, two more
// launches and their gaps), 12 of them for the index, which is no loss where the caller builds it all the same (training).
// Lists of 16 blocks of 64, one sequence; index + block-major / direct / index + direct in us, head_dim 128:
//   4096 tokens x 4 heads 62 / 37 / 53, x 16 (GQA 4) 131 / 101 / 115, x 32 (GQA 4) 233 / 192 / 208; 5000 x 4 69 / 47 / 65;
//   5000 x 32 (GQA 4) 283 / 267 / 284; 6000 x 4 79 / 59 / 78, x 32 (GQA 4) 339 / 354; 7000 x 4 83 / 77; 8192 x 4 100 / 100, x 32
//   505 / 711; 16384 x 4 (GQA 4) 167 / 211
// head_dim 256, lists of 8: 3000 x 4 64 / 47 / 59, 4096 x 4 85 / 74 / 86, 6000 x 8 164 / 175; 64: 4500 x 8 46 / 35 / 46, 8000 x 8
// (16 blocks) 93 / 94.  All of them, and the waves per work-group above, with the kernel's loads drained in every step (see the
// loop): a step that takes less moves the line towards longer sequences.
bool selattn_direct_preferred(int64_t n, int64_t max_len, int hq, int d, int topk, int bk, bool index_needed) {
  if (!(d == 64 || d == 128 || d == 256) || !(bk == 32 || bk == 64 || bk == 128) || topk > 4096 ||
      max_len > (int64_t)bk * DIR_MAX_BLOCKS)
    return false;
  const double rows = (double)n * hq * d / 128, len = (double)max_len;
  const double keys = std::min<double>((double)topk * bk, len);
  return std::hypot(rows * len / 2.95e6, 0.0055 * len) + 5 <= (index_needed ? 21 : 33) + rows * keys / 6.2e5;
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
  DirectParams p = {};
  p.q = q; p.k = k; p.v = v;
  p.q_sn = q_stride_n; p.q_sh = q_stride_h;
  p.k_sn = k_stride_n; p.k_sh = k_stride_h;
  p.v_sn = v_stride_n; p.v_sh = v_stride_h;
  p.o_sn = o_stride_n; p.o_sh = o_stride_h;
  p.topk_idx = topk_idx; p.i_sh = idx_stride_h; p.i_sn = idx_stride_n;
  p.cu = cu_seqlens; p.batch = batch; p.hkv = num_kv_heads; p.g = num_q_heads / num_kv_heads; p.g_shift = group_shift(p.g);
  p.topk = topk; p.max_blk = (int)((max_len + block_size - 1) / block_size); p.n_tokens = total_tokens;
  p.scale_log2 = softmax_scale * LOG2E;
  p.o = o; p.lse = lse; p.merge = merge;
  const int rc = merge.out ? (dtype == FSA_BF16 ? dispatch_direct_fwd<__bf16, true>(head_dim, block_size, p, stream)
                                                : dispatch_direct_fwd<_Float16, true>(head_dim, block_size, p, stream))
                           : (dtype == FSA_BF16 ? dispatch_direct_fwd<__bf16, false>(head_dim, block_size, p, stream)
                                                : dispatch_direct_fwd<_Float16, false>(head_dim, block_size, p, stream));
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
