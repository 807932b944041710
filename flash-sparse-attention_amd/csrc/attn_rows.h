// Query-major attention of a wave: 32 rows (query, head) against 32 keys in a step, K and V from LDS tiles that buffer loads
// fill past the registers.  What the selected forward of short sequences (selattn_direct.hip) and the dense forward
// (cmpattn.hip) have in common.
#pragma once
#include "fsa_common.h"

namespace fsa {

// Four KB of a tile, global memory to LDS: lane l's 16 bytes at voff[j](l) + 1024 j of the buffer land at LDS byte
// `lds` + 1024 j + 16 l (the instruction's offset moves both addresses).
__device__ __forceinline__ void lds_dma4(__amdgpu_buffer_rsrc_t rsrc, const uint32_t* voff, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %5\n\ts_nop 0\n\t"
               "buffer_load_dwordx4 %0, %4, 0 offen lds\n\t"
               "buffer_load_dwordx4 %1, %4, 0 offen offset:1024 lds\n\t"
               "buffer_load_dwordx4 %2, %4, 0 offen offset:2048 lds\n\t"
               "buffer_load_dwordx4 %3, %4, 0 offen offset:3072 lds"
               :: "v"(voff[0]), "v"(voff[1]), "v"(voff[2]), "v"(voff[3]), "s"(rsrc), "s"(lds) : "memory");
}

// The loads of all waves of the work-group have landed, and all of them have read what is overwritten next.
__device__ __forceinline__ void tiles_arrived() { asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// Tiles of 32 K or V rows of a sequence and kv head on their way to LDS.  ANY: of rows that are not 16-byte aligned or lie on
// top of each other; they go through the registers: fetch, and land once there is nothing else to do.
template <typename T, int D, bool ANY = false> struct TileLoads {
  static constexpr int CPR = D / 8, RPI = 64 / CPR, N = 32 / RPI;   // 16-byte chunks per row, rows per load, loads per tile
  static constexpr int NV = RPI >= 4 ? 4 : 16 / RPI;   // lane offsets: 16 rows or more, after which chunk_swizzle repeats itself
  static constexpr int BYTES = 32 * D * 2;
  const char* base;
  uint32_t row_bytes, voff[NV];   // (host: 32 rows span < 2^31 bytes)
  int len;
  __device__ __forceinline__ TileLoads(const void* x, int64_t sn, int64_t sh, int row0, int h, int len_) : len(__builtin_amdgcn_readfirstlane(len_)) {
    const uint64_t b = (uint64_t)(reinterpret_cast<const T*>(x) + (int64_t)row0 * sn + (int64_t)h * sh);   // (uniform, as len and key)
    base = reinterpret_cast<const char*>((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(b >> 32)) << 32 |
                                         (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)b));
    row_bytes = (uint32_t)sn * 2;
    const int lane = threadIdx.x & 63, ld_row = lane / CPR, ld_chunk = lane % CPR;
    // The loading lane picks its source so that the chunks land where chunk_swizzle wants them.  (host: rows are at least 2 D
    // bytes apart where they go straight, so the difference is not negative)
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      const int r = j * RPI + ld_row;
      voff[j] = r * row_bytes + (ld_chunk ^ chunk_swizzle<D>(r)) * 16 - (j & 3) * 1024;
    }
  }
  // PARTS > 1: one of as many equal shares of the loads.  Rows behind the end of the sequence are out of the range of the
  // descriptors and arrive as zeros: no query of the sequence sees them; one at a position behind it does, with score 0, as in
  // the block-major kernels.
  typedef typename Elem<T>::vec8 vec8;
  template <int PARTS> __device__ __forceinline__ void fetch(vec8 (&x)[N / PARTS], int key, int part) const {
    const int lane = threadIdx.x & 63, c = lane % CPR;
#pragma unroll
    for (int i = 0; i < N / PARTS; ++i) {
      const int r = key + (part * (N / PARTS) + i) * RPI + lane / CPR;
      x[i] = load16_at<vec8>(reinterpret_cast<uint64_t>(base) + (uint64_t)(uint32_t)min(r, len - 1) * row_bytes + c * 16);
      if (r >= len) x[i] = zero8<T>();
    }
  }
  template <int PARTS> __device__ __forceinline__ void land(const vec8 (&x)[N / PARTS], uint32_t to, int part) const {
    const int lane = threadIdx.x & 63, c = lane % CPR;
#pragma unroll
    for (int i = 0; i < N / PARTS; ++i) {
      const int r = (part * (N / PARTS) + i) * RPI + lane / CPR;
      store16(const_cast<T*>(lds_ptr<T>(to + r * (D * 2) + (c ^ chunk_swizzle<D>(r)) * 16)), x[i]);
    }
  }
  template <int PARTS = 1> __device__ __forceinline__ void issue(int key, uint32_t to, int part = 0) const {
    static_assert(N / PARTS >= NV, "a share has whole descriptors");
    if constexpr (ANY) {
      vec8 x[N / PARTS];
      fetch<PARTS>(x, key, part);
      land<PARTS>(x, to, part);
      return;
    }
#pragma unroll
    for (int i = 0; i < N / PARTS; i += NV) {
      const int j0 = part * (N / PARTS) + i, first = key + j0 * RPI;
      int rows = max(len - first, 0);   // of the sequence
      asm("" : "+s"(rows));             // (a clamp would be formed by the vector unit)
      rows = min(rows, 32);             // as many as the descriptor serves, or more
      const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(
          const_cast<char*>(base + (uint64_t)(uint32_t)first * row_bytes), 0, (int)((uint32_t)rows * row_bytes), 0x00020000);
#pragma unroll
      for (int j = 0; j < NV; j += 4) lds_dma4(rsrc, &voff[j], to + (j0 + j) * 1024);
    }
  }
};

// Fragments of the tiles, relative to a tile's start: k-step ks of K at k ^ 16 ks, 32 dims from 32 dt of V at v ^ 64 dt.
template <int D> struct TileFrags {
  uint32_t k, v;
  __device__ __forceinline__ TileFrags() {
    const int lane = threadIdx.x & 63, col = lane & 31, hh = lane >> 5, vr = 4 * hh + ((lane & 15) >> 2);
    k = col * (D * 2) + (((hh * (D / 16)) ^ chunk_swizzle<D>(col)) << 4);
    v = vr * (D * 2) + (((2 * ((lane >> 4) & 1) + ((lane & 3) >> 1)) ^ chunk_swizzle<D>(vr)) << 4) + (lane & 1) * 8;
  }
};

// What a wave keeps of its row tile: one row per pair of lanes (col, col + 32).
template <typename T, int D> struct AttnRows {
  typedef typename Elem<T>::vec8 vec8;
  static constexpr int NKS = D / 16, NDT = D / 32;
  float scale_log2;
  int qpos;               // position of the lane's query
  vec8 q[NKS];            // dims hh D/2 + 8 ks .. + 7
  float mref, l;          // reference maximum (scaled scores), sum
  f32x16 o[NDT];

  __device__ __forceinline__ void load_q(const T* row) {
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) q[ks] = load16<vec8>(row + ((threadIdx.x & 63) >> 5) * (D / 2) + ks * 8);
  }
  // The same by way of an LDS tile of the wave's own: a load instruction of whole rows touches 64 / (D / 8) rows instead of 32.
  // `row`: the row of lane col and of lane col + 32.
  static __device__ __forceinline__ void rows_fetch(vec8 (&x)[TileLoads<T, D>::N], const T* row) {
    typedef TileLoads<T, D> L;
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int j = 0; j < L::N; ++j) x[j] = load16_at<vec8>(shfl64((uint64_t)row, j * L::RPI + lane / L::CPR) + lane % L::CPR * 16);
  }
  static __device__ __forceinline__ void rows_to_frags(vec8 (&frag)[NKS], const vec8 (&x)[TileLoads<T, D>::N], T* tile, const TileFrags<D>& f) {
    typedef TileLoads<T, D> L;
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int j = 0; j < L::N; ++j) {
      const int r = j * L::RPI + lane / L::CPR;
      store16(tile + r * D + (lane % L::CPR ^ chunk_swizzle<D>(r)) * 8, x[j]);
    }
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) frag[ks] = load16<vec8>(lds_ptr<T>(lds_addr(tile) + (f.k ^ (16u * ks))));
  }
  __device__ __forceinline__ void load_q_rows(const T* row, T* tile, const TileFrags<D>& f) {
    vec8 x[TileLoads<T, D>::N];
    rows_fetch(x, row);
    rows_to_frags(q, x, tile, f);
  }
  // o * scale to the rows `row` of the lanes, by way of such a tile; rows whose lanes are not `valid` are left out
  __device__ __forceinline__ void store_rows(T* row, bool valid, float scale, T* tile) const {
    typedef TileLoads<T, D> L;
    const int lane = threadIdx.x & 63, col = lane & 31, hh = lane >> 5;
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
      for (int qd = 0; qd < 4; ++qd) {
        typename Elem<T>::vec4 x;
#pragma unroll
        for (int e = 0; e < 4; ++e) x[e] = (T)(o[dt][4 * qd + e] * scale);
        store8(tile + col * D + ((4 * dt + qd) ^ chunk_swizzle<D>(col)) * 8 + 4 * hh, x);
      }
    __builtin_amdgcn_wave_barrier();
    const uint64_t live = __ballot(valid);
#pragma unroll
    for (int j = 0; j < L::N; ++j) {
      const int r = j * L::RPI + lane / L::CPR;
      const vec8 x = load16<vec8>(tile + r * D + (lane % L::CPR ^ chunk_swizzle<D>(r)) * 8);
      const uint64_t to = shfl64((uint64_t)row, r) + lane % L::CPR * 16;
      if (live >> r & 1) store16_at(to, x);
    }
  }
  // q settled: otherwise the compiler waits for it where it is used first, inside the loop and in every step of it, and with it
  // for the tile that was requested a moment before
  __device__ __forceinline__ void settle_q() {
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) asm volatile("" : "+v"(q[ks]));
  }
  __device__ __forceinline__ void clear() {
    mref = -INFINITY;
    l = 0.f;
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
      for (int i = 0; i < 16; ++i) o[dt][i] = 0.f;
  }
  __device__ __forceinline__ void causal(f32x16& s, int key) const {
    const int limit = qpos - key, hh = (threadIdx.x & 63) >> 5;
#pragma unroll
    for (int i = 0; i < 16; ++i)
      if (8 * (i >> 2) + 4 * hh + (i & 3) > limit) s[i] = -INFINITY;
  }
  static __device__ __forceinline__ float lane_max(const f32x16& s) {
    float mx = s[0];
#pragma unroll
    for (int i = 1; i < 16; ++i) mx = fmaxf(mx, s[i]);
    return mx;
  }
  // the reference maximum after scores whose maximum over the lane's own keys is mx
  __device__ __forceinline__ void raise(float mx, bool on) {
    mx = max32(mx) * scale_log2;
    asm volatile("" : "+v"(mx));   // (a select, not a branch over what was computed above)
    mx = on ? mx : -INFINITY;
    // a row that has seen no key yet takes its first maximum as it is: there is nothing to rescale
    mref = mref == -INFINITY ? mx : mref;
    // as in the dense kernels: the reference maximum moves only when some row outgrows it by more than 2^8
    if (__builtin_expect(__any(mx > mref + 8.f), 0)) {
      const float top = fmaxf(mref, mx), alpha = top == -INFINITY ? 1.f : fast_exp2(mref - top);
      l *= alpha;
#pragma unroll
      for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[dt][i] *= alpha;
      mref = top;
    }
  }
  __device__ __forceinline__ float reference(bool on) const { return !on ? INFINITY : mref == -INFINITY ? 0.f : mref; }   // 2^(s - inf) = 0
  __device__ __forceinline__ bool has_nan() const {
    float x = l;
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
      for (int i = 0; i < 16; ++i) x += o[dt][i];
    return x != x;
  }
  // The two halves of a step in the kernels whose waves always have work for the matrix and for the vector unit: scores of the
  // coming step beside the exponentials of this one (EXPS), products with V beside the maximum of the coming scores.
  template <bool EXPS> __device__ __forceinline__ void scores(f32x16& next, const f32x16& s, float ref, vec8 (&pk)[2], uint32_t k_tile, const TileFrags<D>& f) {
    constexpr int AHEAD = 2;   // fragments requested ahead
    vec8 kf[AHEAD + 1];
    float sum = 0.f;
#pragma unroll
    for (int i = 0; i < 16; ++i) next[i] = 0.f;
    auto read = [&](int ks) { kf[ks % (AHEAD + 1)] = load16<vec8>(lds_ptr<T>(k_tile + (f.k ^ (16u * ks)))); };
#pragma unroll
    for (int ks = 0; ks < AHEAD; ++ks) read(ks);
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) {
      if (ks + AHEAD < NKS) read(ks + AHEAD);
      next = Elem<T>::mfma32(kf[ks % (AHEAD + 1)], q[ks], next);
      if constexpr (EXPS) {
#pragma unroll
        for (int i = ks * 16 / NKS; i < (ks + 1) * 16 / NKS; ++i) {
          const float pv = fast_exp2(s[i] * scale_log2 - ref);
          sum += pv;
          pk[i >> 3][i & 7] = (T)pv;
          if ((i & 7) == 7) asm volatile("" : "+v"(pk[i >> 3]), "+v"(sum));   // (here, not in front of its use)
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    if (EXPS) l += sum;   // the lane's own keys: the two lanes of a row are added at the end
  }
  __device__ __forceinline__ float values(const f32x16& next, const vec8 (&pk)[2], uint32_t v_tile, const TileFrags<D>& f) {
    constexpr int AHEAD = 3;
    vec8 vf[AHEAD + 1];
    auto read = [&](int i) { vf[i % (AHEAD + 1)] = swizzled_tr_frag<T, D>(v_tile + (f.v ^ (64u * (i % NDT))), i / NDT); };
#pragma unroll
    for (int i = 0; i < AHEAD; ++i) read(i);
    float mx = -INFINITY;
#pragma unroll
    for (int i = 0; i < 2 * NDT; ++i) {
      if (i + AHEAD < 2 * NDT) read(i + AHEAD);
      o[i % NDT] = Elem<T>::mfma32(vf[i % (AHEAD + 1)], pk[i / NDT], o[i % NDT]);
#pragma unroll
      for (int x = i * 8 / NDT; x < (i + 1) * 8 / NDT; ++x) mx = fmaxf(mx, next[x]);
      __builtin_amdgcn_sched_barrier(0);
    }
    return mx;
  }
  // A step of the second pass, K and V through the wave's own 2 tiles at LDS address `own`: a block that a query did not select
  // must not reach it at all (a key or value of it that is infinite or NaN makes 0 * x NaN in the products), and a block that a
  // list names several times (`times`) counts as often.
  __device__ __forceinline__ void step_carefully(const TileLoads<T, D>& k, const TileLoads<T, D>& v, const TileFrags<D>& f, uint32_t own,
                                                 int key, bool on, float times) {
    k.issue(key, own);
    v.issue(key, own + k.BYTES);
    vm_wait<0>();
    f32x16 s;
#pragma unroll
    for (int i = 0; i < 16; ++i) s[i] = 0.f;
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) s = Elem<T>::mfma32(load16<vec8>(lds_ptr<T>(own + (f.k ^ (16u * ks)))), q[ks], s);
#pragma unroll
    for (int i = 0; i < 16; ++i) s[i] = on ? s[i] : -INFINITY;
    causal(s, key);
    raise(lane_max(s), on);
    const float ref = reference(on);
    vec8 pk[2];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const float pv = on ? fast_exp2(s[i] * scale_log2 - ref) * times : 0.f;
      l += pv;
      pk[i >> 3][i & 7] = (T)pv;
    }
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int dt = 0; dt < NDT; ++dt) {
        const f32x16 x = Elem<T>::mfma32(swizzled_tr_frag<T, D>(own + k.BYTES + (f.v ^ (64u * dt)), j), pk[j], o[dt]);
#pragma unroll
        for (int i = 0; i < 16; ++i) o[dt][i] = on ? x[i] : o[dt][i];
      }
    lds_reads_done();
  }
  // the wave's partial result: [32][D] fp32, 16-byte chunk c of row r at c ^ r; reference and sum to st_m[r], st_l[r]
  static constexpr int XM = D / 4 - 1 < 31 ? D / 4 - 1 : 31;
  __device__ __forceinline__ void park(float* part, float* st_m, float* st_l) const {
    const int lane = threadIdx.x & 63, col = lane & 31, hh = lane >> 5;
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
      for (int qd = 0; qd < 4; ++qd) {
        const int c = (dt * 8 + 2 * qd + hh) ^ (col & XM);
        *reinterpret_cast<f32x4*>(part + col * D + c * 4) = f32x4{o[dt][4 * qd], o[dt][4 * qd + 1], o[dt][4 * qd + 2], o[dt][4 * qd + 3]};
      }
    if (hh == 0) {
      st_m[col] = mref;
      st_l[col] = l;
    }
  }
};

}  // namespace fsa
