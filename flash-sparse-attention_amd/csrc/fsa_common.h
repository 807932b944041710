// Shared device helpers for the gfx950 kernels: 16-bit element traits, MFMA
// wrappers, wave64 shuffles, error plumbing for the C ABI.
#pragma once

#include <hip/hip_runtime.h>
#include <atomic>
#include <stdint.h>
#include <stdio.h>
#include <stdarg.h>

#include "../../include/fsa_hip.h"

namespace fsa {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));

constexpr int WAVE = 64;
constexpr float LOG2E = 1.4426950408889634f;

// ---- element traits -------------------------------------------------------
template <typename T> struct Elem;

template <> struct Elem<__bf16> {
  typedef bf16x8 vec8;
  typedef bf16x4 vec4;
  static __device__ __forceinline__ f32x16 mfma32(vec8 a, vec8 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ f32x4 mfma16(vec8 a, vec8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
  }
};

template <> struct Elem<_Float16> {
  typedef f16x8 vec8;
  typedef f16x4 vec4;
  static __device__ __forceinline__ f32x16 mfma32(vec8 a, vec8 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ f32x4 mfma16(vec8 a, vec8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
  }
};

// 16-byte / 8-byte raw moves (global or LDS) reinterpreted as element vectors.
template <typename V> __device__ __forceinline__ V load16(const void* p) {
  uint4 r = *reinterpret_cast<const uint4*>(p);
  return __builtin_bit_cast(V, r);
}
template <typename V> __device__ __forceinline__ void store16(void* p, V v) {
  *reinterpret_cast<uint4*>(p) = __builtin_bit_cast(uint4, v);
}
// The same at an address that was put together from its halves: global memory, which the compiler cannot see (a flat access
// would wait for LDS as well, and for everything that is on its way).
template <typename V> __device__ __forceinline__ V load16_at(uint64_t at) {
  typedef unsigned int u4_ __attribute__((ext_vector_type(4)));
  return __builtin_bit_cast(V, *reinterpret_cast<const __attribute__((address_space(1))) u4_*>(at));
}
template <typename V> __device__ __forceinline__ void store16_at(uint64_t at, V v) {
  typedef unsigned int u4_ __attribute__((ext_vector_type(4)));
  *reinterpret_cast<__attribute__((address_space(1))) u4_*>(at) = __builtin_bit_cast(u4_, v);
}
// x of lane `lane`, 64 bits
__device__ __forceinline__ uint64_t shfl64(uint64_t x, int lane) {
  return (uint64_t)(uint32_t)__shfl((int)(x >> 32), lane, 64) << 32 | (uint32_t)__shfl((int)(uint32_t)x, lane, 64);
}
// The same 16-byte moves for data that is written once and read once by a later kernel (partial rows):
// marked non-temporal so that they do not displace the K / V blocks and query rows that are reused.
template <typename V> __device__ __forceinline__ V load16_stream(const void* p) {
  typedef unsigned int u4_ __attribute__((ext_vector_type(4)));
  u4_ r = __builtin_nontemporal_load(reinterpret_cast<const u4_*>(p));
  return __builtin_bit_cast(V, r);
}
template <typename V> __device__ __forceinline__ void store16_stream(void* p, V v) {
  typedef unsigned int u4_ __attribute__((ext_vector_type(4)));
  __builtin_nontemporal_store(__builtin_bit_cast(u4_, v), reinterpret_cast<u4_*>(p));
}
template <typename V> __device__ __forceinline__ V load8(const void* p) {
  uint2 r = *reinterpret_cast<const uint2*>(p);
  return __builtin_bit_cast(V, r);
}
template <typename V> __device__ __forceinline__ void store8(void* p, V v) {
  *reinterpret_cast<uint2*>(p) = __builtin_bit_cast(uint2, v);
}

// elements p[0..3] and p[16..19] as one 8-element fragment (two 8-byte moves)
template <typename T> __device__ __forceinline__ typename Elem<T>::vec8 load8x2(const T* p) {
  typename Elem<T>::vec4 lo = load8<typename Elem<T>::vec4>(p);
  typename Elem<T>::vec4 hi = load8<typename Elem<T>::vec4>(p + 16);
  return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
}
// ---- hand-issued 8-byte LDS reads --------------------------------------------------------------
// An LDS instruction that returns 16 bytes per lane (ds_read_b128, ds_read2_b64) delivers 64 bytes per clock
// on gfx950, an 8-byte one (ds_read_b64) 128.  The compiler fuses neighbouring 8-byte reads into the 16-byte
// forms, so the reads that should stay separate are issued by hand.  The compiler does not know that their
// results are still in flight: lds_wait() has to be placed between such reads and the first use of their
// results, with every result passed through it.
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ uint32_t lds_addr(const void* p) {
  return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const void*)p;
}
// the LDS pointer for a byte address
template <typename T> __device__ __forceinline__ const T* lds_ptr(uint32_t addr) {
  return (const T*)(__attribute__((address_space(3))) const T*)(uintptr_t)addr;
}
template <int OFFSET_BYTES> __device__ __forceinline__ u32x2 lds_read8_raw(uint32_t addr) {
  static_assert(OFFSET_BYTES >= 0 && OFFSET_BYTES < 65536, "ds offset field");
  u32x2 r;
  asm volatile("ds_read_b64 %0, %1 offset:%2" : "=v"(r) : "v"(addr), "n"(OFFSET_BYTES));
  return r;
}
template <int N> __device__ __forceinline__ void lds_wait(u32x2 (&r)[N]);
template <> __device__ __forceinline__ void lds_wait<6>(u32x2 (&r)[6]) {
  asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(r[0]), "+v"(r[1]), "+v"(r[2]), "+v"(r[3]), "+v"(r[4]), "+v"(r[5]));
}
template <> __device__ __forceinline__ void lds_wait<8>(u32x2 (&r)[8]) {
  asm volatile("s_waitcnt lgkmcnt(0)"
               : "+v"(r[0]), "+v"(r[1]), "+v"(r[2]), "+v"(r[3]), "+v"(r[4]), "+v"(r[5]), "+v"(r[6]), "+v"(r[7]));
}
template <> __device__ __forceinline__ void lds_wait<16>(u32x2 (&r)[16]) {
  asm volatile("s_waitcnt lgkmcnt(0)"
               : "+v"(r[0]), "+v"(r[1]), "+v"(r[2]), "+v"(r[3]), "+v"(r[4]), "+v"(r[5]), "+v"(r[6]), "+v"(r[7]),
                 "+v"(r[8]), "+v"(r[9]), "+v"(r[10]), "+v"(r[11]), "+v"(r[12]), "+v"(r[13]), "+v"(r[14]),
                 "+v"(r[15]));
}
template <typename T> __device__ __forceinline__ typename Elem<T>::vec8 frag8(u32x2 lo, u32x2 hi) {
  u32x4 x = {lo[0], lo[1], hi[0], hi[1]};
  return __builtin_bit_cast(typename Elem<T>::vec8, x);
}

template <typename T> __device__ __forceinline__ typename Elem<T>::vec8 zero8() {
  uint4 z = make_uint4(0, 0, 0, 0);
  return __builtin_bit_cast(typename Elem<T>::vec8, z);
}

// LDS transposing read (gfx950 ds_read_b64_tr_b16).  Inside every group of 16
// lanes, lane j receives, for e = 0..3, element (j % 4) of the 8-byte word whose
// address was supplied by lane 4*e + j/4 of the group.  With lane s pointing at
// M[r0 + (s%16)/4][c0 + 4*(s%4) ..], lane j therefore gets M[r0 + e][c0 + j],
// e = 0..3: four consecutive rows of one column out of a row-major tile.
template <typename T> __device__ __forceinline__ typename Elem<T>::vec4 lds_read_tr4(const T* p) {
  typedef short s16x4 __attribute__((ext_vector_type(4)));
  typedef __attribute__((address_space(3))) s16x4* lds_ptr;
  s16x4 r = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(p));
  return __builtin_bit_cast(typename Elem<T>::vec4, r);
}

// Eight values of one column (two runs of four consecutive rows, 8 rows apart)
// of a row-major LDS tile, as the k-contiguous MFMA operand of a contraction
// over the tile's rows.  `p` is this lane's address for row r0 + (lane%16)/4.
template <typename T>
__device__ __forceinline__ typename Elem<T>::vec8 lds_read_tr8(const T* p, int stride8rows) {
  typename Elem<T>::vec4 lo = lds_read_tr4<T>(p);
  typename Elem<T>::vec4 hi = lds_read_tr4<T>(p + stride8rows);
  return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
}

// transposing read of 8 consecutive rows r0..r0+7 of one column out of a row-major LDS tile:
// this lane supplies the address of row r0 + (lane%16)/4, columns c0 + 4*(lane%4)
template <typename T>
__device__ __forceinline__ typename Elem<T>::vec8 lds_tr8_rows(const T* p, int stride) {
  typename Elem<T>::vec4 lo = lds_read_tr4<T>(p);
  typename Elem<T>::vec4 hi = lds_read_tr4<T>(p + 4 * stride);
  return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
}

// Layout of an unpadded LDS tile that is read by the 32 x 32 products both ways, 32 rows at 16 bytes ("natural") and, per
// half-wave, four rows at 64 bytes (transposing): chunk c (16 bytes) of row r sits in the place of chunk c ^ chunk_swizzle(r).
// A 16-byte read is served in groups of 16 lanes (lanes 0-3, 12-15, 20-23 and 24-27 make the first), an 8-byte one in
// half-waves; both run at 256 bytes per clock where the bytes of a group fall into different ones of the 64 banks.  Measured,
// clocks per wave instruction: this layout 4.0 natural and 2.2 transposing; rows of 2 D + 16 bytes 4.0 and 8.0, 2 D + 32 bytes
// 8.0 and 4.0, 2 D + 64 bytes 16 and 2.1.
template <int D> __device__ __forceinline__ int chunk_swizzle(int r) {
  return D >= 128 ? (r & 3) << 2 | (r >> 2 & 3) : (r >> 1 & 1) << 2 | (r >> 2 & 3);
}
// Transposed fragment of such a tile: rows 16 j + (0..3, 8..11) of the lane's column.  `addr`: the lane's LDS address in row 0
// (byte column XOR 64 dt included); rows that are 8 apart differ in bit 1 of the swizzle.
template <typename T, int D> __device__ __forceinline__ typename Elem<T>::vec8 swizzled_tr_frag(uint32_t addr, int j) {
  const typename Elem<T>::vec4 lo = lds_read_tr4<T>(lds_ptr<T>(addr + 16 * j * D * 2));
  const typename Elem<T>::vec4 hi = lds_read_tr4<T>(lds_ptr<T>((addr ^ 32u) + (16 * j + 8) * D * 2));
  return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
}

// Loads that go to LDS past the registers are not counted by the compiler: vm_wait<N> waits until only the N youngest memory
// operations of the wave are still on the way.
template <int N> __device__ __forceinline__ void vm_wait() {
  asm volatile("s_waitcnt vmcnt(%0)" :: "n"(N) : "memory");
}
__device__ __forceinline__ void lds_reads_done() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

// 2^x by the hardware instruction alone (1 ulp; results below 2^-126 flush to zero, -inf gives 0): the
// library exp2f adds a denormal-range rescaling that costs several VALU operations per element
__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

// Maximum and sum over the two lanes that are 32 apart: a swap of register halves, no trip through the LDS crossbar (which
// a wave of the dense forward would wait for twice per tile: 8192 tokens, 32 heads: 179 -> 173 us).
__device__ __forceinline__ float max32(float v) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float sum32(float v) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// Maximum of a 64-bit key (hi word compared first) over the wave, returned to every lane, without going through the LDS
// crossbar: prefix maxima inside each row of 16 lanes with the DPP row shifts (lanes shifted in from outside a row read 0),
// the rows combined with the two DPP row broadcasts, the result read from the last lane.
template <int CTRL, int ROW_MASK, bool ZERO_FILL> __device__ __forceinline__ uint32_t dpp_move(uint32_t x) {
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, CTRL, ROW_MASK, 0xf, ZERO_FILL);
}
template <int CTRL, int ROW_MASK, bool ZERO_FILL> __device__ __forceinline__ uint64_t dpp_max_u64(uint64_t x) {
  const uint64_t y = ((uint64_t)dpp_move<CTRL, ROW_MASK, ZERO_FILL>((uint32_t)(x >> 32)) << 32) |
                     dpp_move<CTRL, ROW_MASK, ZERO_FILL>((uint32_t)x);
  return y > x ? y : x;
}
__device__ __forceinline__ uint64_t wave_max_u64(uint64_t x) {
  x = dpp_max_u64<0x111, 0xf, true>(x);
  x = dpp_max_u64<0x112, 0xf, true>(x);
  x = dpp_max_u64<0x114, 0xf, true>(x);
  x = dpp_max_u64<0x118, 0xf, true>(x);
  x = dpp_max_u64<0x142, 0xa, false>(x);
  x = dpp_max_u64<0x143, 0xc, false>(x);
  return ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(x >> 32), 63) << 32) |
         (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)x, 63);
}

// r / g for a row index r >= 0 and a GQA group of g heads: a shift where g is a power of two (g_shift =
// log2 g), the division otherwise (g_shift < 0).  The general division costs some forty instructions and sits in
// the address computation of every gathered row.
__device__ __forceinline__ int div_group(int r, int g, int g_shift) { return g_shift >= 0 ? (r >> g_shift) : r / g; }
static inline int group_shift(int g) {
  if (g <= 0 || (g & (g - 1)) != 0) return -1;
  int s = 0;
  while ((1 << s) < g) ++s;
  return s;
}

// largest i in [0, n) with a[i] <= x, for ascending a[0..n) with a[0] <= x
__device__ __forceinline__ int upper_seg(const int32_t* __restrict__ a, int n, int x) {
  int lo = 0, hi = n;  // invariant a[lo] <= x, a[hi] > x (virtual)
  while (hi - lo > 1) {
    int mid = (lo + hi) >> 1;
    if (a[mid] <= x) lo = mid; else hi = mid;
  }
  return lo;
}

// ---- host-side error plumbing --------------------------------------------
void set_error(const char* fmt, ...);

#define FSA_CHECK_ARG(cond, ...)            \
  do {                                      \
    if (!(cond)) {                          \
      fsa::set_error(__VA_ARGS__);          \
      return FSA_ERR_INVALID;               \
    }                                       \
  } while (0)

#define FSA_CHECK_LAUNCH(what)                                               \
  do {                                                                       \
    hipError_t e__ = hipGetLastError();                                      \
    if (e__ != hipSuccess) {                                                 \
      fsa::set_error("%s: %s", what, hipGetErrorString(e__));                \
      return (int)e__;                                                       \
    }                                                                        \
  } while (0)

// Dynamic LDS beyond 48 KB has to be allowed for every kernel, on every device that runs it: the attribute belongs to the
// pair.  `done` is a static beside the launch of one kernel with one size and remembers the devices by bits; a failure is
// reported every time it happens.  `dev`: the current device where the caller has asked for it already, -1 otherwise.
struct LdsAllowed {
  std::atomic<uint64_t> devices{0};
};
int allow_lds(LdsAllowed& done, const void* kernel, int bytes, int dev = -1);
int set_lds_limit(const void* kernel, int bytes);   // for sizes that change from call to call

// Optional per-kernel timing: while fsa_profile_enable(1) is in effect every
// launch wrapped in a ProfScope is bracketed by HIP events on its stream.
struct ProfScope {
  ProfScope(const char* name, hipStream_t stream);
  ~ProfScope();
  int idx_;
  hipStream_t stream_;
};

// Rows per work-group of a kernel that deals `rows_total` gathered rows to work-groups: `cap` (few partial results,
// long pipelines) where the problem is large enough, less where that would leave the chip idle: at least two
// work-groups for each of the `per_cu` slots of the 256 CUs, down to 128 rows each.  Measured (us, cap alone -> this
// rule): forward + backward of 4096 tokens x 8 heads of 256, 128-key blocks 1076 -> 409; the same rows with one or
// four work-groups per slot 465 - 660.
static inline int balanced_tile_rows(int64_t rows_total, int per_cu, int cap) {
  constexpr int STEP = 128;
  const int64_t r = (rows_total / (2 * 256 * per_cu) + STEP - 1) / STEP * STEP;
  return (int)(r < STEP ? STEP : r > cap ? cap : r);
}

// Forward: upper bound of the rows one work-group takes from a block (a block with more rows is dealt in equal shares to
// several work-groups): measured optimum about 3072 / 4096 / 6144-8192 rows for GQA groups of 1 / 2 / 4.
// Where LDS holds a single work-group per CU (head_dim 256, or 128-key blocks at head_dim 128) 1024 rows balance
// best.
static inline int sel_tile_rows(int64_t n_tokens, int topk, int hkv, int g, int d, int bk) {
  const int kv_bytes = (bk * (d + 8) + bk * (d + 16)) * 2, stage_bytes = 32 * (d + 8) * 2;
  const bool two_wgs = kv_bytes + 4 * stage_bytes <= 80 * 1024;   // SelLds<D, BK>::TWO_WGS
  const int r = 2048 + 1024 * g;
  const int cap = !two_wgs ? 1024 : r < 8192 ? r : 8192;
  return balanced_tile_rows(n_tokens * topk * hkv * g, two_wgs ? 2 : 1, cap);
}

// (tile, kv head) of a work-group of the block-major kernels.  Work-groups go to the eight XCDs in turn, so the tiles of up
// to eight heads are interleaved: an XCD then works on one head, or shares it with few others, and the query rows of that
// head, which the tiles gather over and over, are not fetched into eight L2 caches.  (Forward and backward, 8192 tokens x
// 32 heads of 128 1484 -> 1358 us, 16384 tokens x 16 heads, GQA 4, 1500 -> 1258.)  Rows of one head far beyond an L2 of
// 4 MB are fetched again for every tile either way, and the heads go one after the other (65536 tokens: GQA 1, 17 MB,
// 1448 -> 1416 us interleaved, GQA 4, 67 MB, 5183 -> 5223).
struct HeadOrder {
  int hkv, together;   // kv heads, heads whose tiles are interleaved
};
__device__ __forceinline__ void head_tile(HeadOrder o, int& h, int& tile) {
  const int h0 = blockIdx.y * o.together, heads = min(o.together, o.hkv - h0);
  h = h0 + blockIdx.x % heads;
  tile = blockIdx.x / heads;
}
static inline HeadOrder head_order(int hkv, int64_t row_bytes_per_head) {
  return {hkv, row_bytes_per_head > (32 << 20) ? 1 : hkv < 8 ? hkv : 8};
}
static inline dim3 head_tile_grid(int64_t tiles, HeadOrder o) {
  return dim3((unsigned)(tiles * o.together), (unsigned)((o.hkv + o.together - 1) / o.together));
}

static inline size_t align_up(size_t x, size_t a) { return (x + a - 1) / a * a; }

// Linear compression of up to two tensors of one shape in the same launches (keys and values: each alone has too few
// compressed rows to fill the chip).  Forward: x, w, y and, optionally, pe.  Backward: x, w, dy, dx, dw, and
// pe, dpe, dbias scratch where pe is not null.
struct LcTensors {
  const void *x, *w, *pe, *dy;
  int64_t x_sn, x_sh;
  void *y, *dx, *dw, *dpe;
  float* dbias;
};
int linear_compress_fwd(const LcTensors* t, int n, int dtype, const int32_t* cu_x, const int32_t* cu_y, int batch,
                        int64_t max_y, int h, int d, int ks, int stride, hipStream_t stream);
int linear_compress_bwd(const LcTensors* t, int n, int dtype, const int32_t* cu_x, const int32_t* cu_y, int batch,
                        int64_t max_x, int h, int d, int ks, int stride, hipStream_t stream);

// What the end of the selected forward does beside (or instead of, where `o` is null) storing o and lse: the gated sum of
// the three branches, gate[n] = three weights in the tensors' type, a / c [N, Hq, D] the first and the third branch.
struct MergeEpilogue {
  const void *a = nullptr, *c = nullptr, *gate = nullptr;
  void* out = nullptr;
};
int selattn_fwd(const void* q, const void* k, const void* v, int32_t dtype, int64_t q_stride_n, int64_t q_stride_h,
                int64_t k_stride_n, int64_t k_stride_h, int64_t v_stride_n, int64_t v_stride_h, const int32_t* cu_seqlens,
                int32_t batch, int64_t total_tokens, int32_t num_q_heads, int32_t num_kv_heads, int32_t head_dim, int32_t topk,
                int32_t block_size, int64_t max_blocks, float softmax_scale, const int32_t* cu_blocks, const int32_t* counts,
                const int32_t* starts, const int32_t* sel_tokens, const int32_t* slot_of, const int32_t* tiles, void* o,
                int64_t o_stride_n, int64_t o_stride_h, float* lse, void* workspace, size_t workspace_bytes,
                const MergeEpilogue& merge, hipStream_t stream);

constexpr int DIR_MAX_BLOCKS = 1024;   // of a sequence that the direct forward takes: size of its tables in LDS
bool selattn_direct_preferred(int64_t n, int64_t max_len, int hq, int d, int topk, int bk, bool index_needed);
int selattn_direct_fwd(const void* q, const void* k, const void* v, int32_t dtype, int64_t q_stride_n, int64_t q_stride_h,
                       int64_t k_stride_n, int64_t k_stride_h, int64_t v_stride_n, int64_t v_stride_h, const int32_t* topk_idx,
                       int64_t idx_stride_h, int64_t idx_stride_n, const int32_t* cu_seqlens, int32_t batch,
                       int64_t total_tokens, int64_t max_len, int32_t num_q_heads, int32_t num_kv_heads, int32_t head_dim,
                       int32_t topk, int32_t block_size, float softmax_scale, void* o, int64_t o_stride_n, int64_t o_stride_h,
                       float* lse, const MergeEpilogue& merge, hipStream_t stream);

// What the end of the selected backward adds to dQ before it is stored: gradients of the same queries from other branches,
// and the inverse rotation of the sum (cos / sin pairs [position][D/2] in the tensor's type).  All null: nothing.
struct DqEpilogue {
  const void *add0 = nullptr, *add1 = nullptr;   // [N, Hq, D] contiguous
  const void* rope = nullptr;
  const int32_t* cu = nullptr;                   // positions restart per sequence
  int batch = 0;
};

// A work list to build along with the index: blocks in order, ceil(counts * g / rows) tiles each.  prefix is
// [Hkv, max_blocks + 1], block [Hkv, max_tiles] (the block of every tile); prefix == null: not wanted.
struct TileList {
  int g, rows;
  int32_t* prefix;
  int32_t* block;
  int64_t max_tiles;
  // (count * g is at most the rows of q in one kv head: far below 2^31)
  __device__ __forceinline__ int tiles(int count) const { return (int)(((uint32_t)count * (uint32_t)g + rows - 1) / (uint32_t)rows); }
};

// Work list of the forward / backward main kernel of selected attention; `mem` holds prefix and block one after the other.
TileList selattn_tiles(bool backward, int64_t n_tokens, int hq, int hkv, int d, int topk, int bk, int64_t max_blocks,
                       int32_t* mem);

// fsa_selattn_bwd_tiles with (lse, delta) pairs [N, Hq] given instead of o and lse, and an epilogue of dQ.
int selattn_bwd(const void* q, const void* k, const void* v, const void* o,
                               const void* d_o, const float* lse, int32_t dtype, int64_t q_stride_n,
                               int64_t q_stride_h, int64_t k_stride_n, int64_t k_stride_h,
                               int64_t v_stride_n, int64_t v_stride_h, int64_t o_stride_n,
                               int64_t o_stride_h, int64_t do_stride_n, int64_t do_stride_h,
                               const int32_t* cu_seqlens, int32_t batch, int64_t total_tokens,
                               int32_t num_q_heads, int32_t num_kv_heads, int32_t head_dim,
                               int32_t topk, int32_t block_size, int64_t max_blocks,
                               float softmax_scale, const int32_t* cu_blocks, const int32_t* counts,
                               const int32_t* starts, const int32_t* sel_tokens,
                               const int32_t* slot_of, const int32_t* tiles, void* dq, void* dk, void* dv, void* workspace,
                               size_t workspace_bytes, const float2* stats, const DqEpilogue& epi, void* stream_);

// The compressed and the window attention of a layer, on contiguous tensors and the same queries.
struct LayerAttn {
  int dtype, hq, hkv, head_dim, batch, kernel_size, kernel_stride, window;
  int64_t n, total_ck, max_len;
  float scale;
  const int32_t *cu, *cu_ck;
  const void *q, *k, *v, *ck, *cv;
  void *o_cmp, *o_win;                    // forward
  float *lse_cmp, *lse_win;
  const void* d_out;                      // backward: both branches on the output gradient of the layer, each with its own
  const float2 *stat_cmp, *stat_win;      // (lse, delta) pairs [N, Hq]
  void *dq_cmp, *dq_win, *dck, *dcv, *dk_win, *dv_win;
};
int layer_attn_fwd(const LayerAttn& l, hipStream_t stream);
size_t layer_attn_bwd_workspace_bytes(int64_t n, int64_t total_ck, int64_t max_len, int window, int batch, int hq, int hkv, int d);
int layer_attn_bwd(const LayerAttn& l, void* workspace, hipStream_t stream);

// fsa_build_tiles with an optional tile -> block table [num_kv_heads, max_tiles] (max_tiles >= fsa_max_tiles(...))
int build_tiles(const int32_t* counts, int num_kv_heads, int64_t max_blocks, int group_size, int rows_per_tile,
                int32_t* tile_prefix, int32_t* tile_block, int64_t max_tiles, hipStream_t stream);

}  // namespace fsa
