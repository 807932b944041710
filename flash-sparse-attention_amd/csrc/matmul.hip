// Matrix products of the small layer: several products, or one whose contraction runs over several pairs of operands, in
// one launch.
//
// The projections of a layer and their gradients are twelve library products.  From a few thousand tokens on the library
// is the right tool; below, each call costs the host 20-25 us and most of them leave the chip half idle.  Here q, k and v
// are one launch, so are the four weight gradients, and the gradient of x is one product over the concatenated
// contraction, summed in fp32 and rounded once.  bf16, all five products of a forward and backward, device alone: hidden
// 1024, 8 + 2 heads of 128, 250 tokens 37 us, 2000 tokens 72; hidden 4096, 32 + 8 heads: 250 tokens 165, 1000 tokens 341.
//
// A work-group of four waves, or two such groups that halve the contraction, owns a BM x BN tile of one result.  Operand
// tiles of 64 contraction steps go from memory to LDS past the registers, STAGES - 1 of them ahead of the one being
// multiplied, and a step costs one barrier; an operand whose rows are contiguous along the contraction is read from LDS in
// 16-byte fragments, one whose rows run across it by transposing reads, both without bank conflicts.  Bound by the chain of
// a step (barrier, LDS read, product; some 600 clocks for a 64 x 64 tile alone on a CU) at small sizes and by the traffic
// into LDS at larger ones, 0.7-0.9 PFLOP/s at most.  (Through registers, with address arithmetic for every piece and the
// writes to LDS between two barriers: 2000 tokens, hidden 1024, 97 us for the five products, and 450 for 1000 x 4096.)
#include "fsa_common.h"

#include <algorithm>

namespace fsa {

constexpr int MM_MAX_OUT = 4;
constexpr int MM_BK = 64;
constexpr int MM_GROUP = 256;   // threads that share an operand tile
constexpr uint32_t MM_BUFFER = 0xFFFFFF00u;   // bytes of a buffer: all that an offset can name

struct MmGroup {
  fsa_matmul_out out[MM_MAX_OUT];
  int tile0[MM_MAX_OUT + 1];  // first tile of each result
  int n_out;
};

// Operand tile of ROWS rows (output dimension) x MM_BK steps.  KCONTIG: memory and LDS [row][step]; otherwise [step][row].
// The tile goes to LDS past the registers, 1 KB a wave instruction: chunk c (16 bytes) of line r in the place of chunk
// c ^ chunk_swizzle(r), which is what the loading lane picks its source by.
template <typename T, int ROWS, bool KCONTIG> struct MmOperand {
  typedef typename Elem<T>::vec8 vec8;
  static constexpr int LINE = KCONTIG ? MM_BK : ROWS;              // elements of a line
  static constexpr int CPL = LINE / 8;                             // chunks of a line
  static constexpr int BYTES = ROWS * MM_BK * 2;
  static constexpr int N = BYTES / 1024 / (MM_GROUP / WAVE);       // pieces of 1 KB per wave
  static __device__ __forceinline__ int swizzle(int r) { return chunk_swizzle<LINE>(r); }

  const T* p;          // first row of the tile, the step that is loaded next
  int64_t advance;     // bytes from one tile of steps to the next
  uint32_t off[N];     // of this lane's chunks
  // r_lo: first row of the tile, of `rows` in all; k_lo: first step.  Rows past the end repeat the last ones (their results
  // are not stored).
  __device__ __forceinline__ void use(const T* base, int ld, int wv, int r_lo, int rows, int k_lo) {
    const int lane = threadIdx.x & (WAVE - 1);
    p = base + (KCONTIG ? (int64_t)r_lo * ld + k_lo : (int64_t)k_lo * ld + r_lo);
    advance = (KCONTIG ? MM_BK : (int64_t)MM_BK * ld) * 2;
#pragma unroll
    for (int j = 0; j < N; ++j) {
      const int c = (wv * N + j) * WAVE + lane, a = c / CPL, b = ((c % CPL) ^ swizzle(a)) * 8;
      off[j] = 2u * (KCONTIG ? (uint32_t)min(a, rows - 1 - r_lo) * (uint32_t)ld + b : (uint32_t)a * (uint32_t)ld + min(b, rows - 8 - r_lo));
    }
  }
  // `valid`: steps of the tile that exist; the others become zero (an offset behind the end of the buffer)
  __device__ __forceinline__ void load(uint32_t lds, int wv, int valid) const {
    const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)p, 0, MM_BUFFER, 0x00020000);
    const int lane = threadIdx.x & (WAVE - 1);
#pragma unroll
    for (int j = 0; j < N; ++j) {
      uint32_t o = off[j];
      if (valid < MM_BK) {   // uniform
        const int c = (wv * N + j) * WAVE + lane, a = c / CPL;
        if ((KCONTIG ? ((c % CPL) ^ swizzle(a)) * 8 : a) >= valid) o = MM_BUFFER;
      }
      asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %1, 0 offen lds"
                   :: "v"(o), "s"(rsrc), "s"(lds + (wv * N + j) * 1024) : "memory");
    }
  }
  // LDS address of the lane in a fragment of rows r0 .. r0 + 31, steps 0 .. 15
  static __device__ __forceinline__ uint32_t lane_addr(uint32_t lds, int r0) {
    const int lane = threadIdx.x & (WAVE - 1), hh = lane >> 5;
    if constexpr (KCONTIG) {
      const int r = r0 + (lane & 31);
      return lds + r * (LINE * 2) + ((hh ^ swizzle(r)) << 4);
    } else {
      const int r = 8 * hh + ((lane & 15) >> 2), c = r0 / 8 + 2 * ((lane >> 4) & 1) + ((lane & 3) >> 1);
      return lds + r * (LINE * 2) + ((c ^ swizzle(r)) << 4) + (lane & 1) * 8;
    }
  }
  // fragment of rows r0 + 32 a .., steps 16 kk .. 16 kk + 15 from the address of (r0, 0)
  static __device__ __forceinline__ vec8 frag(uint32_t addr, int a, int kk) {
    if constexpr (KCONTIG) {
      return load16<vec8>(lds_ptr<T>((addr ^ (32u * kk)) + a * 32 * LINE * 2));
    } else {
      const uint32_t at = (addr ^ (64u * a)) + 16 * kk * LINE * 2;
      return __builtin_shufflevector(lds_read_tr4<T>(lds_ptr<T>(at)), lds_read_tr4<T>(lds_ptr<T>((at ^ 16u) + 4 * LINE * 2)),
                                     0, 1, 2, 3, 4, 5, 6, 7);
    }
  }
};

// AK / BK_: the operand's rows are contiguous along the contraction
template <typename T, int BM, int BN, int KS, int STAGES, bool AK, bool BK_>
__global__ void __launch_bounds__(MM_GROUP * KS)
matmul_kernel(MmGroup g, int tiles_per_xcd) {
  typedef typename Elem<T>::vec8 vec8;
  typedef typename Elem<T>::vec4 vec4;
  typedef MmOperand<T, BM, AK> OA;
  typedef MmOperand<T, BN, BK_> OB;
  constexpr int MT = BM / 64, NT = BN / 64;   // 32 x 32 tiles per wave; the waves are 2 x 2
  constexpr int STAGE = OA::BYTES + OB::BYTES, GROUP_BYTES = STAGES * STAGE;
  static_assert(KS == 1 || GROUP_BYTES >= BM * BN * 4, "partial sums of a group");
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem_mm[];
  // work-groups go round the XCDs: consecutive tiles (one row of tiles after the other) to the same L2
  const int tile = (blockIdx.x % 8) * tiles_per_xcd + blockIdx.x / 8;
  if (tile >= g.tile0[g.n_out]) return;
  int o = 0;
  while (o + 1 < g.n_out && tile >= g.tile0[o + 1]) ++o;
  const fsa_matmul_out& out = g.out[o];
  const int nt_n = (out.n + BN - 1) / BN, t = tile - g.tile0[o];
  const int m_lo = t / nt_n * BM, n_lo = t % nt_n * BN;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / WAVE)), grp = wave / 4, wv = wave % 4;
  const int lane = threadIdx.x & 63, col = lane & 31, hh = lane >> 5;
  const int wm = (wv >> 1) * (BM / 2), wn = (wv & 1) * (BN / 2);

  f32x16 acc[MT][NT];
#pragma unroll
  for (int a = 0; a < MT; ++a)
#pragma unroll
    for (int b = 0; b < NT; ++b)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[a][b][i] = 0.f;

  // the contraction as one sequence of steps over all pairs of operands, an equal share of it for each group of waves
  int steps = 0;
  for (int i = 0; i < out.parts; ++i) steps += (out.part[i].k + MM_BK - 1) / MM_BK;
  const int first = steps * grp / KS;
  const int rounds = (steps + KS - 1) / KS;   // of the longest share: every wave meets every barrier
  int left = steps * (grp + 1) / KS - first;
  int part = 0, k_next = min(first, steps - 1) * MM_BK;
  while (part + 1 < out.parts && k_next >= (out.part[part].k + MM_BK - 1) / MM_BK * MM_BK) {
    k_next -= (out.part[part].k + MM_BK - 1) / MM_BK * MM_BK;
    ++part;
  }
  OA oa;
  OB ob;
  int k_part;
  auto use_part = [&]() {
    const fsa_matmul_part& p = out.part[part];
    oa.use((const T*)p.a, (int)p.lda, wv, m_lo, out.m, k_next);
    ob.use((const T*)p.b, (int)p.ldb, wv, n_lo, out.n, k_next);
    k_part = p.k;
  };
  use_part();
  const uint32_t lds = lds_addr(smem_mm) + grp * GROUP_BYTES;
  // Always loads, so that the number of loads in flight is known at every point; behind the end of a share they are zeros.
  auto load = [&](int stage) {
    const int valid = left > 0 ? k_part - k_next : 0;
    oa.load(lds + stage * STAGE, wv, valid);
    ob.load(lds + stage * STAGE + OA::BYTES, wv, valid);
    if (--left > 0) {
      k_next += MM_BK;
      if (k_next < k_part) {
        oa.p = (const T*)((const char*)oa.p + oa.advance);
        ob.p = (const T*)((const char*)ob.p + ob.advance);
      } else {
        k_next = 0;
        ++part;
        use_part();
      }
    }
  };
  const uint32_t a_addr = OA::lane_addr(lds, wm), b_addr = OB::lane_addr(lds + OA::BYTES, wn);
  // fragments of AHEAD steps are requested before the first of their products
  constexpr int KK = MM_BK / 16, AHEAD = MT * NT >= 4 ? 2 : KK;
  auto multiply = [&](int stage, int next) {
    const uint32_t at = stage * STAGE;
    vec8 fa[AHEAD][MT], fb[AHEAD][NT];
    auto request = [&](int kk) {
#pragma unroll
      for (int a = 0; a < MT; ++a) fa[kk % AHEAD][a] = OA::frag(a_addr + at, a, kk);
#pragma unroll
      for (int b = 0; b < NT; ++b) fb[kk % AHEAD][b] = OB::frag(b_addr + at, b, kk);
    };
#pragma unroll
    for (int kk = 0; kk < AHEAD; ++kk) request(kk);
    load(next);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) {
#pragma unroll
      for (int a = 0; a < MT; ++a)
#pragma unroll
        for (int b = 0; b < NT; ++b)
          acc[a][b] = Elem<T>::mfma32(fb[kk % AHEAD][b], fa[kk % AHEAD][a], acc[a][b]);  // C^T: a lane holds one row of C
      if (kk + AHEAD < KK) {
        request(kk + AHEAD);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };
#pragma unroll
  for (int s = 0; s < STAGES - 1; ++s) load(s);
  int stage = 0;
  for (int r = 0; r < rounds; ++r) {
    vm_wait<(STAGES - 2) * (OA::N + OB::N)>();
    __syncthreads();   // this stage has arrived, and every wave has multiplied the one that is loaded next
    multiply(stage, stage == 0 ? STAGES - 1 : stage - 1);
    if (++stage == STAGES) stage = 0;
  }
  vm_wait<0>();
  if constexpr (KS > 1) {   // the groups' sums, each in the order of the registers
    __syncthreads();
    float* mine = reinterpret_cast<float*>(smem_mm + grp * GROUP_BYTES) + wv * (MT * NT * 16 * 64) + lane;
    if (grp > 0) {
#pragma unroll
      for (int a = 0; a < MT; ++a)
#pragma unroll
        for (int b = 0; b < NT; ++b)
#pragma unroll
          for (int i = 0; i < 16; ++i) mine[((a * NT + b) * 16 + i) * 64] = acc[a][b][i];
    }
    __syncthreads();
    if (grp > 0) return;
#pragma unroll
    for (int o_ = 1; o_ < KS; ++o_) {
      const float* other = mine + o_ * (GROUP_BYTES / 4);
#pragma unroll
      for (int a = 0; a < MT; ++a)
#pragma unroll
        for (int b = 0; b < NT; ++b)
#pragma unroll
          for (int i = 0; i < 16; ++i) acc[a][b][i] += other[((a * NT + b) * 16 + i) * 64];
    }
  }
#pragma unroll
  for (int a = 0; a < MT; ++a) {
    const int m = m_lo + wm + 32 * a + col;
    if (m >= out.m) continue;
#pragma unroll
    for (int b = 0; b < NT; ++b)
#pragma unroll
      for (int qd = 0; qd < 4; ++qd) {
        const int n = n_lo + wn + 32 * b + 8 * qd + 4 * hh;
        if (n >= out.n) continue;
        const int64_t at = (int64_t)m * out.ldc + n;
        f32x4 v = {acc[a][b][4 * qd], acc[a][b][4 * qd + 1], acc[a][b][4 * qd + 2], acc[a][b][4 * qd + 3]};
        if (out.add) {
          const vec4 e = load8<vec4>((const T*)out.add + at);
#pragma unroll
          for (int i = 0; i < 4; ++i) v[i] += (float)e[i];
        }
        vec4 r;
#pragma unroll
        for (int i = 0; i < 4; ++i) r[i] = (T)v[i];
        store8((T*)out.c + at, r);
      }
  }
}

template <typename T, int BM, int BN, int KS, int STAGES, bool AK, bool BK_>
static int launch_matmul(MmGroup& g, hipStream_t stream) {
  constexpr int LDS = KS * STAGES * (BM + BN) * MM_BK * 2;
  static LdsAllowed allowed;
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess) dev = -1;
  if (int rc_ = allow_lds(allowed, (const void*)matmul_kernel<T, BM, BN, KS, STAGES, AK, BK_>, LDS, dev)) return rc_;
  int tiles = 0;
  for (int i = 0; i < g.n_out; ++i) {
    g.tile0[i] = tiles;
    tiles += ((g.out[i].m + BM - 1) / BM) * ((g.out[i].n + BN - 1) / BN);
  }
  g.tile0[g.n_out] = tiles;
  const int per = (tiles + 7) / 8;
  ProfScope ps_("matmul", stream);
  matmul_kernel<T, BM, BN, KS, STAGES, AK, BK_><<<8 * per, MM_GROUP * KS, LDS, stream>>>(g, per);
  return 0;
}

// Tiles of 64 x 64 keep the most work-groups in flight, 128 x 128 load the least per product; two groups of waves halve the
// contraction where there is no more than one tile for a CU.  us, hidden 1024 (output projection, 16 steps | gradients of the
// weights): 1000 tokens 64 x 64 split 7.1, whole 8.0; 2000 tokens 64 x 64 9.9 | 25.0, 128 x 64 split 10.1 | 29.9, 128 x 128
// split 12.6 | 22.8; 4000 tokens 18.4 | 43.5, 19.2 | 51.2, 15.5 | 38.4, 128 x 128 whole 16.6 | 46.7; 8000 tokens 32.2, 36.0,
// 29.2, 24.6.  Hidden 4096, 500 tokens (64 steps): 40.6, 32.7, 36.9.  A result that keeps the order of its sum is not split:
// q, k and v of 2000 tokens, hidden 1024, 64 x 64 14.0, 128 x 128 15.5; 500 tokens of hidden 4096 54.5 and 47.4.
template <typename T, bool AK, bool BK_> static int dispatch_matmul(MmGroup& g, bool in_order, hipStream_t stream) {
  int64_t big = 0, small = 0;
  int steps = 0;
  for (int i = 0; i < g.n_out; ++i) {
    big += ((g.out[i].m + 127) / 128) * (int64_t)((g.out[i].n + 127) / 128);
    small += ((g.out[i].m + 63) / 64) * (int64_t)((g.out[i].n + 63) / 64);
    int k = 0;
    for (int j = 0; j < g.out[i].parts; ++j) k += (g.out[i].part[j].k + MM_BK - 1) / MM_BK;
    steps = std::max(steps, k);
  }
  if (in_order)
    return small <= 768 && small * steps <= 768 * 32 ? launch_matmul<T, 64, 64, 1, 3, AK, BK_>(g, stream)
                                                     : launch_matmul<T, 128, 128, 1, 2, AK, BK_>(g, stream);
  if (small <= 256 && steps >= 8) return launch_matmul<T, 64, 64, 2, 3, AK, BK_>(g, stream);
  if (big > 256) return launch_matmul<T, 128, 128, 1, 2, AK, BK_>(g, stream);
  if (steps < 16) return launch_matmul<T, 64, 64, 1, 3, AK, BK_>(g, stream);
  if (big > 128) return launch_matmul<T, 128, 128, 2, 2, AK, BK_>(g, stream);
  return launch_matmul<T, 128, 64, 2, 3, AK, BK_>(g, stream);
}

}  // namespace fsa

using namespace fsa;

extern "C" int fsa_matmul(const fsa_matmul_out* outs, int32_t n_out, int32_t form, int32_t dtype, void* stream_) {
  FSA_CHECK_ARG(outs && n_out >= 1 && n_out <= MM_MAX_OUT, "fsa_matmul: 1 to %d results", MM_MAX_OUT);
  FSA_CHECK_ARG((form & ~FSA_MM_IN_ORDER) >= FSA_MM_NT && (form & ~FSA_MM_IN_ORDER) <= FSA_MM_TN, "fsa_matmul: unknown form %d", form);
  FSA_CHECK_ARG(dtype == FSA_BF16 || dtype == FSA_FP16, "fsa_matmul: dtype must be bf16 or fp16");
  const bool in_order = form & FSA_MM_IN_ORDER;
  form &= ~FSA_MM_IN_ORDER;
  MmGroup g = {};
  g.n_out = n_out;
  const bool ak = form != FSA_MM_TN, bk = form == FSA_MM_NT;
  for (int i = 0; i < n_out; ++i) {
    const fsa_matmul_out& o = g.out[i] = outs[i];
    FSA_CHECK_ARG(o.c && o.parts >= 1 && o.parts <= 3 && o.m >= 1 && o.n >= 1, "fsa_matmul: bad result %d", i);
    FSA_CHECK_ARG((uintptr_t)o.c % 8 == 0 && (uintptr_t)o.add % 8 == 0 && o.ldc >= o.n && o.ldc % 4 == 0 && o.n % 8 == 0 &&
                      (ak || o.m % 8 == 0), "fsa_matmul: result %d is not aligned", i);
    for (int j = 0; j < o.parts; ++j) {
      const fsa_matmul_part& p = o.part[j];
      FSA_CHECK_ARG(p.a && p.b && p.k >= 1 && (uintptr_t)p.a % 16 == 0 && (uintptr_t)p.b % 16 == 0 && p.lda % 8 == 0 &&
                        p.ldb % 8 == 0 && p.lda >= (ak ? p.k : o.m) && p.ldb >= (bk ? p.k : o.n) && (!ak || p.k % 8 == 0) &&
                        p.lda * (ak ? o.m : p.k) < (1ll << 31) && p.ldb * (bk ? o.n : p.k) < (1ll << 31),
                    "fsa_matmul: bad operands of result %d", i);
    }
  }
  hipStream_t stream = (hipStream_t)stream_;
#define FSA_CALL(T)                                                     \
  (form == FSA_MM_NT   ? dispatch_matmul<T, true, true>(g, in_order, stream)      \
   : form == FSA_MM_NN ? dispatch_matmul<T, true, false>(g, in_order, stream)     \
                       : dispatch_matmul<T, false, false>(g, in_order, stream))
  const int rc = dtype == FSA_BF16 ? FSA_CALL(__bf16) : FSA_CALL(_Float16);
#undef FSA_CALL
  if (rc) return rc;
  FSA_CHECK_LAUNCH("fsa_matmul");
  return 0;
}
