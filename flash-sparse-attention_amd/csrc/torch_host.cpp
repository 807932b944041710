// Host path between torch tensors and the C ABI of libfsa_gfx950.so, as a Python extension module (fsa_hip._native).
//
// At short sequences and in decoding the host, not the chip, sets the pace: the same calls made from Python (tensor
// attributes, ctypes argument conversion, one Python autograd node per operator) cost 56 us for a forward and 200 us
// for a forward and backward of the operator, several times what the kernels take.  Here a call is argument checks, a
// few allocations from torch's caching allocator and the launches, and the autograd node runs without the interpreter.
//
// Error mapping: preconditions of a wrapper are AssertionError, tensors that are not on a device RuntimeError, what the
// C ABI refuses ValueError, launch errors RuntimeError.
#include <torch/extension.h>

#include <ATen/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <dlfcn.h>
#include <hip/hip_runtime_api.h>

#include <array>
#include <cmath>
#include <optional>
#include <tuple>
#include <vector>

#include "../../include/fsa_hip.h"

namespace py = pybind11;
using at::Tensor;
using std::optional;

namespace {

// ---- the C ABI, resolved from the library file that fsa_hip._lib names ----
#define FSA_API(X)                                                                                                     \
  X(fsa_last_error) X(fsa_native_head_dim) X(fsa_pad_head_dim) X(fsa_index_workspace_bytes) X(fsa_build_index)         \
  X(fsa_build_index_tiles) X(fsa_selattn_tiles_bytes) X(fsa_split_topk_blocks) X(fsa_selattn_fwd_workspace_bytes)      \
  X(fsa_selattn_fwd_tiles) X(fsa_selattn_bwd_workspace_bytes) X(fsa_selattn_bwd_tiles) X(fsa_decode_workspace_bytes) \
  X(fsa_decode_cmpattn) X(fsa_decode_topk) X(fsa_decode_selattn) X(fsa_decode_layer_workspace_bytes)                   \
  X(fsa_decode_layer_project) X(fsa_decode_layer_attend) X(fsa_linear_compress_fwd)                                    \
  X(fsa_layer_saved_bytes) X(fsa_layer_workspace_bytes) X(fsa_layer_forward) X(fsa_layer_backward) \
  X(fsa_matmul) X(fsa_selattn_direct_preferred) X(fsa_selattn_direct_fwd)
struct Api {
#define FSA_FIELD(f) decltype(&::f) f = nullptr;
  FSA_API(FSA_FIELD)
#undef FSA_FIELD
} api;

void bind_library(const std::string& path) {
  void* lib = dlopen(path.c_str(), RTLD_NOW | RTLD_LOCAL);
  TORCH_CHECK(lib, "cannot load ", path, ": ", dlerror());
#define FSA_RESOLVE(f)                                           \
  api.f = reinterpret_cast<decltype(api.f)>(dlsym(lib, #f));     \
  TORCH_CHECK(api.f, path, " does not export " #f);
  FSA_API(FSA_RESOLVE)
#undef FSA_RESOLVE
}

struct NoKernel {};   // a size that the fused calls do not take, found out late
struct AssertionFailed : std::runtime_error {
  using std::runtime_error::runtime_error;
};
#define FSA_ASSERT(cond, msg) \
  do {                        \
    if (!(cond)) throw AssertionFailed(msg); \
  } while (0)

void check(int rc, const char* what) {
  if (rc == 0) return;
  const char* msg = api.fsa_last_error();
  TORCH_CHECK_VALUE(rc > 0, what, ": ", msg, " (code ", rc, ")");
  TORCH_CHECK(false, what, ": HIP error ", rc, ": ", msg);
}

void need_device(const Tensor& t) {
  TORCH_CHECK(t.is_cuda(), "fsa_hip: tensors must live on a ROCm device; there is no CPU path");
}
template <typename... Ts> void need_device(const Tensor& t, const Ts&... rest) {
  need_device(t);
  need_device(rest...);
}

// The kernels have no forward-mode derivative.  An autograd node says so by itself, but without a gradient to record there
// is no node, and a tangent would be lost without a word.
void refuse_tangent(const Tensor& t) {
  if (t.defined())
    TORCH_CHECK_NOT_IMPLEMENTED(!t._fw_grad(/*level=*/0).defined(), "fsa_hip: forward-mode differentiation is not implemented");
}
template <typename... Ts> void refuse_tangent(const Tensor& t, const Ts&... rest) {
  refuse_tangent(t);
  refuse_tangent(rest...);
}

bool is16(const Tensor& t) { return t.scalar_type() == at::kBFloat16 || t.scalar_type() == at::kHalf; }
int dtype_code(const Tensor& t) { return t.scalar_type() == at::kBFloat16 ? FSA_BF16 : FSA_FP16; }
void* stream_of(const Tensor& t) { return (void*)c10::hip::getCurrentHIPStream(t.device().index()).stream(); }
const int32_t* i32(const Tensor& t) { return static_cast<const int32_t*>(t.data_ptr()); }
float* f32(const Tensor& t) { return static_cast<float*>(t.data_ptr()); }

Tensor empty_like_opts(at::IntArrayRef size, const Tensor& like, at::ScalarType type) {
  return at::empty(size, like.options().dtype(type));
}
Tensor empty_i32(at::IntArrayRef size, const Tensor& like) { return empty_like_opts(size, like, at::kInt); }
Tensor empty_f32(at::IntArrayRef size, const Tensor& like) { return empty_like_opts(size, like, at::kFloat); }
Tensor scratch(size_t bytes, const Tensor& like) { return empty_like_opts({(int64_t)bytes}, like, at::kByte); }

// ---- head dims the kernels are not built for: zero-padded copies of the next built size ----
int64_t native_dim(int64_t d) {
  const int n = api.fsa_native_head_dim((int32_t)std::min<int64_t>(d, 1 << 20));
  TORCH_CHECK_VALUE(n > 0, "head_dim ", d, " is not supported (at most 256)");
  return n;
}
// [..., H, d] -> contiguous [..., H, d_to]: the leading columns copied, the rest zero
Tensor resize_d(const Tensor& t, int64_t d_to) {
  const int64_t d = t.size(-1);
  if (d == d_to) return t;
  const Tensor rows = t.dim() == 3 ? t : t.reshape({-1, t.size(-2), d});
  if (t.numel() == 0 || !is16(t) || !t.is_cuda() || rows.stride(2) != 1 || d % 4 || d_to % 4 || rows.stride(0) % 4 ||
      rows.stride(1) % 4 || (uintptr_t)t.data_ptr() % 8)
    // what the C helper does not take (empty tensors, fp32 gradients of parameters, odd head dims): torch copies
    return (d_to > d ? at::constant_pad_nd(t, {0, d_to - d}) : t.narrow(-1, 0, d_to)).contiguous();
  auto sizes = t.sizes().vec();
  sizes.back() = d_to;
  Tensor out = at::empty(sizes, t.options());
  check(api.fsa_pad_head_dim(rows.data_ptr(), rows.stride(0), rows.stride(1), (int32_t)d, out.data_ptr(),
                             rows.size(1) * d_to, d_to, (int32_t)d_to, rows.size(0), (int32_t)rows.size(1),
                             stream_of(t)),
        "fsa_pad_head_dim");
  return out;
}
Tensor unit_stride(const Tensor& t) { return t.stride(-1) == 1 ? t : t.contiguous(); }

double default_scale(const optional<double>& s, int64_t d) { return s ? *s : 1.0 / std::sqrt((double)d); }

// ---- selected attention ----
// Inverted block -> query index of one call: raw pointers into arrays that somebody else keeps alive.
struct IndexView {
  const int32_t *cu, *cu_blocks, *counts, *starts, *sel, *slot;
  const int32_t *tiles_fwd, *tiles_bwd;  // work lists, null: the library builds them
  int64_t batch, n, hkv, topk, block, max_blocks;
};

void check_topk(const Tensor& topk_idx, const Tensor& cu) {
  need_device(topk_idx, cu);
  FSA_ASSERT(topk_idx.scalar_type() == at::kInt && cu.scalar_type() == at::kInt, "topk_idx and cu_seqlens must be int32");
  FSA_ASSERT(topk_idx.dim() == 3 && topk_idx.stride(2) == 1, "topk_idx must be [num_kv_heads, N, T] with unit stride");
}

std::vector<Tensor> build_index(const Tensor& topk_idx, const Tensor& cu, int64_t block) {
  check_topk(topk_idx, cu);
  const int64_t hkv = topk_idx.size(0), n = topk_idx.size(1), topk = topk_idx.size(2), batch = cu.numel() - 1;
  const int64_t max_blocks = (n + block - 1) / block + batch;
  const c10::OptionalDeviceGuard guard(topk_idx.device());
  const std::vector<Tensor> mem = {empty_i32({batch + 1}, topk_idx), empty_i32({hkv, max_blocks}, topk_idx),
                                   empty_i32({hkv, max_blocks + 1}, topk_idx), empty_i32({hkv, n * topk}, topk_idx),
                                   empty_i32({hkv, n, topk}, topk_idx)};
  const size_t bytes = api.fsa_index_workspace_bytes(n, (int32_t)topk, (int32_t)hkv, max_blocks);
  Tensor ws = scratch(bytes, topk_idx);
  check(api.fsa_build_index(i32(topk_idx), topk_idx.stride(0), topk_idx.stride(1), i32(cu), (int32_t)batch, n,
                            (int32_t)hkv, (int32_t)topk, (int32_t)block, max_blocks, (int32_t*)i32(mem[0]),
                            (int32_t*)i32(mem[1]), (int32_t*)i32(mem[2]), (int32_t*)i32(mem[3]),
                            (int32_t*)i32(mem[4]), ws.data_ptr(), bytes, stream_of(topk_idx)),
        "fsa_build_index");
  return mem;
}

Tensor split_topk_blocks(const Tensor& topk_idx, const Tensor& cu, int64_t block, int64_t factor) {
  check_topk(topk_idx, cu);
  const c10::OptionalDeviceGuard guard(topk_idx.device());
  Tensor out = empty_i32({topk_idx.size(0), topk_idx.size(1), topk_idx.size(2) * factor}, topk_idx);
  check(api.fsa_split_topk_blocks(i32(topk_idx), topk_idx.stride(0), topk_idx.stride(1), i32(cu),
                                  (int32_t)cu.numel() - 1, topk_idx.size(1), (int32_t)topk_idx.size(0),
                                  (int32_t)topk_idx.size(2), (int32_t)block, (int32_t)factor, (int32_t*)i32(out),
                                  stream_of(topk_idx)),
        "fsa_split_topk_blocks");
  return out;
}

// Index and work lists of one operator call, in one allocation.
struct Index {
  Tensor cu, mem;
  int64_t n, hkv, topk, block, max_blocks, hq, d;
  bool forward, backward;   // whose work lists are there

  IndexView view() const {
    const int64_t batch = cu.numel() - 1;
    int64_t at = 0;
    const int32_t* base = i32(mem);
    auto part = [&](int64_t ints) {
      const int32_t* p = base + at;
      at += (ints + 63) / 64 * 64;
      return p;
    };
    IndexView v{};
    v.cu = i32(cu);
    v.cu_blocks = part(batch + 1);
    v.counts = part(hkv * max_blocks);
    v.starts = part(hkv * (max_blocks + 1));
    v.sel = part(hkv * n * topk);
    v.slot = part(hkv * n * topk);
    v.tiles_fwd = forward ? part(tile_ints(false)) : nullptr;
    v.tiles_bwd = backward ? part(tile_ints(true)) : nullptr;
    v.batch = batch;
    v.n = n;
    v.hkv = hkv;
    v.topk = topk;
    v.block = block;
    v.max_blocks = max_blocks;
    return v;
  }
  int64_t tile_ints(bool bwd) const {
    return (int64_t)api.fsa_selattn_tiles_bytes(bwd, n, (int32_t)hq, (int32_t)hkv, (int32_t)d, (int32_t)topk,
                                                (int32_t)block, max_blocks) / 4;
  }
  int64_t total_ints() const {
    auto r = [](int64_t x) { return (x + 63) / 64 * 64; };
    return r(cu.numel()) + r(hkv * max_blocks) + r(hkv * (max_blocks + 1)) + 2 * r(hkv * n * topk) +
           (forward ? r(tile_ints(false)) : 0) + (backward ? r(tile_ints(true)) : 0);
  }
};

// Blocks of 256 keys run as pairs of 128-key blocks (the same key set for every query).
Tensor kernel_blocks(const Tensor& topk_idx, const Tensor& cu, int64_t& block) {
  check_topk(topk_idx, cu);
  if (block != 256) return topk_idx;
  block = 128;
  return split_topk_blocks(topk_idx, cu, 256, 2);
}
Index kernel_index(const Tensor& topk_idx, const Tensor& cu, int64_t block, int64_t hq, int64_t d, bool forward, bool backward) {
  Index x;
  x.cu = cu;
  x.hkv = topk_idx.size(0);
  x.n = topk_idx.size(1);
  x.topk = topk_idx.size(2);
  x.block = block;
  x.max_blocks = (x.n + block - 1) / block + cu.numel() - 1;
  x.hq = hq;
  x.d = d;
  x.forward = forward;
  x.backward = backward;
  const c10::OptionalDeviceGuard guard(topk_idx.device());
  x.mem = empty_i32({x.total_ints()}, topk_idx);
  const IndexView v = x.view();
  const size_t bytes = api.fsa_index_workspace_bytes(x.n, (int32_t)x.topk, (int32_t)x.hkv, x.max_blocks);
  Tensor ws = scratch(bytes, topk_idx);
  check(api.fsa_build_index_tiles(i32(topk_idx), topk_idx.stride(0), topk_idx.stride(1), v.cu, (int32_t)v.batch, x.n,
                                  (int32_t)x.hkv, (int32_t)x.topk, (int32_t)block, x.max_blocks, (int32_t*)v.cu_blocks,
                                  (int32_t*)v.counts, (int32_t*)v.starts, (int32_t*)v.sel, (int32_t*)v.slot,
                                  (int32_t)hq, (int32_t)d, (int32_t*)v.tiles_fwd, (int32_t*)v.tiles_bwd, ws.data_ptr(),
                                  bytes, stream_of(topk_idx)),
        "fsa_build_index");
  return x;
}

void check_qkv(const Tensor& q, const Tensor& k, const Tensor& v) {
  need_device(q, k, v);
  FSA_ASSERT(is16(q), "q must be bf16 or fp16");
  FSA_ASSERT(q.scalar_type() == k.scalar_type() && k.scalar_type() == v.scalar_type(), "q, k, v must have one dtype");
  FSA_ASSERT(q.dim() == 3 && k.dim() == 3 && v.dim() == 3, "q, k, v must be [N, H, D]");
  FSA_ASSERT(q.stride(2) == 1 && k.stride(2) == 1 && v.stride(2) == 1, "q, k, v must have unit stride in head_dim");
  FSA_ASSERT(k.size(1) > 0 && q.size(1) % k.size(1) == 0, "num_q_heads must be a multiple of num_kv_heads");
  FSA_ASSERT(k.sizes() == v.sizes() && q.size(0) == k.size(0) && q.size(2) == k.size(2), "shapes of q, k, v do not match");
}

// head_dim one of the built sizes
std::pair<Tensor, Tensor> selattn_fwd_native(const Tensor& q, const Tensor& k, const Tensor& v, const IndexView& x,
                                             double scale) {
  const int64_t n = q.size(0), hq = q.size(1), d = q.size(2), hkv = k.size(1);
  FSA_ASSERT(hkv == x.hkv && n == x.n, "index does not belong to these tensors");
  const c10::OptionalDeviceGuard guard(q.device());
  Tensor o = at::empty({n, hq, d}, q.options()), lse = empty_f32({hq, n}, q);
  const size_t bytes = api.fsa_selattn_fwd_workspace_bytes(n, (int32_t)hq, (int32_t)hkv, (int32_t)d, (int32_t)x.topk,
                                                           x.max_blocks);
  Tensor ws = scratch(bytes, q);
  check(api.fsa_selattn_fwd_tiles(q.data_ptr(), k.data_ptr(), v.data_ptr(), dtype_code(q), q.stride(0), q.stride(1),
                            k.stride(0), k.stride(1), v.stride(0), v.stride(1), x.cu, (int32_t)x.batch, n, (int32_t)hq,
                            (int32_t)hkv, (int32_t)d, (int32_t)x.topk, (int32_t)x.block, x.max_blocks, (float)scale,
                            x.cu_blocks, x.counts, x.starts, x.sel, x.slot, x.tiles_fwd, o.data_ptr(), hq * d, d, f32(lse),
                            ws.data_ptr(), bytes, stream_of(q)),
        "fsa_selattn_fwd");
  return {o, lse};
}

// Short sequences: from the block lists (kernel_blocks), without an index.  The lengths are on the device and are not read
// back.  A packed batch is priced as one sequence of three quarters of its tokens, which is the mean length that a row finds
// where two sequences share the tokens 85 : 15.  (As one sequence of all of them, batches of short documents take the
// block-major kernels: 3000 tokens x 4 heads of 256 in 4, 6 blocks of 64, 71 us against 36.  A batch that is one long sequence but
// for a few tokens may be up to a quarter slower than with them.)
bool direct(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& topk_idx, int64_t batch, int64_t block, bool index_needed) {
  const int64_t n = q.size(0), d = q.size(2), len = batch > 1 ? n - n / 4 : n;
  auto rows_ok = [&](const Tensor& t) {   // they go to LDS by 16-byte buffer loads
    return t.stride(0) >= d && t.stride(0) * n < (int64_t)1 << 30 && (uintptr_t)t.data_ptr() % 16 == 0;
  };
  return n >= 1 && n <= 1024 * block &&   // the kernels' limit, whatever the price
         topk_idx.size(0) == k.size(1) && topk_idx.size(1) == n && rows_ok(k) && rows_ok(v) &&
         api.fsa_selattn_direct_preferred(n, len, (int32_t)q.size(1), (int32_t)d, (int32_t)topk_idx.size(2), (int32_t)block,
                                          index_needed) == 1;
}
std::pair<Tensor, Tensor> selattn_direct(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& topk_idx, const Tensor& cu,
                                         int64_t block, double scale) {
  const int64_t n = q.size(0), hq = q.size(1), d = q.size(2), hkv = k.size(1);
  const c10::OptionalDeviceGuard guard(q.device());
  Tensor o = at::empty({n, hq, d}, q.options()), lse = empty_f32({hq, n}, q);
  check(api.fsa_selattn_direct_fwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), dtype_code(q), q.stride(0), q.stride(1), k.stride(0),
                                   k.stride(1), v.stride(0), v.stride(1), i32(topk_idx), topk_idx.stride(0), topk_idx.stride(1),
                                   i32(cu), (int32_t)cu.numel() - 1, n, n, (int32_t)hq, (int32_t)hkv, (int32_t)d,
                                   (int32_t)topk_idx.size(2), (int32_t)block, (float)scale, o.data_ptr(), hq * d, d, f32(lse),
                                   stream_of(q)),
        "fsa_selattn_fwd");
  return {o, lse};
}

std::tuple<Tensor, Tensor, Tensor> selattn_bwd_native(const Tensor& q, const Tensor& k, const Tensor& v,
                                                      const Tensor& o_, const Tensor& do_, const Tensor& lse_,
                                                      const IndexView& x, double scale) {
  const int64_t n = q.size(0), hq = q.size(1), d = q.size(2), hkv = k.size(1);
  const c10::OptionalDeviceGuard guard(q.device());
  const Tensor o = unit_stride(o_), d_o = unit_stride(do_), lse = lse_.contiguous();
  Tensor dq = at::empty({n, hq, d}, q.options());
  Tensor dk = at::empty({n, hkv, d}, q.options()), dv = at::empty({n, hkv, d}, q.options());
  const size_t bytes = api.fsa_selattn_bwd_workspace_bytes(n, (int32_t)hq, (int32_t)hkv, (int32_t)d, (int32_t)x.topk,
                                                           (int32_t)x.block, x.max_blocks);
  Tensor ws = scratch(bytes, q);
  check(api.fsa_selattn_bwd_tiles(q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), d_o.data_ptr(), f32(lse),
                            dtype_code(q), q.stride(0), q.stride(1), k.stride(0), k.stride(1), v.stride(0), v.stride(1),
                            o.stride(0), o.stride(1), d_o.stride(0), d_o.stride(1), x.cu, (int32_t)x.batch, n,
                            (int32_t)hq, (int32_t)hkv, (int32_t)d, (int32_t)x.topk, (int32_t)x.block, x.max_blocks,
                            (float)scale, x.cu_blocks, x.counts, x.starts, x.sel, x.slot, x.tiles_bwd, dq.data_ptr(), dk.data_ptr(),
                            dv.data_ptr(), ws.data_ptr(), bytes, stream_of(q)),
        "fsa_selattn_bwd");
  return {dq, dk, dv};
}

// [cu_seqlens, cu_blocks, counts, starts, sel_tokens, slot_of] as fsa_hip.ops.SelIndex holds them
IndexView view_of(const std::vector<Tensor>& t, int64_t topk, int64_t block, int64_t max_blocks) {
  return {i32(t[0]), i32(t[1]), i32(t[2]), i32(t[3]), i32(t[4]), i32(t[5]), nullptr, nullptr, t[0].numel() - 1,
          t[5].size(1), t[5].size(0), topk, block, max_blocks};
}

// `lists`: the block lists of the index, where short sequences may run from them as the operator's do
std::pair<Tensor, Tensor> selattn_fwd(const Tensor& q, const Tensor& k, const Tensor& v, const std::vector<Tensor>& index,
                                      int64_t topk, int64_t block, int64_t max_blocks, optional<double> scale_,
                                      const optional<Tensor>& lists) {
  check_qkv(q, k, v);
  if (lists) check_topk(*lists, index[0]);
  const int64_t d = q.size(2), dn = native_dim(d);
  const double scale = default_scale(scale_, d);
  const Tensor qn = resize_d(q, dn), kn = resize_d(k, dn), vn = resize_d(v, dn);
  auto [o, lse] = lists && direct(qn, kn, vn, *lists, index[0].numel() - 1, block, true)
                      ? selattn_direct(qn, kn, vn, *lists, index[0], block, scale)
                      : selattn_fwd_native(qn, kn, vn, view_of(index, topk, block, max_blocks), scale);
  return {resize_d(o, d), lse};
}

// The same from the lists alone, for callers that keep no index: (o, lse) of the forward that training takes
std::pair<Tensor, Tensor> selattn_fwd_lists(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& topk_idx, int64_t block,
                                            const Tensor& cu, optional<double> scale_) {
  check_qkv(q, k, v);
  const int64_t d = q.size(2), dn = native_dim(d);
  const double scale = default_scale(scale_, d);
  const Tensor ids = kernel_blocks(topk_idx, cu, block), qn = resize_d(q, dn), kn = resize_d(k, dn), vn = resize_d(v, dn);
  auto [o, lse] = direct(qn, kn, vn, ids, cu.numel() - 1, block, true)
                      ? selattn_direct(qn, kn, vn, ids, cu, block, scale)
                      : selattn_fwd_native(qn, kn, vn, kernel_index(ids, cu, block, q.size(1), dn, true, false).view(), scale);
  return {resize_d(o, d), lse};
}

void check_bwd(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& o, const Tensor& d_o, const Tensor& lse) {
  check_qkv(q, k, v);
  need_device(o, d_o, lse);
  FSA_ASSERT(o.scalar_type() == q.scalar_type() && d_o.scalar_type() == q.scalar_type() && lse.scalar_type() == at::kFloat,
             "o and do must have q's dtype, lse float32");
  FSA_ASSERT(o.sizes() == q.sizes() && d_o.sizes() == q.sizes(), "o and do must have q's shape");
}

std::tuple<Tensor, Tensor, Tensor> selattn_bwd(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& o,
                                               const Tensor& d_o, const Tensor& lse, const std::vector<Tensor>& index,
                                               int64_t topk, int64_t block, int64_t max_blocks, optional<double> scale_) {
  check_bwd(q, k, v, o, d_o, lse);
  const int64_t d = q.size(2), dn = native_dim(d);
  auto [dq, dk, dv] =
      selattn_bwd_native(resize_d(q, dn), resize_d(k, dn), resize_d(v, dn), resize_d(o, dn), resize_d(d_o, dn), lse,
                         view_of(index, topk, block, max_blocks), default_scale(scale_, d));
  return {resize_d(dq, d), resize_d(dk, d), resize_d(dv, d)};
}

// The operator as one autograd node.  Padded copies (head dims that are not built) are what is saved, so the backward
// does not make them again.
struct SelectedAttention : torch::autograd::Function<SelectedAttention> {
  static Tensor forward(torch::autograd::AutogradContext* ctx, const Tensor& q, const Tensor& k, const Tensor& v,
                        const Tensor& topk_idx, int64_t block, const Tensor& cu, double scale) {
    const int64_t d = q.size(2), dn = native_dim(d);
    const Tensor ids = kernel_blocks(topk_idx, cu, block);
    const Tensor qn = resize_d(q, dn), kn = resize_d(k, dn), vn = resize_d(v, dn);
    const bool from_lists = direct(qn, kn, vn, ids, cu.numel() - 1, block, true);
    const Index x = kernel_index(ids, cu, block, q.size(1), dn, !from_lists, true);
    auto [on, lse] = from_lists ? selattn_direct(qn, kn, vn, ids, cu, block, scale) : selattn_fwd_native(qn, kn, vn, x.view(), scale);
    ctx->save_for_backward({qn, kn, vn, on, lse, x.cu, x.mem});
    ctx->saved_data["ints"] = std::vector<int64_t>{d, x.n, x.hkv, x.topk, x.block, x.max_blocks, x.hq, x.d, x.forward};
    ctx->saved_data["scale"] = scale;
    return resize_d(on, d);
  }
  static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx,
                                                 torch::autograd::variable_list grads) {
    const auto s = ctx->get_saved_variables();
    const auto ints = ctx->saved_data["ints"].toIntVector();
    const Tensor d_o = resize_d(grads[0], s[0].size(2));
    const Index x{s[5], s[6], ints[1], ints[2], ints[3], ints[4], ints[5], ints[6], ints[7], ints[8] != 0, true};
    auto [dq, dk, dv] =
        selattn_bwd_native(s[0], s[1], s[2], s[3], d_o, s[4], x.view(), ctx->saved_data["scale"].toDouble());
    return {resize_d(dq, ints[0]), resize_d(dk, ints[0]), resize_d(dv, ints[0]), Tensor(), Tensor(), Tensor(), Tensor()};
  }
};

Tensor selected_attention(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& topk_idx, int64_t block,
                          const Tensor& cu, optional<double> scale_) {
  refuse_tangent(q, k, v);
  FSA_ASSERT(block == 32 || block == 64 || block == 128 || block == 256, "block_size must be 32, 64, 128 or 256");
  check_qkv(q, k, v);
  check_topk(topk_idx, cu);
  const double scale = default_scale(scale_, q.size(2));
  if (at::GradMode::is_enabled() && (q.requires_grad() || k.requires_grad() || v.requires_grad()))
    return SelectedAttention::apply(q, k, v, topk_idx, block, cu, scale);
  const int64_t d = q.size(2), dn = native_dim(d);
  const Tensor ids = kernel_blocks(topk_idx, cu, block), qn = resize_d(q, dn), kn = resize_d(k, dn), vn = resize_d(v, dn);
  if (direct(qn, kn, vn, ids, cu.numel() - 1, block, false)) return resize_d(selattn_direct(qn, kn, vn, ids, cu, block, scale).first, d);
  const Index x = kernel_index(ids, cu, block, q.size(1), dn, true, false);
  return resize_d(selattn_fwd_native(qn, kn, vn, x.view(), scale).first, d);
}

// ---- one-step decode ----
std::tuple<Tensor, Tensor, optional<Tensor>> decode_cmpattn(const Tensor& q, const Tensor& ck, const Tensor& cv,
                                                            const Tensor& cu_ck, const Tensor& pos, int64_t kernel_size,
                                                            int64_t kernel_stride, int64_t max_ck,
                                                            optional<double> scale_, bool want_scores, bool as_written) {
  need_device(q, ck, cv, cu_ck, pos);
  FSA_ASSERT(is16(q) && q.scalar_type() == ck.scalar_type() && ck.scalar_type() == cv.scalar_type(),
             "q, ck, cv must be bf16 or fp16 of one dtype");
  FSA_ASSERT(q.dim() == 3 && q.stride(2) == 1 && ck.stride(2) == 1 && cv.stride(2) == 1, "unit stride in head_dim");
  const int64_t b = q.size(0), hq = q.size(1), d = q.size(2), hkv = ck.size(1);
  const double scale = default_scale(scale_, d);
  const int64_t dn = native_dim(d);
  if (dn != d) {
    auto [o, lse, raw] = decode_cmpattn(resize_d(q, dn), resize_d(ck, dn), resize_d(cv, dn), cu_ck, pos, kernel_size,
                                        kernel_stride, max_ck, scale, want_scores, as_written);
    return {resize_d(o, d), lse, raw};
  }
  const c10::OptionalDeviceGuard guard(q.device());
  Tensor o = at::empty({b, hq, d}, q.options()), lse = empty_f32({hq, b}, q);
  const int64_t ld = (std::max<int64_t>(max_ck, 1) + 3) / 4 * 4, max_keys = std::max<int64_t>(max_ck, 0);
  optional<Tensor> raw;
  if (want_scores) raw = empty_f32({hkv, b, ld}, q);
  const size_t bytes = std::max<size_t>(
      256, api.fsa_decode_workspace_bytes((int32_t)b, (int32_t)hq, (int32_t)hkv, (int32_t)d, max_keys));
  Tensor ws = scratch(bytes, q);
  check(api.fsa_decode_cmpattn(q.data_ptr(), ck.data_ptr(), cv.data_ptr(), dtype_code(q), q.stride(0), q.stride(1),
                               ck.stride(0), ck.stride(1), cv.stride(0), cv.stride(1), i32(cu_ck), i32(pos), (int32_t)b,
                               (int32_t)hq, (int32_t)hkv, (int32_t)d, (int32_t)kernel_size, (int32_t)kernel_stride,
                               (float)scale, as_written ? 1 : 0, max_keys, o.data_ptr(), f32(lse),
                               raw ? f32(*raw) : nullptr, ld, ws.data_ptr(), bytes, stream_of(q)),
        "fsa_decode_cmpattn");
  return {o, lse, raw};
}

std::pair<Tensor, optional<Tensor>> decode_topk(const Tensor& raw, const Tensor& lse, const Tensor& cu_ck,
                                                const Tensor& pos, const Tensor& seqlens, int64_t num_q_heads,
                                                int64_t kernel_size, int64_t kernel_stride, int64_t block_size,
                                                int64_t topk, int64_t max_blocks, int64_t init_blocks,
                                                int64_t local_blocks, double scale, bool as_written,
                                                bool return_block_score, bool scores_to_bf16) {
  need_device(raw, lse, cu_ck, pos, seqlens);
  const int64_t hkv = raw.size(0), b = raw.size(1);
  const c10::OptionalDeviceGuard guard(raw.device());
  Tensor idx = empty_i32({hkv, b, topk}, raw);
  optional<Tensor> score;
  if (return_block_score) score = empty_f32({hkv, b, max_blocks}, raw);
  check(api.fsa_decode_topk(f32(raw), raw.size(2), f32(lse), i32(cu_ck), i32(pos), i32(seqlens), (int32_t)b,
                            (int32_t)num_q_heads, (int32_t)hkv, (int32_t)kernel_size, (int32_t)kernel_stride,
                            (int32_t)block_size, (int32_t)topk, (int32_t)init_blocks, (int32_t)local_blocks,
                            as_written ? 1 : 0, scores_to_bf16 ? 1 : 0, (float)scale, max_blocks, (int32_t*)i32(idx),
                            score ? f32(*score) : nullptr, stream_of(raw)),
        "fsa_decode_topk");
  return {idx, score};
}

std::pair<Tensor, Tensor> decode_selattn(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& cu_k,
                                         const Tensor& topk_idx, int64_t block_size, optional<double> scale_,
                                         const optional<Tensor>& seqlens) {
  need_device(q, k, v, cu_k, topk_idx);
  FSA_ASSERT(!seqlens || (seqlens->is_cuda() && seqlens->scalar_type() == at::kInt && seqlens->numel() == q.size(0)),
             "seqlens must be int32 [B] on the device");
  FSA_ASSERT(is16(q) && q.scalar_type() == k.scalar_type() && k.scalar_type() == v.scalar_type(),
             "q and the caches must be bf16 or fp16 of one dtype");
  FSA_ASSERT(topk_idx.scalar_type() == at::kInt && topk_idx.is_contiguous(), "topk_idx must be contiguous int32");
  FSA_ASSERT(q.stride(2) == 1 && k.stride(2) == 1 && v.stride(2) == 1, "unit stride in head_dim");
  const int64_t b = q.size(0), hq = q.size(1), d = q.size(2), hkv = k.size(1), topk = topk_idx.size(2);
  FSA_ASSERT(topk_idx.size(0) == hkv && topk_idx.size(1) == b, "topk_idx must be [num_kv_heads, B, T]");
  const double scale = default_scale(scale_, d);
  const int64_t dn = native_dim(d);
  if (dn != d) {
    auto [o, lse] =
        decode_selattn(resize_d(q, dn), resize_d(k, dn), resize_d(v, dn), cu_k, topk_idx, block_size, scale, seqlens);
    return {resize_d(o, d), lse};
  }
  const c10::OptionalDeviceGuard guard(q.device());
  Tensor o = at::empty({b, hq, d}, q.options()), lse = empty_f32({hq, b}, q);
  const size_t bytes = std::max<size_t>(256, api.fsa_decode_workspace_bytes((int32_t)b, (int32_t)hq, (int32_t)hkv,
                                                                            (int32_t)d, topk * ((block_size + 31) / 32) * 32));
  Tensor ws = scratch(bytes, q);
  check(api.fsa_decode_selattn(q.data_ptr(), k.data_ptr(), v.data_ptr(), dtype_code(q), q.stride(0), q.stride(1),
                               k.stride(0), k.stride(1), v.stride(0), v.stride(1), i32(cu_k),
                               seqlens ? i32(*seqlens) : nullptr, i32(topk_idx), (int32_t)b, (int32_t)hq, (int32_t)hkv,
                               (int32_t)d, (int32_t)topk, (int32_t)block_size, (float)scale, o.data_ptr(), f32(lse),
                               ws.data_ptr(), bytes, stream_of(q)),
        "fsa_decode_selattn");
  return {o, lse};
}

// One compressed row from `rows` [kernel_size, H, D] (head_dim one of the built sizes).
Tensor compress_window(const Tensor& rows, const Tensor& w, const optional<Tensor>& pe, const Tensor& cu_x,
                       const Tensor& cu_y) {
  const int64_t ks = rows.size(0), h = rows.size(1), d = rows.size(2);
  Tensor y = at::empty({1, h, d}, rows.options());
  const Tensor bias_rows = !pe ? Tensor() : (uintptr_t)pe->data_ptr() % 16 ? pe->clone() : *pe;
  check(api.fsa_linear_compress_fwd(rows.data_ptr(), w.data_ptr(), pe ? bias_rows.data_ptr() : nullptr, dtype_code(rows),
                                    rows.stride(0), rows.stride(1), i32(cu_x), i32(cu_y), 1, 1, (int32_t)h, (int32_t)d,
                                    (int32_t)ks, (int32_t)ks, y.data_ptr(), nullptr, stream_of(rows)),
        "fsa_linear_compress_fwd");
  return y;
}

// The sizes and places that the fused calls of the layer take for granted.  What does not pass is left to the composition
// of the single operators, whose own checks refuse it (a projection of another width, a weight on another device) or
// which serves it.
bool plain_input(const Tensor& t, const Tensor& x, at::IntArrayRef sizes) {
  return t.is_cuda() && t.device() == x.device() && t.scalar_type() == x.scalar_type() && t.is_contiguous() &&
         t.sizes() == sizes && (uintptr_t)t.data_ptr() % 16 == 0;
}
bool layer_config_ok(int64_t hq, int64_t hkv, int64_t d, int64_t ks, int64_t st, int64_t hidden) {
  // (window sizes: what LinearCompress takes)
  return hidden >= 8 && hidden % 8 == 0 && (d == 64 || d == 128 || d == 256) && hq % hkv == 0 && ks % st == 0 &&
         (ks == 16 || ks == 32 || ks == 64 || ks == 128);
}
bool projections_ok(const Tensor& x, const Tensor& w_q, const Tensor& w_k, const Tensor& w_v, const Tensor& w_gate,
                    const Tensor& w_o, int64_t hq, int64_t hkv, int64_t d, int64_t hidden) {
  return plain_input(w_q, x, {hq * d, hidden}) && plain_input(w_k, x, {hkv * d, hidden}) &&
         plain_input(w_v, x, {hkv * d, hidden}) && plain_input(w_gate, x, {3, hidden}) && plain_input(w_o, x, {hidden, hq * d});
}
bool compression_ok(const Tensor& x, const Tensor& w_ck, const Tensor& w_cv, const Tensor& pe, int64_t hkv, int64_t ks, int64_t d) {
  return plain_input(w_ck, x, {hkv, ks * d, d}) && plain_input(w_cv, x, {hkv, ks * d, d}) && plain_input(pe, x, {hkv, ks, d});
}
bool frequencies_ok(const Tensor& x, const Tensor& inv_freq, int64_t d) {
  return inv_freq.device() == x.device() && inv_freq.scalar_type() == at::kFloat && inv_freq.is_contiguous() &&
         inv_freq.numel() == d / 2;
}

// One token of one request through the whole layer.  nullopt: sizes, types or layouts the kernels are not built for (the
// caller then composes the step from the single operators); otherwise y [1, hidden], the new k and v rows and, if the
// token completes a compression window, the new compressed rows.
using DecodeLayerOut = std::tuple<Tensor, Tensor, Tensor, optional<Tensor>, optional<Tensor>>;
optional<DecodeLayerOut> decode_layer(const Tensor& x, const std::vector<Tensor>& caches, const std::vector<Tensor>& weights,
                                      const Tensor& w_ck, const Tensor& w_cv, const Tensor& pe, const Tensor& inv_freq,
                                      double rope_scale, const std::array<int64_t, 10>& shape) {
  const auto [hq, hkv, d, ks, st, bs, topk, init_blocks, local_blocks, window] = shape;
  refuse_tangent(x, w_ck, w_cv, pe);
  for (const Tensor& t : caches) refuse_tangent(t);
  for (const Tensor& t : weights) refuse_tangent(t);
  if (caches.size() != 4 || weights.size() != 5 || x.dim() != 2 || x.size(0) != 1) return std::nullopt;
  const Tensor &k = caches[0], &v = caches[1], &ck = caches[2], &cv = caches[3];
  auto rows_ok = [&](const Tensor& t) {
    return t.is_cuda() && t.device() == x.device() && t.scalar_type() == x.scalar_type() && t.dim() == 3 && t.size(1) == hkv &&
           t.size(2) == d && t.stride(2) == 1 && t.stride(0) >= 0 && t.stride(1) >= 0 && t.stride(0) % 8 == 0 &&
           t.stride(1) % 8 == 0 && (uintptr_t)t.data_ptr() % 16 == 0;
  };
  const int64_t hidden = x.size(1);
  if (!is16(x) || !plain_input(x, x, {1, hidden}) || hkv < 1 || hq < 1 || st < 1 || bs < 1 ||
      !layer_config_ok(hq, hkv, d, ks, st, hidden) || hq / hkv > 16 || hkv > 1024)
    return std::nullopt;
  for (const Tensor& t : caches)
    if (!rows_ok(t)) return std::nullopt;
  const int64_t L = k.size(0);
  if (L < ks - 1 || L < 1 || (L + bs) / bs > 16384 || v.size(0) != L || ck.size(0) != cv.size(0)) return std::nullopt;
  if (!projections_ok(x, weights[0], weights[1], weights[2], weights[3], weights[4], hq, hkv, d, hidden) ||
      !compression_ok(x, w_ck, w_cv, pe, hkv, ks, d) || !frequencies_ok(x, inv_freq, d))
    return std::nullopt;
  const bool completes = (L + 1 - ks) % st == 0;
  if (ck.size(0) + completes < 1) return std::nullopt;

  const c10::OptionalDeviceGuard guard(x.device());
  Tensor y = at::empty({1, hidden}, x.options());
  Tensor k_new = at::empty({1, hkv, d}, x.options()), v_new = at::empty({1, hkv, d}, x.options());
  fsa_decode_layer_args a = {};
  a.x = x.data_ptr();
  a.w_q = weights[0].data_ptr();
  a.w_k = weights[1].data_ptr();
  a.w_v = weights[2].data_ptr();
  a.w_gate = weights[3].data_ptr();
  a.w_o = weights[4].data_ptr();
  a.k_cache = k.data_ptr();
  a.v_cache = v.data_ptr();
  a.ck_cache = ck.data_ptr();
  a.cv_cache = cv.data_ptr();
  a.k_stride_n = k.stride(0);
  a.k_stride_h = k.stride(1);
  a.v_stride_n = v.stride(0);
  a.v_stride_h = v.stride(1);
  a.ck_stride_n = ck.stride(0);
  a.ck_stride_h = ck.stride(1);
  a.cv_stride_n = cv.stride(0);
  a.cv_stride_h = cv.stride(1);
  a.inv_freq = f32(inv_freq);
  a.cache_len = L;
  a.ck_len = ck.size(0);
  a.dtype = dtype_code(x);
  a.hidden = (int32_t)hidden;
  a.num_q_heads = (int32_t)hq;
  a.num_kv_heads = (int32_t)hkv;
  a.head_dim = (int32_t)d;
  a.kernel_size = (int32_t)ks;
  a.kernel_stride = (int32_t)st;
  a.block_size = (int32_t)bs;
  a.topk = (int32_t)topk;
  a.init_blocks = (int32_t)init_blocks;
  a.local_blocks = (int32_t)local_blocks;
  a.window = (int32_t)window;
  a.softmax_scale = (float)(1.0 / std::sqrt((double)d));
  a.rope_scale = (float)rope_scale;
  a.k_new = k_new.data_ptr();
  a.v_new = v_new.data_ptr();
  a.y = y.data_ptr();
  a.workspace_bytes = api.fsa_decode_layer_workspace_bytes(&a);
  Tensor ws = scratch(a.workspace_bytes, x);
  a.workspace = ws.data_ptr();
  check(api.fsa_decode_layer_project(&a, stream_of(x)), "fsa_decode_layer");
  optional<Tensor> ck_new, cv_new;
  if (completes) {
    const auto opts = x.options().dtype(at::kInt);
    const Tensor cu_x = at::arange(0, 2 * ks, ks, opts), cu_y = at::arange(0, 2, 1, opts);
    ck_new = compress_window(at::cat({k.narrow(0, L - ks + 1, ks - 1), k_new}), w_ck, pe, cu_x, cu_y);
    cv_new = compress_window(at::cat({v.narrow(0, L - ks + 1, ks - 1), v_new}), w_cv, std::nullopt, cu_x, cu_y);
    a.ck_new = ck_new->data_ptr();
    a.cv_new = cv_new->data_ptr();
  }
  check(api.fsa_decode_layer_attend(&a, stream_of(x)), "fsa_decode_layer");
  return DecodeLayerOut{y, k_new, v_new, ck_new, cv_new};
}

// ---- the layer: projections of q, k, v and the attention core as one autograd node ----
using LayerShape = std::array<int64_t, 11>;  // Hq, Hkv, D, kernel_size, stride, block, topk, init, local, window, hidden
struct LayerSizes {
  int64_t total_ck, max_len, max_ck;
};

fsa_layer_args layer_args(const Tensor& x, const Tensor& cu, const Tensor& w_gate, const Tensor& w_ck, const Tensor& w_cv,
                          const Tensor& pe, const Tensor& inv_freq, double rope_scale, const LayerShape& shape,
                          const LayerSizes& z) {
  fsa_layer_args a = {};
  a.dtype = dtype_code(x);
  a.num_q_heads = (int32_t)shape[0];
  a.num_kv_heads = (int32_t)shape[1];
  a.head_dim = (int32_t)shape[2];
  a.kernel_size = (int32_t)shape[3];
  a.kernel_stride = (int32_t)shape[4];
  a.block_size = (int32_t)shape[5];
  a.topk = (int32_t)shape[6];
  a.init_blocks = (int32_t)shape[7];
  a.local_blocks = (int32_t)shape[8];
  a.window = (int32_t)shape[9];
  a.hidden = (int32_t)shape[10];
  a.batch = (int32_t)cu.numel() - 1;
  a.total_tokens = x.size(0);
  a.total_ck = z.total_ck;
  a.max_len = z.max_len;
  a.max_ck = z.max_ck;
  a.softmax_scale = (float)(1.0 / std::sqrt((double)shape[2]));
  a.rope_scale = (float)rope_scale;
  a.x = x.data_ptr();
  a.w_gate = w_gate.data_ptr();
  a.w_ck = w_ck.data_ptr();
  a.w_cv = w_cv.data_ptr();
  a.pe = pe.data_ptr();
  a.cu_seqlens = i32(cu);
  a.inv_freq = f32(inv_freq);
  return a;
}

// The end of a copy to the host, to wait for without waiting for what is queued behind it.
struct HostCopy {
  hipEvent_t event = nullptr;
  void record(hipStream_t stream) {
    TORCH_CHECK(hipEventCreateWithFlags(&event, hipEventDisableTiming) == hipSuccess && hipEventRecord(event, stream) == hipSuccess,
                "cannot record an event");
  }
  void wait() { TORCH_CHECK(hipEventSynchronize(event) == hipSuccess, "the copy of cu_seqlens to the host failed"); }
  ~HostCopy() {
    if (event) (void)hipEventDestroy(event);
  }
};

// Whether the products of a layer run as fsa_matmul launches instead of library calls: a bound on the operations of q, k and
// v.  A whole pass of one sequence, library / ours in us (below some 225 us in training and 77 in inference the library's
// products cost the host more than the device):
//   hidden 4096, 32 + 8 heads: inference 300 tokens (15e9) 129 / 127, 700 (35e9) 171 / 174; training 700 tokens 586 / 584
//   hidden 2048, 16 + 4 heads: inference 1000 tokens (13e9) 122 / 112, 2000 (25e9) 167 / 162; training 2500 (31e9) 744 / 709
//   hidden 1024,  8 + 2 heads: inference 5000 tokens (16e9) 216 / 206, 8000 (25e9) 331 / 322; training 9000 (28e9) 1357 / 1192
// The line suits the wide layer; narrower ones are handed over earlier than they need be.
bool own_products(int64_t n, int64_t hidden, const LayerShape& shape) {
  return 2.0 * (double)n * (double)hidden * (double)((shape[0] + 2 * shape[1]) * shape[2]) <= 24e9;
}

fsa_matmul_out product(const Tensor& c, const Tensor* add = nullptr) {
  fsa_matmul_out o = {};
  o.m = (int32_t)c.size(0);
  o.n = (int32_t)c.size(1);
  o.c = c.data_ptr();
  o.ldc = c.stride(0);
  o.add = add ? add->data_ptr() : nullptr;
  return o;
}
void add_part(fsa_matmul_out& o, const Tensor& a, const Tensor& b, int64_t k) {
  o.part[o.parts++] = {a.data_ptr(), b.data_ptr(), a.stride(0), b.stride(0), (int32_t)k};
}
void matmul(const fsa_matmul_out* outs, int n, int form, const Tensor& like) {
  check(api.fsa_matmul(outs, n, form, dtype_code(like), stream_of(like)), "fsa_matmul");
}

struct LayerForward {
  Tensor q, k, v, saved, out, topk_idx, y;   // out: merged heads; y: their projection
};
// `lens`: host copy of cu_seqlens that is on its way (batches of several sequences), waited for when the projections are
// queued; null: one sequence, as long as x.
LayerForward layer_forward(const Tensor& x, const Tensor& cu, const Tensor& w_q, const Tensor& w_k, const Tensor& w_v,
                           const Tensor& w_o, const Tensor& w_gate, const Tensor& w_ck, const Tensor& w_cv, const Tensor& pe,
                           const Tensor& inv_freq, double rope_scale, const LayerShape& shape, LayerSizes& z,
                           const Tensor* lens, HostCopy* copied, bool training) {
  LayerForward f;
  const bool own = own_products(x.size(0), x.size(1), shape);
  if (own) {
    Tensor* y[3] = {&f.q, &f.k, &f.v};
    const Tensor* w[3] = {&w_q, &w_k, &w_v};
    fsa_matmul_out o[3];
    for (int i = 0; i < 3; ++i) {
      *y[i] = at::empty({x.size(0), w[i]->size(0)}, x.options());
      o[i] = product(*y[i]);
      add_part(o[i], x, *w[i], x.size(1));
    }
    matmul(o, 3, FSA_MM_NT | FSA_MM_IN_ORDER, x);   // the block selection depends on their last bits
  } else {
    f.q = at::linear(x, w_q);
    f.k = at::linear(x, w_k);
    f.v = at::linear(x, w_v);
  }
  if (lens) {
    copied->wait();
    const int32_t* c = i32(*lens);
    z = {0, 0, 0};
    for (int64_t s = 0; s + 1 < lens->numel(); ++s) {
      const int64_t len = c[s + 1] - c[s], nc = len >= shape[3] ? (len - shape[3]) / shape[4] + 1 : 0;
      z.total_ck += nc;
      z.max_len = std::max(z.max_len, len);
      z.max_ck = std::max(z.max_ck, nc);
    }
    if (z.total_ck < 1) throw NoKernel();  // no sequence has a compressed key
  }
  fsa_layer_args a = layer_args(x, cu, w_gate, w_ck, w_cv, pe, inv_freq, rope_scale, shape, z);
  a.inference = !training;
  a.q = f.q.data_ptr();
  a.k = f.k.data_ptr();
  a.v = f.v.data_ptr();
  a.saved_bytes = api.fsa_layer_saved_bytes(&a);
  a.workspace_bytes = api.fsa_layer_workspace_bytes(&a, 0);
  f.saved = scratch(a.saved_bytes, x);
  Tensor ws = scratch(a.workspace_bytes, x);
  a.saved = f.saved.data_ptr();
  a.workspace = ws.data_ptr();
  f.out = at::empty({x.size(0), shape[0] * shape[2]}, x.options());
  const int64_t t_out = std::min<int64_t>(shape[6], (z.max_len + shape[5] - 1) / shape[5]);
  f.topk_idx = empty_i32({shape[1], x.size(0), t_out}, x);
  check(api.fsa_layer_forward(&a, f.out.data_ptr(), (int32_t*)i32(f.topk_idx), stream_of(x)), "fsa_layer_forward");
  if (own) {
    f.y = at::empty({x.size(0), w_o.size(0)}, x.options());
    fsa_matmul_out o = product(f.y);
    add_part(o, f.out, w_o, f.out.size(1));
    matmul(&o, 1, FSA_MM_NT, x);
  } else {
    f.y = at::linear(f.out, w_o);
  }
  return f;
}

// Inputs with gradients first: x, w_q, w_k, w_v, w_o, w_gate, w_ck, w_cv, pe.
struct LayerCore : torch::autograd::Function<LayerCore> {
  static torch::autograd::variable_list forward(torch::autograd::AutogradContext* ctx, const Tensor& x, const Tensor& w_q,
                                                const Tensor& w_k, const Tensor& w_v, const Tensor& w_o, const Tensor& w_gate,
                                                const Tensor& w_ck, const Tensor& w_cv, const Tensor& pe, const Tensor& cu,
                                                const Tensor& inv_freq, double rope_scale, const LayerShape* shape,
                                                LayerSizes z, const Tensor* lens, HostCopy* copied) {
    LayerForward f = layer_forward(x, cu, w_q, w_k, w_v, w_o, w_gate, w_ck, w_cv, pe, inv_freq, rope_scale, *shape, z, lens,
                                   copied, true);
    const Tensor merged = w_o.requires_grad() ? f.out : Tensor();
    ctx->save_for_backward({x, w_q, w_k, w_v, w_o, w_gate, w_ck, w_cv, pe, cu, inv_freq, f.k, f.v, f.saved, merged});
    ctx->saved_data["shape"] = std::vector<int64_t>(shape->begin(), shape->end());
    ctx->saved_data["sizes"] = std::vector<int64_t>{z.total_ck, z.max_len, z.max_ck};
    ctx->saved_data["rope_scale"] = rope_scale;
    ctx->mark_non_differentiable({f.topk_idx});
    ctx->set_materialize_grads(false);
    return {f.y, f.topk_idx};
  }

  static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx, torch::autograd::variable_list grads) {
    if (!grads[0].defined()) return torch::autograd::variable_list(16);
    const auto s = ctx->get_saved_variables();
    const Tensor &x = s[0], &w_q = s[1], &w_k = s[2], &w_v = s[3], &w_o = s[4], &w_gate = s[5], &w_ck = s[6], &w_cv = s[7],
                 &pe = s[8], &cu = s[9], &k = s[11], &v = s[12], &saved = s[13], &merged = s[14];
    const auto shape_v = ctx->saved_data["shape"].toIntVector(), sizes = ctx->saved_data["sizes"].toIntVector();
    LayerShape shape;
    std::copy(shape_v.begin(), shape_v.end(), shape.begin());
    const c10::OptionalDeviceGuard guard(x.device());
    const Tensor dy = grads[0].contiguous();
    const bool own = own_products(x.size(0), x.size(1), shape) && (uintptr_t)dy.data_ptr() % 16 == 0;
    Tensor d_out;
    if (own) {
      d_out = at::empty({dy.size(0), w_o.size(1)}, dy.options());
      fsa_matmul_out o = product(d_out);
      add_part(o, dy, w_o, w_o.size(0));
      matmul(&o, 1, FSA_MM_NN, x);
    } else {
      d_out = at::mm(dy, w_o);
    }
    fsa_layer_args a = layer_args(x, cu, w_gate, w_ck, w_cv, pe, s[10], ctx->saved_data["rope_scale"].toDouble(), shape,
                                  {sizes[0], sizes[1], sizes[2]});
    a.q = a.k = k.data_ptr();  // the un-rotated q is not needed again
    a.v = v.data_ptr();
    a.saved = saved.data_ptr();
    a.saved_bytes = saved.numel();
    a.workspace_bytes = api.fsa_layer_workspace_bytes(&a, 1);
    const bool need_x = ctx->needs_input_grad(0);
    Tensor dx, dq = at::empty({x.size(0), w_q.size(0)}, x.options()), dk = at::empty_like(k), dv = at::empty_like(v);
    Tensor dw_gate = at::empty_like(w_gate), dw_ck = at::empty_like(w_ck), dw_cv = at::empty_like(w_cv), dpe = at::empty_like(pe);
    if (need_x) dx = at::empty_like(x);
    {
      Tensor ws = scratch(a.workspace_bytes, x);
      a.workspace = ws.data_ptr();
      fsa_layer_grads g = {d_out.data_ptr(), dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), need_x ? dx.data_ptr() : nullptr,
                           dw_gate.data_ptr(), dw_ck.data_ptr(), dw_cv.data_ptr(), dpe.data_ptr()};
      check(api.fsa_layer_backward(&a, &g, stream_of(x)), "fsa_layer_backward");
    }
    // weight gradients d^T x (the output projection: dy^T merged), and the share of dx on top of the gate's, without
    // separate sums over [N, hidden]
    Tensor dw[4];
    const Tensor d[4] = {dq, dk, dv, dy};
    const Tensor* rhs[4] = {&x, &x, &x, &merged};
    const Tensor* w[4] = {&w_q, &w_k, &w_v, &w_o};
    fsa_matmul_out o[4];
    int n_out = 0;
    for (int i = 0; i < 4; ++i) {
      if (!ctx->needs_input_grad(1 + i)) continue;
      if (own) {
        dw[i] = at::empty_like(*w[i]);
        o[n_out] = product(dw[i]);
        add_part(o[n_out++], d[i], *rhs[i], x.size(0));
      } else {
        dw[i] = at::mm(d[i].t(), *rhs[i]);
      }
    }
    if (n_out) matmul(o, n_out, FSA_MM_TN, x);
    if (need_x && own) {
      o[0] = product(dx, &dx);
      for (int i = 0; i < 3; ++i) add_part(o[0], d[i], *w[i], d[i].size(1));
      matmul(o, 1, FSA_MM_NN, x);
    } else if (need_x) {
      for (int i = 0; i < 3; ++i) dx.addmm_(d[i], *w[i]);
    }
    auto wanted = [&](int i, const Tensor& t) { return ctx->needs_input_grad(i) ? t : Tensor(); };
    return {dx,       dw[0],    dw[1],    dw[2],    dw[3],    wanted(5, dw_gate), wanted(6, dw_ck), wanted(7, dw_cv), wanted(8, dpe),
            Tensor(), Tensor(), Tensor(), Tensor(), Tensor(), Tensor(),           Tensor()};
  }
};

// nullopt: sizes, types or layouts the kernels are not built for (the caller composes the layer from the single operators).
optional<std::pair<Tensor, Tensor>> layer_core(const Tensor& x, const Tensor& cu, const Tensor& w_q, const Tensor& w_k,
                                               const Tensor& w_v, const Tensor& w_o, const Tensor& w_gate,
                                               const Tensor& w_ck, const Tensor& w_cv, const Tensor& pe, const Tensor& inv_freq, double rope_scale,
                                               const LayerShape& shape, bool exact_lens) {
  const int64_t hq = shape[0], hkv = shape[1], d = shape[2], ks = shape[3], st = shape[4], bs = shape[5], hidden = shape[10];
  refuse_tangent(x, w_q, w_k, w_v, w_o, w_gate, w_ck, w_cv, pe);
  if (!is16(x) || x.dim() != 2 || x.size(0) < 1 || !plain_input(x, x, {x.size(0), hidden}) || hkv < 1 || hq < 1 || st < 1 ||
      !layer_config_ok(hq, hkv, d, ks, st, hidden) || (bs != 32 && bs != 64 && bs != 128) || bs % st ||
      shape[6] < std::max<int64_t>(1, shape[7] + shape[8]) || !cu.is_cuda() || cu.device() != x.device() ||
      cu.scalar_type() != at::kInt || cu.dim() != 1 || cu.numel() < 2 || !cu.is_contiguous() || !frequencies_ok(x, inv_freq, d) ||
      !projections_ok(x, w_q, w_k, w_v, w_gate, w_o, hq, hkv, d, hidden) || !compression_ok(x, w_ck, w_cv, pe, hkv, ks, d))
    return std::nullopt;
  const c10::OptionalDeviceGuard guard(x.device());
  const int64_t n = x.size(0);
  // Upper bounds are all the kernels need.  One sequence: its length is at most that of x.  More sequences: the same
  // bounds, as long as grids sized for the whole of x cost less than a wait for the device; otherwise (or where exact
  // shapes are wanted) the lengths are copied to the host while the projections run.
  const int64_t batch = cu.numel() - 1, most_ck = batch == 1 ? (n >= ks ? (n - ks) / st + 1 : 0) : n / st;
  LayerSizes z = {most_ck, n, n >= ks ? (n - ks) / st + 1 : 0};
  Tensor lens;
  HostCopy copied;
  if (exact_lens || (batch > 1 && n * batch > 32768)) {
    lens = at::empty({cu.numel()}, at::TensorOptions().dtype(at::kInt).pinned_memory(true));
    lens.copy_(cu, /*non_blocking=*/true);
    copied.record((hipStream_t)stream_of(x));
  } else if (z.max_ck < 1) {
    return std::nullopt;
  }
  const Tensor* lp = lens.defined() ? &lens : nullptr;
  bool grad = false;
  for (const Tensor* t : {&x, &w_q, &w_k, &w_v, &w_o, &w_gate, &w_ck, &w_cv, &pe}) grad |= t->requires_grad();
  try {
    if (grad && at::GradMode::is_enabled()) {
      const auto out = LayerCore::apply(x, w_q, w_k, w_v, w_o, w_gate, w_ck, w_cv, pe, cu, inv_freq, rope_scale, &shape, z, lp,
                                        &copied);
      return std::make_pair(out[0], out[1]);
    }
    const LayerForward f =
        layer_forward(x, cu, w_q, w_k, w_v, w_o, w_gate, w_ck, w_cv, pe, inv_freq, rope_scale, shape, z, lp, &copied, false);
    return std::make_pair(f.y, f.topk_idx);
  } catch (const NoKernel&) {
    return std::nullopt;
  }
}

}  // namespace

PYBIND11_MODULE(_native, m) {
  py::register_exception_translator([](std::exception_ptr p) {
    try {
      if (p) std::rethrow_exception(p);
    } catch (const AssertionFailed& e) {
      PyErr_SetString(PyExc_AssertionError, e.what());
    }
  });
  m.def("bind_library", &bind_library);
  m.def("build_index", &build_index);
  m.def("split_topk_blocks", &split_topk_blocks);
  m.def("selattn_fwd", &selattn_fwd);
  m.def("selattn_fwd_lists", &selattn_fwd_lists);
  m.def("selattn_bwd", &selattn_bwd);
  m.def("selected_attention", &selected_attention);
  m.def("decode_cmpattn", &decode_cmpattn);
  m.def("decode_topk", &decode_topk);
  m.def("decode_selattn", &decode_selattn);
  m.def("decode_layer", &decode_layer);
  m.def("layer_core", &layer_core, py::call_guard<py::gil_scoped_release>());
}
