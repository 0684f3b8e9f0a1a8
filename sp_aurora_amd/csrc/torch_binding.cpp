// CPython module sp_aurora_amd._native: the host path of the public calls, from torch tensors to the C ABI.
//
// A call of the operator on a small block lasts 5 to 15 us on the GPU, and what Python and ctypes spent in front of it
// was as much again (12 us forward, 150 us for a forward and a backward through torch.autograd.Function).  The
// functions here take the arguments that a well-formed call has - contiguous head dim, 16-byte aligned rows, one device, one
// dtype - allocate the results and enqueue the kernels; the differentiable ones are C++ autograd nodes, whose backward runs on
// the autograd thread without the interpreter.  For anything else (an argument that needs a copy, a check that fails,
// a forward entry point that refuses) they return None, and the Python code behind them does the copy or raises the error.
#include <Python.h>
#include <hip/hip_runtime_api.h>

#include <ATen/core/Tensor.h>
#include <ATen/ops/empty.h>
#include <ATen/ops/zeros.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/GradMode.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>
#include <torch/csrc/utils/pybind.h>

#include <cmath>

#include "../../include/sp_aurora_hip.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

constexpr auto kFp8 = at::kFloat8_e4m3fn;

int dtype_code(at::ScalarType t) { return t == at::kFloat ? SPA_F32 : t == at::kBFloat16 ? SPA_BF16 : t == at::kHalf ? SPA_F16 : -1; }

// Rows that the kernels can address: inner stride 1, base and every other stride a multiple of `bytes`.
bool rows_ok(const Tensor& t, int64_t bytes = 16) {
  const auto st = t.strides();
  const int64_t esz = t.element_size(), n = t.dim();
  if (st[n - 1] != 1 || ((uintptr_t)t.const_data_ptr() % bytes) != 0) return false;
  for (int64_t i = 0; i + 1 < n; ++i)
    if ((st[i] * esz) % bytes != 0) return false;
  return true;
}

// One operand as the C ABI takes it: pointer, (batch, head, seq) strides in elements, sizes.  shards: of a rank-stacked tensor;
// pitch: rows from one shard to the next where a sequence's rows lie in shards, 0 where they follow each other.
struct View {
  void* p = nullptr;
  int64_t st[3] = {0, 0, 0};
  int B = 0, H = 0, S = 0, D = 0, shards = 1, pitch = 0;
  bool same_shape(const View& o) const { return B == o.B && H == o.H && S == o.S && D == o.D; }
};

// [B,S,H,D] (bshd) or [B,H,S,D]; `part` of a packed [B,S,n,H,D] tensor when part >= 0; a rank-stacked [P,B,s,H,D] tensor as the
// sequences [B,P*s,H,D] in shards.
bool view_of(const Tensor& t, bool bshd, View& v, int part = -1) {
  const auto sz = t.sizes();
  const auto st = t.strides();
  for (const int64_t n : sz)
    if (n <= 0 || n > 0x7fffffffLL) return false;
  v.p = t.data_ptr();
  if (part >= 0) {
    if (t.dim() != 5) return false;
    v.B = (int)sz[0]; v.S = (int)sz[1]; v.H = (int)sz[3]; v.D = (int)sz[4];
    v.st[0] = st[0]; v.st[1] = st[3]; v.st[2] = st[1];
    v.p = (char*)v.p + part * st[2] * (int64_t)t.element_size();
    return true;
  }
  if (t.dim() == 5) {
    if (!bshd || sz[0] * sz[2] > 0x7fffffffLL || st[2] <= 0) return false;
    v.B = (int)sz[1]; v.S = (int)(sz[0] * sz[2]); v.H = (int)sz[3]; v.D = (int)sz[4];
    v.st[0] = st[1]; v.st[1] = st[3]; v.st[2] = st[2];
    v.shards = (int)sz[0];
    if (sz[0] > 1 && st[0] != sz[2] * st[2]) {
      if (st[0] % st[2] != 0 || st[0] / st[2] < sz[2] || st[0] / st[2] > 0x7fffffffLL) return false;
      v.pitch = (int)(st[0] / st[2]);
    }
    return true;
  }
  if (t.dim() != 4) return false;
  const int s = bshd ? 1 : 2, h = bshd ? 2 : 1;
  v.B = (int)sz[0]; v.S = (int)sz[s]; v.H = (int)sz[h]; v.D = (int)sz[3];
  v.st[0] = st[0]; v.st[1] = st[h]; v.st[2] = st[s];
  return true;
}

// A packed [rows,H,D] tensor; strides (head, row).
bool view_thd(const Tensor& t, View& v) {
  if (t.dim() != 3) return false;
  const auto sz = t.sizes();
  for (const int64_t n : sz)
    if (n <= 0 || n > 0x7fffffffLL) return false;
  v.p = t.data_ptr();
  v.B = 1; v.S = (int)sz[0]; v.H = (int)sz[1]; v.D = (int)sz[2];
  v.st[0] = t.stride(1); v.st[1] = t.stride(0);
  return true;
}

// Rows that lie over each other (a broadcast): the backward's kernels cannot stream such a q or gradient, whose rows past the end have
// to be out of the tensor's range.
bool rows_shared(const View& v, int row) { return v.S > 1 && v.st[row] < v.D; }

bool on_device(const Tensor& t, const Tensor& q) { return t.is_cuda() && t.device() == q.device(); }

// fp32 [n, H] on q's device.
bool scale_ok(const Tensor& t, const Tensor& q, int64_t n, int64_t H) {
  return t.defined() && on_device(t, q) && t.scalar_type() == at::kFloat && t.dim() == 2 && t.size(0) == n && t.size(1) == H && t.is_contiguous();
}

// The stream that is current on the calling thread (of the current device, as torch.cuda.current_stream()).
void* current_stream() { return c10::hip::getCurrentHIPStream().stream(); }

float softmax_scale_or_default(double scale, int D) { return (float)(std::isnan(scale) ? 1.0 / std::sqrt((double)D) : scale); }

Tensor empty_f32(at::IntArrayRef sizes, const Tensor& like) { return at::empty(sizes, like.options().dtype(at::kFloat)); }

// ---------------------------------------------------------------- forward
// One block call (ks, vs: e4m3 K / V).  Few query rows against many keys: the keys split over the grid, the chunks' results in a
// workspace (not while the stream is being captured: the workspace would not outlive this call); a call that the split entries do not take
// runs whole.
int block_fwd(const View& q, const View& k, const View& v, const View& o, float* lse, const float* ks, const float* vs, float scale, int mask, int dtype,
              const Tensor& like, void* stream) {
  if (mask == SPA_MASK_NONE && dtype != SPA_F32 && (q.D == 64 || q.D == 128)) {
    int n = spa_flash_fwd_splitkv_suggest(q.B, q.H, q.S, k.S, q.D, mask, dtype);
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    if (n > 1 && (hipStreamIsCapturing((hipStream_t)stream, &cap) != hipSuccess || cap != hipStreamCaptureStatusNone)) n = 1;
    if (n > 1) {
      const Tensor ws = at::empty({spa_flash_fwd_splitkv_workspace_bytes(q.B, q.H, q.S, q.D, n, dtype)}, like.options().dtype(at::kByte));
      const int rc =
          ks ? spa_flash_fwd_splitkv_fp8kv(q.p, k.p, v.p, ks, vs, o.p, lse, ws.data_ptr(), q.B, q.H, q.S, k.S, q.D, n, q.st, k.st, v.st, o.st, scale,
                                           dtype, stream)
             : spa_flash_fwd_splitkv(q.p, k.p, v.p, o.p, lse, ws.data_ptr(), q.B, q.H, q.S, k.S, q.D, n, q.st, k.st, v.st, o.st, scale, dtype, stream);
      if (rc == SPA_OK) return rc;
    }
  }
  if (ks) return spa_flash_fwd_fp8kv(q.p, k.p, v.p, ks, vs, o.p, lse, q.B, q.H, q.S, k.S, q.D, q.st, k.st, v.st, o.st, scale, mask, dtype, stream);
  return spa_flash_fwd(q.p, k.p, v.p, o.p, lse, q.B, q.H, q.S, k.S, q.D, q.st, k.st, v.st, o.st, scale, mask, dtype, stream);
}

// (out, lse) of one block call; false: not a call for this path.
bool flash_fwd(const Tensor& q, const Tensor& k, const Tensor& v, double scale_or_nan, bool causal, bool bshd, const Tensor& q_scale,
               const Tensor& k_scale, const Tensor& v_scale, int out_dtype, Tensor& out, Tensor& lse) {
  if (q.dim() != 4 || k.dim() != 4 || v.dim() != 4 || !q.is_cuda() || !on_device(k, q) || !on_device(v, q)) return false;
  const bool q8 = q.scalar_type() == kFp8, kv8 = k.scalar_type() == kFp8;
  if (v.scalar_type() != k.scalar_type() || (q8 && !kv8) || (!kv8 && k.scalar_type() != q.scalar_type())) return false;
  const int dtype = q8 ? out_dtype : dtype_code(q.scalar_type());
  if (dtype < 0) return false;
  View a, b, c;
  if (!rows_ok(q) || !rows_ok(k, kv8 && !q8 ? 8 : 16) || !rows_ok(v, q8 ? 16 : kv8 ? 8 : 16) || !view_of(q, bshd, a) || !view_of(k, bshd, b) ||
      !view_of(v, bshd, c) || !b.same_shape(c) || a.B != b.B || a.H != b.H || a.D != b.D)
    return false;
  if (kv8 && (!scale_ok(k_scale, q, a.B, a.H) || !scale_ok(v_scale, q, a.B, a.H) || (q8 && !scale_ok(q_scale, q, a.B, a.H)))) return false;
  const float scale = softmax_scale_or_default(scale_or_nan, a.D);
  void* const stream = current_stream();
  const c10::DeviceGuard guard(q.device());
  out = at::empty(q.sizes(), q8 ? q.options().dtype(dtype == SPA_F16 ? at::kHalf : at::kBFloat16) : q.options());
  lse = empty_f32({a.B, a.H, a.S}, q);
  View o;
  view_of(out, bshd, o);
  float* const lp = (float*)lse.data_ptr();
  const int mask = causal ? SPA_MASK_CAUSAL : SPA_MASK_NONE;
  const float* const ks = kv8 ? (const float*)k_scale.const_data_ptr() : nullptr;
  const float* const vs = kv8 ? (const float*)v_scale.const_data_ptr() : nullptr;
  if (q8)
    return spa_flash_fwd_fp8qkv(a.p, b.p, c.p, (const float*)q_scale.const_data_ptr(), ks, vs, o.p, lp, a.B, a.H, a.S, b.S, a.D, a.st, b.st, c.st,
                                o.st, scale, mask, dtype, stream) == SPA_OK;
  return block_fwd(a, b, c, o, lp, ks, vs, scale, mask, dtype, q, stream) == SPA_OK;
}

bool cu_ok(const Tensor& cu, const Tensor& q) {
  return on_device(cu, q) && cu.scalar_type() == at::kInt && cu.dim() == 1 && cu.numel() >= 2 && cu.is_contiguous();
}

bool varlen_fwd(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& cu_q, const Tensor& cu_k, int64_t max_q, int64_t max_k,
                double scale_or_nan, bool causal, const Tensor& k_scale, const Tensor& v_scale, Tensor& out, Tensor& lse, int shards = 1,
                bool zigzag = false) {
  if (!q.is_cuda() || !on_device(k, q) || !on_device(v, q) || !cu_ok(cu_q, q) || !cu_ok(cu_k, q) || cu_q.numel() != cu_k.numel()) return false;
  const bool kv8 = k.scalar_type() == kFp8;
  const int dtype = dtype_code(q.scalar_type());
  View a, b, c, o;
  if (dtype < 0 || v.scalar_type() != k.scalar_type() || (!kv8 && k.scalar_type() != q.scalar_type()) || !view_thd(q, a) || !view_thd(k, b) ||
      !view_thd(v, c) || !b.same_shape(c) || a.H != b.H || a.D != b.D || !rows_ok(q) || !(kv8 ? k.is_contiguous() && v.is_contiguous() : rows_ok(k) && rows_ok(v)))
    return false;
  const int nseq = (int)cu_q.numel() - 1;
  if (kv8 && (!scale_ok(k_scale, q, nseq, a.H) || !scale_ok(v_scale, q, nseq, a.H))) return false;
  const float scale = softmax_scale_or_default(scale_or_nan, a.D);
  void* const stream = current_stream();
  const c10::DeviceGuard guard(q.device());
  out = at::empty(q.sizes(), q.options());
  lse = empty_f32({a.H, a.S}, q);
  view_thd(out, o);
  const int mask = causal ? SPA_MASK_CAUSAL : SPA_MASK_NONE;
  const int* const cq = (const int*)cu_q.const_data_ptr();
  const int* const ck = (const int*)cu_k.const_data_ptr();
  float* const lp = (float*)lse.data_ptr();
  if (shards > 1) {
    // P stacked shards, cu_q describes one of them
    if (kv8 || a.S % shards != 0 || b.S != a.S || b.st[1] != c.st[1]) return false;
    const spa_shards rows = {shards, a.S / shards, a.S / shards, zigzag};
    return spa_attention_fwd_varlen(a.p, b.p, c.p, o.p, lp, cq, nseq, a.H, a.S / shards, (int)max_q, a.D, a.st, b.st, c.st, o.st, &rows, scale, mask,
                                    dtype, stream) == SPA_OK;
  }
  // few query rows: the keys in chunks, as in flash_fwd (a call that the split entry does not take runs whole)
  const int chunk = causal ? 0 : spa_flash_fwd_varlen_splitkv_suggest(nseq, a.H, b.S, (int)max_q, (int)max_k, a.D, dtype);
  hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
  if (chunk > 0 && hipStreamIsCapturing((hipStream_t)stream, &cap) == hipSuccess && cap == hipStreamCaptureStatusNone) {
    const Tensor ws = at::empty({spa_flash_fwd_varlen_splitkv_workspace_bytes(nseq, a.H, b.S, (int)max_q, (int)max_k, a.D, chunk)},
                                q.options().dtype(at::kByte));
    if (spa_flash_fwd_varlen_splitkv(a.p, b.p, c.p, kv8 ? (const float*)k_scale.const_data_ptr() : nullptr,
                                     kv8 ? (const float*)v_scale.const_data_ptr() : nullptr, o.p, lp, ws.data_ptr(), cq, ck, nseq, a.H, a.S, b.S,
                                     (int)max_q, (int)max_k, a.D, chunk, a.st, b.st, c.st, o.st, scale, dtype, stream) == SPA_OK)
      return true;
  }
  if (kv8)
    return spa_flash_fwd_varlen_fp8kv(a.p, b.p, c.p, (const float*)k_scale.const_data_ptr(), (const float*)v_scale.const_data_ptr(), o.p, lp, cq, ck,
                                      nseq, a.H, a.S, b.S, (int)max_q, (int)max_k, a.D, a.st, b.st, c.st, o.st, scale, mask, dtype, stream) == SPA_OK;
  return spa_flash_fwd_varlen(a.p, b.p, c.p, o.p, lp, cq, ck, nseq, a.H, a.S, b.S, (int)max_q, (int)max_k, a.D, a.st, b.st, c.st, o.st, scale, mask,
                              dtype, stream) == SPA_OK;
}

// ---------------------------------------------------------------- differentiable calls
// The operands of a differentiable call are separate tensors, q and a packed kv, or one packed qkv: `n` tensors, and the
// gradients come back packed the same way, each written once by the kernels.
struct Operands {
  View q, k, v;
};
bool operands(const Tensor* t, int n, Operands& o) {
  if (n == 3) return view_of(t[0], true, o.q) && view_of(t[1], true, o.k) && view_of(t[2], true, o.v);
  if (n == 2) return view_of(t[0], true, o.q) && view_of(t[1], true, o.k, 0) && view_of(t[1], true, o.v, 1);
  return view_of(t[0], true, o.q, 0) && view_of(t[0], true, o.k, 1) && view_of(t[0], true, o.v, 2);
}
bool differentiable_ok(const Tensor* t, int n) {
  const int dtype = dtype_code(t[0].scalar_type());
  if (dtype < 0 || !t[0].is_cuda()) return false;
  for (int i = 0; i < n; ++i)
    if (!on_device(t[i], t[0]) || t[i].scalar_type() != t[0].scalar_type() || t[i].dim() < 3 || !rows_ok(t[i])) return false;
  return true;
}
// Rows from one shard to the next in a compact tensor of the operand's shape (0: they follow each other), as results and gradients are.
int compact_pitch(const View& v) { return v.shards > 1 && v.B > 1 ? v.B * (v.S / v.shards) : 0; }

// Where the rows lie: false when the operands do not agree among each other or with compact results (rank-stacked tensors that are a
// view of [B,S,H,D]: their rows follow each other, those of the results do not).  zigzag: shards of a zigzag-sharded [B,S,H,D]
// ring, 0 = none.
bool rows_of(const View& q, const View& k, const View& v, int64_t zigzag, spa_shards& rows, const spa_shards*& arg) {
  arg = nullptr;
  if (q.pitch != k.pitch || q.pitch != v.pitch || q.pitch != compact_pitch(q)) return false;
  if (q.pitch) {
    if (zigzag || k.S != q.S) return false;
    rows = {q.shards, q.pitch, q.S / q.shards, 0};
    arg = &rows;
  } else if (zigzag) {
    if (zigzag < 1 || k.S != q.S || q.S % (2 * zigzag) != 0) return false;
    rows = {(int)zigzag, (int)(q.S / zigzag), (int)(q.S / zigzag), 1};
    arg = &rows;
  }
  return !arg || k.st[2] == v.st[2];
}

bool attention_ok(const Tensor* t, int n, int64_t zigzag) {
  Operands o;
  spa_shards rows;
  const spa_shards* arg;
  if (!differentiable_ok(t, n) || !operands(t, n, o)) return false;
  if (n < 3 && (t[n - 1].dim() != 5 || t[n - 1].size(2) != 4 - n)) return false;
  if (n == 3 && (t[0].dim() != t[1].dim() || t[0].dim() != t[2].dim() || (t[0].dim() == 5 && t[0].sizes() != t[1].sizes()))) return false;
  if (rows_shared(o.q, 2)) return false;
  if (!o.k.same_shape(o.v) || o.q.B != o.k.B || o.q.H != o.k.H || o.q.D != o.k.D || (o.q.D != 32 && o.q.D != 64 && o.q.D != 128)) return false;
  if (!rows_of(o.q, o.k, o.v, zigzag, rows, arg)) return false;
  if (!arg) return true;
  // (what the kernels for rows in shards do not take: 2 GiB and more per (batch, head))
  const int64_t span = (int64_t)(rows.shards - 1) * rows.pitch + o.q.S / rows.shards, esz = t[0].element_size();
  for (const View* v : {&o.q, &o.k, &o.v})
    if (((span - 1) * v->st[2] + v->D) * esz >= 0x7fffffffLL) return false;
  return true;
}

// Saved tensors as the kernels can read them: what a saved-tensor hook hands back need not lie as what was saved.
void to_kernel_rows(variable_list& saved, int n) {
  for (int i = 0; i < n; ++i)
    if (!rows_ok(saved[i])) saved[i] = saved[i].contiguous();
}

void check(int rc) { TORCH_CHECK(rc == SPA_OK, "[spa ", rc, "] ", spa_last_error()); }

// A forward that an entry point refuses, thrown through the autograd node that is being made: the call is one for the Python path.
struct Refused {};
void accepted(bool yes) {
  if (!yes) throw Refused();
}

// Block attention over whole sequences (every ring whose contiguous shards this GPU holds is that: the blocks of the ring
// tile the score matrix).
template <int N>
struct Attention : public torch::autograd::Function<Attention<N>> {
  static variable_list forward_of(const Tensor* t, double scale_or_nan, bool causal, int64_t zigzag) {
    Operands x;
    operands(t, N, x);
    const Tensor& q = t[0];
    void* const stream = current_stream();
    const c10::DeviceGuard guard(q.device());
    Tensor out = N == 1 ? at::empty({x.q.B, x.q.S, x.q.H, x.q.D}, q.options()) : at::empty(q.sizes(), q.options());  // (compact: pitch B * s)
    Tensor lse = empty_f32({x.q.B, x.q.H, x.q.S}, q);
    View o;
    view_of(out, true, o);
    spa_shards rows;
    const spa_shards* shards;
    const float scale = softmax_scale_or_default(scale_or_nan, x.q.D);
    const int mask = causal ? SPA_MASK_CAUSAL : SPA_MASK_NONE, dtype = dtype_code(q.scalar_type());
    rows_of(x.q, x.k, x.v, zigzag, rows, shards);
    if (shards)
      accepted(spa_attention_fwd(x.q.p, x.k.p, x.v.p, o.p, (float*)lse.data_ptr(), x.q.B, x.q.H, x.q.S, x.q.D, x.q.st, x.k.st, x.v.st, o.st, shards,
                                 scale, mask, dtype, stream) == SPA_OK);
    else
      accepted(block_fwd(x.q, x.k, x.v, o, (float*)lse.data_ptr(), nullptr, nullptr, scale, mask, dtype, q, stream) == SPA_OK);
    return {out, lse};
  }
  static variable_list save(AutogradContext* ctx, const Tensor* t, double scale, bool causal, int64_t zigzag) {
    variable_list r = forward_of(t, scale, causal, zigzag);
    variable_list saved(t, t + N);
    saved.insert(saved.end(), r.begin(), r.end());
    ctx->save_for_backward(std::move(saved));
    ctx->saved_data["scale"] = scale;
    ctx->saved_data["causal"] = causal;
    ctx->saved_data["zigzag"] = zigzag;
    ctx->mark_non_differentiable({r[1]});
    ctx->set_materialize_grads(false);  // (the lse has none: a fill of 2 to 5 us a pass)
    return r;
  }
  template <typename... Args>
  static variable_list forward(AutogradContext* ctx, Args... args) {
    return unpack(ctx, std::make_index_sequence<N>{}, args...);
  }
  template <size_t... I, typename... Args>
  static variable_list unpack(AutogradContext* ctx, std::index_sequence<I...>, Args&... args) {
    auto all = std::tie(args...);
    const Tensor t[N] = {std::get<I>(all)...};
    return save(ctx, t, std::get<N>(all), std::get<N + 1>(all), std::get<N + 2>(all));
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    variable_list saved = ctx->get_saved_variables();
    to_kernel_rows(saved, N + 1);
    const double scale_or_nan = ctx->saved_data["scale"].toDouble();
    const bool causal = ctx->saved_data["causal"].toBool();
    Operands x, g;
    const Tensor &q = saved[0], &out = saved[N], &lse = saved[N + 1];
    void* const stream = current_stream();
    const c10::DeviceGuard guard(q.device());
    if (!grads[0].defined()) grads[0] = at::zeros(out.sizes(), out.options());
    View o, d;
    spa_shards rows;
    const spa_shards* shards;
    TORCH_CHECK(operands(saved.data(), N, x) && rows_of(x.q, x.k, x.v, ctx->saved_data["zigzag"].toInt(), rows, shards) &&
                    view_of(out, true, o) && o.same_shape(x.q) && o.pitch == x.q.pitch && lse.is_contiguous(),
                "saved tensors came back in another layout");
    const Tensor dout = rows_ok(grads[0]) && view_of(grads[0], true, d) && d.pitch == o.pitch && !rows_shared(d, 2) ? grads[0] : grads[0].contiguous();
    variable_list back;
    for (int i = 0; i < N; ++i) back.push_back(at::empty(saved[i].sizes(), saved[i].options()));
    operands(back.data(), N, g);
    const Tensor delta = empty_f32(lse.sizes(), lse);
    d = View();
    TORCH_CHECK(view_of(dout, true, d) && o.same_shape(d) && dout.scalar_type() == q.scalar_type(), "bad gradient of the output");
    const int dtype = dtype_code(q.scalar_type());
    check(spa_attention_bwd(x.q.p, x.k.p, x.v.p, o.p, d.p, (const float*)lse.const_data_ptr(), (float*)delta.data_ptr(), g.q.p, g.k.p, g.v.p,
                            x.q.B, x.q.H, x.q.S, x.k.S, x.q.D, x.q.st, x.k.st, x.v.st, o.st, d.st, g.q.st, g.k.st, g.v.st, shards,
                            softmax_scale_or_default(scale_or_nan, x.q.D), causal ? SPA_MASK_CAUSAL : SPA_MASK_NONE, dtype, stream));
    back.resize(N + 3);
    return back;
  }
};

bool wants_grad(const Tensor* t, int n) {
  if (!c10::GradMode::is_enabled()) return false;
  for (int i = 0; i < n; ++i)
    if (t[i].requires_grad()) return true;
  return false;
}

// Calls whose derivative or recording is another mechanism's business: forward-mode tangents, torch.func transforms, a trace.  The
// Python autograd functions refuse or record them.
bool transformed(const Tensor* t, int n) {
  if (torch::jit::tracer::isTracing() || c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode)) return true;
  for (int i = 0; i < n; ++i)
    if (t[i]._fw_grad(0).defined()) return true;
  return false;
}

// Packed batch of sequences of different lengths.
struct VarlenAttention : public torch::autograd::Function<VarlenAttention> {
  static variable_list forward(AutogradContext* ctx, Tensor q, Tensor k, Tensor v, Tensor cu_q, Tensor cu_k, int64_t max_q, int64_t max_k, double scale,
                               bool causal, bool covered, int64_t shards, bool zigzag) {
    Tensor out, lse;
    accepted(varlen_fwd(q, k, v, cu_q, cu_k, max_q, max_k, scale, causal, Tensor(), Tensor(), out, lse, (int)shards, zigzag));
    ctx->save_for_backward({q, k, v, out, lse, cu_q, cu_k});
    ctx->saved_data["max_q"] = max_q;
    ctx->saved_data["max_k"] = max_k;
    ctx->saved_data["scale"] = scale;
    ctx->saved_data["causal"] = causal;
    ctx->saved_data["covered"] = covered;
    ctx->saved_data["shards"] = shards;
    ctx->saved_data["zigzag"] = zigzag;
    ctx->mark_non_differentiable({lse});
    ctx->set_materialize_grads(false);
    return {out, lse};
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    variable_list s = ctx->get_saved_variables();
    to_kernel_rows(s, 4);
    const Tensor &q = s[0], &out = s[3], &lse = s[4];
    void* const stream = current_stream();
    const c10::DeviceGuard guard(q.device());
    if (!grads[0].defined()) grads[0] = at::zeros(out.sizes(), out.options());
    View a, b, c, d, g[3];
    const Tensor dout = rows_ok(grads[0]) && view_thd(grads[0], d) && !rows_shared(d, 1) ? grads[0] : grads[0].contiguous();
    TORCH_CHECK(view_thd(q, a) && view_thd(s[1], b) && view_thd(s[2], c) && lse.is_contiguous() && cu_ok(s[5], q) && cu_ok(s[6], q),
                "saved tensors came back in another layout");
    TORCH_CHECK(view_thd(dout, d) && a.same_shape(d), "bad gradient of the output");
    // the kernels write the rows of the sequences; other rows' gradients are zero
    const bool covered = ctx->saved_data["covered"].toBool();
    variable_list back;
    for (int i = 0; i < 3; ++i) {
      back.push_back(covered ? at::empty(s[i].sizes(), s[i].options()) : at::zeros(s[i].sizes(), s[i].options()));
      view_thd(back[i], g[i]);
    }
    const Tensor delta = empty_f32(lse.sizes(), lse);
    const int dtype = dtype_code(q.scalar_type());
    View o;
    view_thd(out, o);
    const int P = (int)ctx->saved_data["shards"].toInt();
    const spa_shards rows = {P, a.S / P, a.S / P, ctx->saved_data["zigzag"].toBool()};
    check(spa_attention_bwd_varlen(a.p, b.p, c.p, o.p, d.p, (const float*)lse.const_data_ptr(), (float*)delta.data_ptr(), g[0].p, g[1].p, g[2].p,
                                   (const int*)s[5].const_data_ptr(), (const int*)s[6].const_data_ptr(), (int)s[5].numel() - 1, a.H, a.S / P, b.S / P,
                                   (int)ctx->saved_data["max_q"].toInt(), (int)ctx->saved_data["max_k"].toInt(), a.D, a.st, b.st, c.st, o.st, d.st, g[0].st,
                                   g[1].st, g[2].st, P > 1 ? &rows : nullptr, softmax_scale_or_default(ctx->saved_data["scale"].toDouble(), a.D),
                                   ctx->saved_data["causal"].toBool() ? SPA_MASK_CAUSAL : SPA_MASK_NONE, dtype, stream));
    back.resize(12);
    return back;
  }
};

// ---------------------------------------------------------------- Python side
// Arguments come positionally from this package's own functions; a tensor argument that is no tensor (or a number that is no
// number) is a call for the Python path, which raises what it always raised.
bool tensor_arg(PyObject* o, Tensor& t) {
  if (!THPVariable_CheckExact(o)) return false;  // (a subclass has a say in what is done with it)
  t = THPVariable_Unpack(o);
  return true;
}
bool optional_tensor(PyObject* o, Tensor& t) { return o == Py_None || tensor_arg(o, t); }
bool scale_arg(PyObject* o, double& x) {
  if (o == Py_None) {
    x = NAN;
    return true;
  }
  if (!PyFloat_Check(o) && !PyLong_Check(o)) return false;
  x = PyFloat_AsDouble(o);
  if (PyErr_Occurred()) {
    PyErr_Clear();
    return false;
  }
  return std::isfinite(x);
}
bool int_arg(PyObject* o, int64_t& x) {  // (a number past 64 bits is the Python path's)
  if (!PyLong_Check(o)) return false;
  int past = 0;
  x = PyLong_AsLongLongAndOverflow(o, &past);
  return past == 0;
}
bool flag_arg(PyObject* o) {
  const int r = PyObject_IsTrue(o);
  if (r < 0) throw python_error();
  return r != 0;
}
PyObject* pair(const Tensor& out, const Tensor& lse) {
  PyObject* const r = PyTuple_New(2);
  if (!r) throw python_error();
  PyTuple_SET_ITEM(r, 0, THPVariable_Wrap(out));
  PyTuple_SET_ITEM(r, 1, THPVariable_Wrap(lse));
  return r;
}

// flash_fwd(q, k, v, scale, causal, bshd, q_scale, k_scale, v_scale, out_dtype_code)
PyObject* py_flash_fwd(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Tensor q, k, v, qs, ks, vs, out, lse;
  double scale;
  int64_t out_dtype;
  if (n != 10 || !tensor_arg(a[0], q) || !tensor_arg(a[1], k) || !tensor_arg(a[2], v) || !scale_arg(a[3], scale) || !optional_tensor(a[6], qs) ||
      !optional_tensor(a[7], ks) || !optional_tensor(a[8], vs) || !int_arg(a[9], out_dtype))
    Py_RETURN_NONE;
  const bool causal = flag_arg(a[4]), bshd = flag_arg(a[5]);
  bool done;
  {
    pybind11::gil_scoped_release no_gil;
    done = flash_fwd(q, k, v, scale, causal, bshd, qs, ks, vs, (int)out_dtype, out, lse);
  }
  if (!done) Py_RETURN_NONE;
  return pair(out, lse);
  END_HANDLE_TH_ERRORS
}

// varlen_fwd(q, k, v, cu_q, cu_k, max_q, max_k, scale, causal, k_scale, v_scale)
PyObject* py_varlen_fwd(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Tensor q, k, v, cq, ck, ks, vs, out, lse;
  double scale;
  int64_t mq, mk;
  if (n != 11 || !tensor_arg(a[0], q) || !tensor_arg(a[1], k) || !tensor_arg(a[2], v) || !tensor_arg(a[3], cq) || !tensor_arg(a[4], ck) ||
      !int_arg(a[5], mq) || !int_arg(a[6], mk) || !scale_arg(a[7], scale) || !optional_tensor(a[9], ks) || !optional_tensor(a[10], vs))
    Py_RETURN_NONE;
  const bool causal = flag_arg(a[8]);
  bool done = false;
  if (mq > 0 && mk > 0 && mq <= 0x7fffffffLL && mk <= 0x7fffffffLL) {
    pybind11::gil_scoped_release no_gil;
    done = varlen_fwd(q, k, v, cq, ck, mq, mk, scale, causal, ks, vs, out, lse);
  }
  if (!done) Py_RETURN_NONE;
  return pair(out, lse);
  END_HANDLE_TH_ERRORS
}

// attention(tensors..., scale, causal, zigzag shards or 0): q, k, v | q, kv | qkv
template <int N, size_t... I>
PyObject* attention(PyObject* const* a, std::index_sequence<I...>) {
  HANDLE_TH_ERRORS
  Tensor t[N];
  double scale;
  for (int i = 0; i < N; ++i)
    if (!tensor_arg(a[i], t[i])) Py_RETURN_NONE;
  int64_t zigzag;
  if (!scale_arg(a[N], scale) || !int_arg(a[N + 2], zigzag)) Py_RETURN_NONE;
  if (zigzag < 0 || zigzag > 0x3fffffffLL || transformed(t, N) || !attention_ok(t, N, zigzag)) Py_RETURN_NONE;
  const bool causal = flag_arg(a[N + 1]);
  variable_list r;
  try {
    pybind11::gil_scoped_release no_gil;
    r = wants_grad(t, N) ? Attention<N>::apply(t[I]..., scale, causal, zigzag) : Attention<N>::forward_of(t, scale, causal, zigzag);
  } catch (const Refused&) {
    Py_RETURN_NONE;
  }
  return pair(r[0], r[1]);
  END_HANDLE_TH_ERRORS
}
PyObject* py_attention(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n == 6) return attention<3>(a, std::make_index_sequence<3>{});
  if (n == 5) return attention<2>(a, std::make_index_sequence<2>{});
  if (n == 4) return attention<1>(a, std::make_index_sequence<1>{});
  Py_RETURN_NONE;
}

bool varlen_shards_ok(const View& q, const View& k, const View& v, int64_t longest, int64_t shards, int64_t esz) {
  if (shards == 1) return true;
  if (q.S % shards != 0 || k.S != q.S || k.st[1] != v.st[1]) return false;
  for (const View* x : {&q, &k, &v})
    if ((((shards - 1) * (q.S / shards) + longest - 1) * x->st[1] + x->D) * esz >= 0x7fffffffLL) return false;
  return true;
}

// varlen_attention(q, k, v, cu_q, cu_k, max_q, max_k, scale, causal, covered, shards, zigzag)
PyObject* py_varlen_attention(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Tensor t[5];
  double scale;
  int64_t mq, mk, shards;
  if (n != 12 || !int_arg(a[10], shards)) Py_RETURN_NONE;
  for (int i = 0; i < 5; ++i)
    if (!tensor_arg(a[i], t[i])) Py_RETURN_NONE;
  if (!int_arg(a[5], mq) || !int_arg(a[6], mk) || !scale_arg(a[7], scale)) Py_RETURN_NONE;
  const bool causal = flag_arg(a[8]), covered = flag_arg(a[9]), zigzag = flag_arg(a[11]);
  if (transformed(t, 3) || !differentiable_ok(t, 3) || !cu_ok(t[3], t[0]) || !cu_ok(t[4], t[0]) || mq <= 0 || mk <= 0 || mq > 0x7fffffffLL || mk > 0x7fffffffLL ||
      shards < 1 || shards > 0xffffLL)
    Py_RETURN_NONE;
  variable_list r(2);
  try {
    pybind11::gil_scoped_release no_gil;
    if (wants_grad(t, 3)) {
      View x, y, z;
      if (!view_thd(t[0], x) || !view_thd(t[1], y) || !view_thd(t[2], z) || !y.same_shape(z) || rows_shared(x, 1) || x.H != y.H || x.D != y.D || mq > x.S || mk > y.S ||
          t[3].numel() != t[4].numel() || !varlen_shards_ok(x, y, z, mq, shards, t[0].element_size()) || (x.D != 32 && x.D != 64 && x.D != 128))
        r.clear();
      else
        r = VarlenAttention::apply(t[0], t[1], t[2], t[3], t[4], mq, mk, scale, causal, covered, shards, zigzag);
    } else if (!varlen_fwd(t[0], t[1], t[2], t[3], t[4], mq, mk, scale, causal, Tensor(), Tensor(), r[0], r[1], (int)shards, zigzag)) {
      r.clear();
    }
  } catch (const Refused&) {
    Py_RETURN_NONE;
  }
  if (r.empty()) Py_RETURN_NONE;
  return pair(r[0], r[1]);
  END_HANDLE_TH_ERRORS
}

// merge(out_acc [B,S,H,D] fp32, lse_acc [B,S,H,1] over a contiguous [B,H,S] buffer, blk_out [B,H,S,D] or [B,S,H,D], blk_lse [B,H,S]):
// True when the kernel was enqueued.  merge(None, None, blk_out [B,H,S,D], blk_lse): new accumulators (out, lse) holding the block.
PyObject* py_merge(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Tensor acc, lse, blk, bl;
  if (n != 4 || !optional_tensor(a[0], acc) || !optional_tensor(a[1], lse) || !tensor_arg(a[2], blk) || !tensor_arg(a[3], bl)) Py_RETURN_NONE;
  const bool first = !acc.defined();
  const int dtype = dtype_code(blk.scalar_type());
  View x, y;
  if (!blk.is_cuda() || !on_device(bl, blk) || dtype < 0 || blk.dim() != 4 || bl.dim() != 3 || bl.scalar_type() != at::kFloat || !bl.is_contiguous() ||
      !rows_ok(blk) || first != !lse.defined())
    Py_RETURN_NONE;
  if (!first) {
    // (a block whose dims 1, 2 are those of the accumulator swapped is in operator layout)
    const bool bhsd = acc.dim() == 4 && blk.size(1) != acc.size(1) && blk.size(2) == acc.size(1);
    if (acc.dim() != 4 || lse.dim() != 4 || !on_device(acc, blk) || !on_device(lse, blk) || acc.scalar_type() != at::kFloat ||
        lse.scalar_type() != at::kFloat || !rows_ok(acc) || !view_of(acc, true, x) || !view_of(blk, !bhsd, y) || !x.same_shape(y) || lse.size(0) != x.B ||
        lse.size(1) != x.S || lse.size(2) != x.H || lse.size(3) != 1 || (x.B > 1 && lse.stride(0) != (int64_t)x.H * x.S) ||
        (x.S > 1 && lse.stride(1) != 1) || (x.H > 1 && lse.stride(2) != x.S))
      Py_RETURN_NONE;
  } else if (!view_of(blk, false, y)) {
    Py_RETURN_NONE;
  }
  if (bl.size(0) != y.B || bl.size(1) != y.H || bl.size(2) != y.S) Py_RETURN_NONE;
  int rc;
  {
    pybind11::gil_scoped_release no_gil;
    void* const stream = current_stream();
    const c10::DeviceGuard guard(blk.device());
    if (first) {
      acc = empty_f32({y.B, y.S, y.H, y.D}, blk);
      lse = empty_f32({y.B, y.H, y.S}, blk);
      view_of(acc, true, x);
    }
    rc = spa_merge((float*)x.p, (float*)lse.data_ptr(), y.p, (const float*)bl.const_data_ptr(), x.B, x.H, x.S, x.D, x.st, y.st, dtype, first, stream);
    if (first) lse = lse.transpose(1, 2).unsqueeze(-1);
  }
  if (rc != SPA_OK) Py_RETURN_NONE;
  if (first) return pair(acc, lse);
  Py_RETURN_TRUE;
  END_HANDLE_TH_ERRORS
}

#define FAST(name, fn) {name, (PyCFunction)(void (*)(void))fn, METH_FASTCALL, nullptr}
PyMethodDef methods[] = {FAST("flash_fwd", py_flash_fwd), FAST("varlen_fwd", py_varlen_fwd), FAST("attention", py_attention),
                         FAST("varlen_attention", py_varlen_attention), FAST("merge", py_merge), {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_native", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__native(void) { return PyModule_Create(&module); }
