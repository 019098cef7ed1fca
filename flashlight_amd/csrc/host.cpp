// Native host path of the front ends: what ops.dispatch does for an ordinary call, without the interpreter.
//
// A short call is bound by its host side: through the ctypes binding it spent 12 us on filling the parameter struct field
// by field, on a differentiable call 100 us in the custom-operator layers, against 5 to 20 us on the GPU.  `forward` here
// takes the call when it is of the plain kind (dense 16-bit tensors on the current device, compiled head dims, shapes and
// strides the kernels address as they are, no tracer, transform or dispatch mode at work), allocates the result and
// launches; with a gradient asked for it hangs a node on the result whose backward launches the gradient kernels.  For
// anything else, wrong arguments included, it returns None and the Python code does what it always did: the conversions,
// the compositions, the error messages.  It keeps no state between calls beyond the addresses of the C ABI's functions.
#define PY_SSIZE_T_CLEAN
#include <ATen/ATen.h>
#include <ATen/TensorUtils.h>
#include <ATen/core/LegacyTypeDispatch.h>
#include <Python.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/functions/basic_ops.h>
#include <torch/csrc/autograd/python_variable.h>

#include <algorithm>
#include <cmath>

#include "flashlight_amd.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

struct Api {
  int (*fwd)(const fl_attn_params*, void*) = nullptr;
  int (*bwd)(const fl_attn_bwd_params*, void*, uint64_t, void*) = nullptr;
  uint64_t (*workspace)(const fl_attn_params*) = nullptr;
  uint64_t (*bwd_workspace)(const fl_attn_params*) = nullptr;
  uint64_t (*bwd_split_bytes)(const fl_attn_params*) = nullptr;
  int (*rows_plan)(const fl_attn_params*, uint64_t*) = nullptr;
  uint64_t (*shared_bias_bwd_bytes)(const fl_attn_params*) = nullptr;
  int (*shared_bias_bwd)(const fl_attn_shared_bias_bwd_params*, void*) = nullptr;
  const char* (*last_error)(void) = nullptr;
  int (*fwd_ungated)(const fl_attn_params*, void*, void*) = nullptr;
} g_api;
constexpr int kApiFunctions = 10;

// One call's arguments.  The tensors are the caller's; `doc`, `bias` and `gate` may be undefined.
struct Call {
  Tensor q, k, v, doc, bias[2], gate;
  int64_t bias_div[2] = {1, 1};
  double scale = 0;
  int64_t mask_kind = 0, window = 0, prefix = 0, alibi_heads = 0;
  double softcap = 0, lambda = 0;
  bool diff = false, seq_major = false;
  bool wants_grad = false;
  // Calls of the Evoformer front end: the leading axes of its [*, S, H, D] operands, of which q, k, v and gate here are the
  // [prod(*), H, S, D] views and the biases the kernels' 4-D form.  Its gradients hang on the operands as the caller passed them,
  // in one node (as views of their own the operands and the result cost a dozen nodes, 80 of 110 us of a short backward pass).
  std::vector<int64_t> lead;
  Tensor given_q, given_k, given_v, given_bias[2], given_gate;  // with `lead`: the operands as the caller passed them
};

// [*, S, H, D] -> its [prod(*), H, S, D] view; undefined where the leading axes do not merge.
Tensor heads_first(const Tensor& t, size_t lead) {
  const auto sizes = t.sizes();
  int64_t rows = 1;
  for (size_t i = 0; i < lead; ++i) rows *= sizes[i];
  const int64_t merged[4] = {rows, sizes[lead], sizes[lead + 1], sizes[lead + 2]};
  const auto st = at::detail::computeStride(sizes, t.strides(), at::IntArrayRef(merged, 4));
  if (!st) return Tensor();
  const at::AutoDispatchBelowADInplaceOrView plainly;  // (a view for the kernels' use, which autograd does not see)
  const int64_t size4[4] = {rows, merged[2], merged[1], merged[3]}, stride4[4] = {(*st)[0], (*st)[2], (*st)[1], (*st)[3]};
  return t.as_strided(at::IntArrayRef(size4, 4), at::IntArrayRef(stride4, 4));
}

// A bias broadcastable to [*, H, S, S] in the kernels' form, [Bb, H or 1, S or 1, S] with batch entry b reading Bb index
// b / div: as evoformer._as_kernel_bias, undefined where that would copy.
Tensor kernel_bias(const Tensor& b, const std::vector<int64_t>& lead, int64_t H, int64_t S, int64_t& div) {
  const int64_t nl = (int64_t)lead.size(), missing = nl + 3 - b.dim();
  if (missing < 0 || b.dim() == 0) return Tensor();
  const auto size = [&](int64_t i) { return i < missing ? 1 : b.size(i - missing); };
  if ((size(nl) != H && size(nl) != 1) || (size(nl + 1) != S && size(nl + 1) != 1) || size(nl + 2) != S) return Tensor();
  int64_t split = nl, nb = 1;
  while (split > 0 && size(split - 1) == 1) --split;
  for (int64_t i = 0; i < split; ++i) {
    if (size(i) != lead[i]) return Tensor();
    nb *= lead[i];
  }
  div = 1;
  for (int64_t i = split; i < nl; ++i) div *= lead[i];
  const int64_t shape[4] = {nb, size(nl), size(nl + 1), S};
  const auto st = at::detail::computeStride(b.sizes(), b.strides(), at::IntArrayRef(shape, 4));
  const at::AutoDispatchBelowADInplaceOrView plainly;
  return st ? b.as_strided(at::IntArrayRef(shape, 4), *st) : Tensor();
}

// dense, dim-contiguous rows in 16-byte pieces: what the kernels address as it lies
bool addressable(const Tensor& t) {
  if (t.stride(3) != 1 || (reinterpret_cast<uintptr_t>(t.const_data_ptr()) & 15)) return false;
  for (int i = 0; i < 3; ++i)
    if (t.stride(i) % 8 || t.stride(i) < 0) return false;
  return true;
}

// an ordinary GPU tensor: no transform's wrapper, no lazy conjugate or negation, nothing that dispatches to Python
bool plain(const Tensor& t) {
  using c10::DispatchKey;
  static const c10::DispatchKeySet odd({DispatchKey::FuncTorchBatched, DispatchKey::FuncTorchGradWrapper, DispatchKey::BatchedNestedTensor,
                                        DispatchKey::Python, DispatchKey::PythonTLSSnapshot, DispatchKey::Functionalize,
                                        DispatchKey::Conjugate, DispatchKey::Negative, DispatchKey::ZeroTensor,
                                        DispatchKey::FuncTorchVmapMode, DispatchKey::PreDispatch});
  return t.defined() && t.is_cuda() && t.layout() == at::kStrided && !t.key_set().has_any(odd);
}

// a dispatch mode, a functional transform or a tracer is at work on this thread
bool mode_active() {
  using c10::DispatchKey;
  static const c10::DispatchKeySet modes({DispatchKey::FuncTorchDynamicLayerFrontMode, DispatchKey::FuncTorchDynamicLayerBackMode,
                                          DispatchKey::FuncTorchVmapMode, DispatchKey::Python, DispatchKey::Functionalize, DispatchKey::PreDispatch});
  return c10::impl::TorchDispatchModeTLS::any_modes_set() || c10::impl::tls_local_dispatch_key_set().included_.has_any(modes);
}

void set_strides(int64_t* to, const Tensor& t) {
  for (int i = 0; i < 4; ++i) to[i] = t.stride(i);
}

int element_type(const Tensor& t) {
  return t.scalar_type() == at::kBFloat16 ? FL_BF16 : t.scalar_type() == at::kHalf ? FL_F16 : -1;
}

// Fills what the forward and the backward share.
void fill(const Call& c, fl_attn_params& p) {
  const Tensor &q = c.q, &k = c.k, &v = c.v;
  const int two = c.diff ? 2 : 1;
  p.dtype = element_type(q);
  p.q = q.const_data_ptr();
  p.k = k.const_data_ptr();
  p.v = v.const_data_ptr();
  set_strides(p.q_strides, q);
  set_strides(p.k_strides, k);
  set_strides(p.v_strides, v);
  p.B = (int32_t)q.size(0);
  p.Hq = (int32_t)(q.size(1) / two);
  p.Hkv = (int32_t)(k.size(1) / two);
  p.Lq = (int32_t)q.size(2);
  p.Lk = (int32_t)k.size(2);
  p.Dqk = (int32_t)q.size(3);
  p.Dv = (int32_t)v.size(3);
  p.scale = (float)c.scale;
  p.mask_kind = (int32_t)c.mask_kind;
  p.window = (int32_t)c.window;
  p.prefix = (int32_t)c.prefix;
  p.alibi_heads = (int32_t)c.alibi_heads;
  p.softcap = (float)c.softcap;
  p.diff = c.diff;
  p.lambda = (float)c.lambda;
  if (c.doc.defined()) {
    p.doc_ids = c.doc.const_data_ptr<int64_t>();
    p.doc_stride = c.doc.size(0) == p.B && p.B > 1 ? c.doc.stride(0) : 0;
  }
  for (int i = 0; i < 2; ++i) {
    const Tensor& b = c.bias[i];
    if (!b.defined()) continue;
    const int64_t want[4] = {p.B / c.bias_div[i], p.Hq, p.Lq, p.Lk};
    p.bias[i] = b.const_data_ptr();
    p.bias_dtype[i] = b.scalar_type() == at::kFloat ? FL_F32 : p.dtype;
    p.bias_batch_div[i] = (int32_t)c.bias_div[i];
    for (int ax = 0; ax < 4; ++ax) p.bias_strides[i][ax] = b.size(ax) == want[ax] && want[ax] != 1 ? b.stride(ax) : 0;
  }
  if (c.gate.defined()) {
    p.gate = c.gate.const_data_ptr();
    set_strides(p.gate_strides, c.gate);
  }
}

void* current_stream() { return c10::hip::getCurrentHIPStream().stream(); }

// Into how many chunks the front end cuts the keys of an unmasked call whose rows are independent (ops._split_over_keys: the
// chunks run as heads or batch entries of one launch of the tile kernel, with results in fp32, and a second launch merges
// them); 0: it does not.  `groups` counts the tile kernel's workgroups without chunks.
int64_t key_chunks(const fl_attn_params& p, const Tensor& k, const Tensor& v, int64_t groups) {
  if (groups >= 256 || p.Lk < 4096) return 0;
  // one batch entry with dense rows: chunks of a multiple of 8 keys as batch entries, the rest is one more; otherwise the
  // caches have to be one block, and the chunks divide them into heads
  const bool one = p.B == 1 && p.k_strides[2] == p.Dqk && p.v_strides[2] == p.Dv;
  if (!one && !(k.is_contiguous() && v.is_contiguous())) return 0;
  // One round of workgroups, two per compute unit; where half as many chunks would leave an eighth of that idle, up to two
  // rounds.  (More only make partial results: 8 heads, 256 queries, 65536 keys, head dim 128: 107 us with 2048 workgroups,
  // 106 with 1024, 87 with 512; 128 heads' tiles of 8192 keys 125, 96, 89; 192 of 16384 keys 238, 227, 240.)
  for (int64_t c = 64; c > 1; c /= 2)
    if ((groups * c <= 512 || (groups * c <= 1024 && groups * c / 2 < 448)) &&
        (one ? p.Lk / c / 8 * 8 >= 512 : p.Lk % (8 * c) == 0 && p.Lk / c >= 512))
      return c;
  return 0;
}

// Whether those chunks are the better way where the few-rows kernel would take the call (fl_attn_rows_plan).  It reads K and V
// for every 16 rows, from L2: 256 workgroups together 150 keys per microsecond each at head dim 64, 100 at 128, and 8 us for a
// start and a merge where they work on chunks.  The tile kernel reads them once for 128 rows: 64 and 50 keys per microsecond in
// a workgroup of its own compute unit, 28 and 25 with two on each, and 9 us.  Estimates in microseconds, from 50 shapes of 33 to
// 4096 rows over 4096 to 131072 keys; with up to 32 rows the keys are read once there, too.
// (few-rows kernel without chunks -> this rule: 32 heads over 8, 16 queries, 32768 keys, head dim 128: 284 -> 38 us; 8 heads, 64
// queries, 65536 keys: 563 -> 57; 2 heads, 48 queries, 32768 keys: 285 -> 19; 8 heads, 128 queries, 4096 keys, 64: 26 -> 15.)
bool chunks_beat_rows_kernel(const fl_attn_params& p, int64_t groups, int64_t chunks) {
  const int64_t units = (int64_t)p.B * p.Hkv, rows = (int64_t)(p.Hq / p.Hkv) * p.Lq;
  if (rows <= 32) return false;
  const int64_t base = std::min<int64_t>(256, units * ((rows + 15) / 16)), own = 256 / base;
  const bool narrow = p.Dqk <= 64;
  const double by_rows = (double)p.Lk / own / (narrow ? 150 : 100) + (own > 1 ? 8 : 0);
  const double by_chunks = 9 + std::max((double)p.Lk / chunks / (narrow ? 64 : 50), (double)groups * p.Lk / 512 / (narrow ? 28 : 25));
  return by_chunks < by_rows;
}

// Launches the forward of `c` into a fresh tensor; an undefined tensor if the C ABI refuses (the Python path then says why).
// `lse`: when given, receives the row statistics; `ungated` the result before the gate.
Tensor launch_forward(const Call& c, Tensor* lse, Tensor* ungated = nullptr) {
  fl_attn_params p = {};
  fill(c, p);
  Tensor q = c.q, out;
  const auto opt = q.options().requires_grad(false);
  const int64_t row = (int64_t)p.Hq * p.Dv;  // (seq_major: memory order [batch, position, head, dim])
  if (c.seq_major) out = at::empty_strided({p.B, p.Hq, p.Lq, p.Dv}, {row * p.Lq, p.Dv, row, 1}, opt);
  else out = at::empty({p.B, p.Hq, p.Lq, p.Dv}, opt);
  p.o = out.data_ptr();
  set_strides(p.o_strides, out);
  if (lse) {
    *lse = at::empty({p.B, p.Hq, p.Lq}, opt.dtype(at::kFloat));
    p.lse = lse->data_ptr<float>();
  }
  if (ungated) {
    *ungated = at::empty_strided(out.sizes(), out.strides(), opt);
    return g_api.fwd_ungated(&p, ungated->data_ptr(), current_stream()) == 0 ? out : Tensor();
  }
  uint64_t bytes = 0;
  Tensor ws;
  if (c.doc.defined()) {
    bytes = g_api.workspace(&p);
  } else {
    const bool rows_kernel = g_api.rows_plan(&p, &bytes);
    const bool rows_independent = c.mask_kind == FL_MASK_NONE && !p.gate && !p.diff && !p.alibi_heads && !lse && !c.seq_major &&
                                  (!p.bias[0] || (p.bias_strides[0][1] == 0 && p.bias_strides[0][2] == 0)) &&
                                  (!p.bias[1] || (p.bias_strides[1][1] == 0 && p.bias_strides[1][2] == 0));
    if (rows_independent) {
      // (without a mask the G query heads of a key / value head may as well be G times as many rows of one head: one
      // workgroup then reads the keys for all of them)
      const int64_t group = p.Hq / p.Hkv;
      const bool pack = group > 1 && group * p.Lq <= 128 && q.is_contiguous();
      const int64_t groups = pack ? (int64_t)p.B * p.Hkv : (int64_t)p.B * p.Hq * ((p.Lq + 127) / 128);
      // few workgroups against many keys: the Python path cuts the keys into chunks
      const auto whole_row = [&](const Tensor& b) { return !b.defined() || (b.is_contiguous() && b.size(3) == p.Lk); };
      if (whole_row(c.bias[0]) && whole_row(c.bias[1])) {
        const int64_t chunks = key_chunks(p, c.k, c.v, groups);
        if (chunks && (!rows_kernel || chunks_beat_rows_kernel(p, groups, chunks))) return Tensor();
      }
      if (pack && !rows_kernel) {
        p.Hq = p.Hkv;
        p.Lq = (int32_t)(group * p.Lq);
        p.q_strides[1] = p.Lq * q.stride(2);
        p.o_strides[1] = p.Lq * out.stride(2);
      }
    }
  }
  if (bytes) {
    ws = at::empty({(int64_t)bytes}, opt.dtype(at::kByte));
    p.workspace = ws.data_ptr();
    p.workspace_bytes = bytes;
    if (!c.doc.defined()) p.flags = FL_FLAG_SCRATCH;
  }
  return g_api.fwd(&p, current_stream()) == 0 ? out : Tensor();
}

struct Refused {};  // the C ABI does not take the call: the Python path then says why

// Fresh memory in the operand's own order where that is dense, contiguous otherwise.
Tensor empty_for_gradient(const Tensor& t) {
  const auto opt = t.options().requires_grad(false);
  return t.is_non_overlapping_and_dense() ? at::empty_strided(t.sizes(), t.strides(), opt) : at::empty(t.sizes(), opt);
}

// The call's scalars, kept with the node between forward and backward.
void keep_scalars(AutogradContext* ctx, const Call& c) {
  ctx->saved_data["i"] = std::vector<int64_t>{c.mask_kind, c.window, c.prefix, c.alibi_heads, c.bias_div[0], c.bias_div[1]};
  ctx->saved_data["f"] = std::vector<double>{c.scale, c.softcap};
}
void take_scalars(AutogradContext* ctx, Call& c) {
  const auto ints = ctx->saved_data["i"].toIntVector();
  const auto floats = ctx->saved_data["f"].toDoubleVector();
  c.mask_kind = ints[0];
  c.window = ints[1];
  c.prefix = ints[2];
  c.alibi_heads = ints[3];
  c.bias_div[0] = ints[4];
  c.bias_div[1] = ints[5];
  c.scale = floats[0];
  c.softcap = floats[1];
}

// Under create_graph the gradients say that they have none of their own, instead of looking like constants.
void once_differentiable(variable_list& grads, bool grad_mode) {
  if (!grad_mode) return;
  variable_list some;
  for (auto& t : grads)
    if (t.defined()) some.push_back(t.detach().requires_grad_(true));
  some = (*std::make_shared<torch::autograd::DelayedError>("flashlight_amd: the gradients are not differentiable a second time",
                                                           (int64_t)some.size()))(std::move(some));
  size_t i = 0;
  for (auto& t : grads)
    if (t.defined()) t = some[i++];
}

Tensor prepare_dout(const Tensor& grad, const Tensor& like) {
  Tensor d = grad.to(like.scalar_type());
  return addressable(d) ? d : d.contiguous();
}

struct Attention : torch::autograd::Function<Attention> {
  static Tensor forward(AutogradContext* ctx, const Tensor& q, const Tensor& k, const Tensor& v, const Call& c) {
    Tensor lse;
    Tensor out = launch_forward(c, &lse);
    if (!out.defined()) throw Refused();
    ctx->save_for_backward({q, k, v, out, lse});
    keep_scalars(ctx, c);
    if (c.doc.defined()) ctx->saved_data["doc"] = c.doc;
    return out;
  }

  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const auto saved = ctx->get_saved_variables();
    Call c;
    c.q = saved[0];
    c.k = saved[1];
    c.v = saved[2];
    take_scalars(ctx, c);
    if (ctx->saved_data.count("doc")) c.doc = ctx->saved_data["doc"].toTensor();
    const Tensor &out = saved[3], &lse = saved[4];
    variable_list result(4);
    if (!grads[0].defined()) return result;
    const bool grad_mode = at::GradMode::is_enabled();
    {
      at::AutoGradMode off(false);
      const Tensor dout = prepare_dout(grads[0], c.q);
      fl_attn_bwd_params b = {};
      fill(c, b.fwd);
      b.fwd.o = const_cast<void*>(out.const_data_ptr());
      set_strides(b.fwd.o_strides, out);
      b.fwd.lse = const_cast<float*>(lse.const_data_ptr<float>());
      Tensor dq = empty_for_gradient(c.q), dk = empty_for_gradient(c.k), dv = empty_for_gradient(c.v);
      b.dout = dout.const_data_ptr();
      b.dq = dq.data_ptr();
      b.dk = dk.data_ptr();
      b.dv = dv.data_ptr();
      set_strides(b.dout_strides, dout);
      set_strides(b.dq_strides, dq);
      set_strides(b.dk_strides, dk);
      set_strides(b.dv_strides, dv);
      // scratch in one block: the row sums, the document table, partial sums
      const auto up = [](uint64_t bytes) { return (bytes + 255) / 256 * 256; };
      const uint64_t table = g_api.bwd_workspace(&b.fwd), split = g_api.bwd_split_bytes(&b.fwd), sums = up(4 * (uint64_t)lse.numel());
      Tensor scratch = at::empty({(int64_t)(sums + up(table) + split)}, lse.options().dtype(at::kByte));
      unsigned char* const at = scratch.data_ptr<unsigned char>();
      b.delta = reinterpret_cast<float*>(at);
      if (table) {
        b.fwd.workspace = at + sums;
        b.fwd.workspace_bytes = table;
      }
      const int rc = g_api.bwd(&b, split ? at + sums + up(table) : nullptr, split, current_stream());
      TORCH_CHECK(rc == 0, "flashlight_amd error ", rc, ": ", g_api.last_error());
      result[0] = dq;
      result[1] = dk;
      result[2] = dv;
    }
    once_differentiable(result, grad_mode);
    return result;
  }
};

// The result of an Evoformer call as its caller sees it, [*, S, H, D], from the kernels' sequence-major 4-D one.
Tensor with_lead(const Tensor& out, const std::vector<int64_t>& lead) {
  std::vector<int64_t> sizes(lead);
  sizes.insert(sizes.end(), {out.size(2), out.size(1), out.size(3)});
  std::vector<int64_t> strides(sizes.size());
  int64_t s = 1;
  for (size_t i = sizes.size(); i-- > 0; s *= sizes[i]) strides[i] = s;
  const at::AutoDispatchBelowADInplaceOrView plainly;  // (the caller's tensor, not a view of one it never sees)
  return out.as_strided(sizes, strides);
}

// Calls with a bias shared by batch entries, and optionally the gate (fl_attn_shared_bias_bwd).  bias[0] is the shared
// operand here, bias[1] the row per batch entry, which takes no gradient.  The tensors are the caller's, `c` holds the kernels'
// views of them.
struct SharedBias : torch::autograd::Function<SharedBias> {
  static Tensor forward(AutogradContext* ctx, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& bias,
                        const std::optional<Tensor>& row, const std::optional<Tensor>& gate, const Call& c) {
    Tensor lse, ungated;
    Tensor out = launch_forward(c, &lse, gate ? &ungated : nullptr);
    if (!out.defined()) throw Refused();
    if (!c.lead.empty()) out = with_lead(out, c.lead);
    // (the gradients are formed from the attention's own result: a nearly closed gate leaves the gated one few bits)
    ctx->save_for_backward({q, k, v, bias, row.value_or(Tensor()), gate.value_or(Tensor()), gate ? ungated : out, lse});
    keep_scalars(ctx, c);
    ctx->saved_data["lead"] = c.lead;
    return out;
  }

  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const auto saved = ctx->get_saved_variables();
    variable_list result(7);
    if (!grads[0].defined()) return result;
    const bool grad_mode = at::GradMode::is_enabled();
    {
      at::AutoDispatchBelowAutograd below;
      Call c;
      take_scalars(ctx, c);
      c.lead = ctx->saved_data["lead"].toIntVector();
      const size_t nl = c.lead.size();
      const auto view = [&](const Tensor& t) {
        if (!nl || !t.defined()) return t;
        const Tensor x = heads_first(t, nl);
        return x.defined() ? x : heads_first(t.contiguous(), nl);
      };
      c.q = view(saved[0]);
      c.k = view(saved[1]);
      c.v = view(saved[2]);
      c.gate = view(saved[5]);
      for (int i = 0; i < 2; ++i) {
        int64_t div;
        c.bias[i] = nl && saved[3 + i].defined() ? kernel_bias(saved[3 + i], c.lead, c.q.size(1), c.q.size(2), div) : saved[3 + i];
      }
      const Tensor out = c.gate.defined() ? saved[6] : view(saved[6]);
      const Tensor& lse = saved[7];
      Tensor dout = view(grads[0].to(c.q.scalar_type()));
      if (!addressable(dout) || dout.stride(2) >= 1 << 20) {  // (the kernels' offsets inside one (batch entry, head))
        dout = nl ? dout.transpose(1, 2).contiguous().transpose(1, 2) : dout.contiguous();
      }
      fl_attn_shared_bias_bwd_params b = {};
      fill(c, b.fwd);
      b.fwd.o = const_cast<void*>(out.const_data_ptr());
      set_strides(b.fwd.o_strides, out);
      b.fwd.lse = const_cast<float*>(lse.const_data_ptr<float>());
      if (c.gate.defined()) b.fwd.flags = FL_FLAG_UNGATED;
      // the gradients lie as the caller's operands do
      const auto gradient = [&](Tensor& to, const Tensor& like, int64_t* strides) -> void* {
        to = empty_for_gradient(like);
        set_strides(strides, view(to));
        return to.data_ptr();
      };
      b.dout = dout.const_data_ptr();
      set_strides(b.dout_strides, dout);
      b.dq = gradient(result[0], saved[0], b.dq_strides);
      b.dk = gradient(result[1], saved[1], b.dk_strides);
      b.dv = gradient(result[2], saved[2], b.dv_strides);
      if (c.gate.defined()) b.dgate = gradient(result[5], saved[5], b.dgate_strides);
      if (ctx->needs_input_grad(3)) {
        TORCH_CHECK(c.bias[0].size(0) == b.fwd.B / c.bias_div[0], "one gradient per ", c.bias_div[0], " batch entries, ",
                    c.bias[0].size(0), " operands");
        result[3] = at::empty(saved[3].sizes(), saved[3].options());
        b.dbias = result[3].data_ptr();
      }
      const uint64_t bytes = g_api.shared_bias_bwd_bytes(&b.fwd);
      Tensor ws = at::empty({(int64_t)bytes}, lse.options().dtype(at::kByte));
      b.workspace = ws.data_ptr();
      b.workspace_bytes = bytes;
      const int rc = g_api.shared_bias_bwd(&b, current_stream());
      TORCH_CHECK(rc == 0, "flashlight_amd error ", rc, ": ", g_api.last_error());
    }
    once_differentiable(result, grad_mode);
    return result;
  }
};

std::optional<Tensor> given(const Tensor& t) { return t.defined() ? std::optional<Tensor>(t) : std::nullopt; }

// ---- Python boundary -----------------------------------------------------------------------------------------------------

bool take_tensor(PyObject* o, Tensor& t) {
  if ((PyObject*)Py_TYPE(o) != THPVariableClass) return false;  // (subclasses and Parameters go the Python way)
  t = THPVariable_Unpack(o);
  return plain(t);
}

// Other Python threads run while this one allocates and launches (the allocator may go to the driver, the launch queue may
// be full).
struct WithoutGil {
  PyThreadState* state = PyEval_SaveThread();
  ~WithoutGil() { PyEval_RestoreThread(state); }
};

// The call itself; an undefined tensor if the C ABI does not take it.
Tensor attend(const Call& c) {
  const WithoutGil no_gil;
  if (!c.wants_grad) return launch_forward(c, nullptr);
  try {
    if (!c.lead.empty())
      return SharedBias::apply(c.given_q, c.given_k, c.given_v, c.given_bias[0], given(c.given_bias[1]), given(c.given_gate), c);
    return c.bias[0].defined() ? SharedBias::apply(c.q, c.k, c.v, c.bias[0], given(c.bias[1]), given(c.gate), c)
                               : Attention::apply(c.q, c.k, c.v, c);
  } catch (const Refused&) {
    return Tensor();
  }
}

// ---- what the native path takes ------------------------------------------------------------------------------------------

bool operands_fit(const Call& c) {
  const Tensor &q = c.q, &k = c.k, &v = c.v;
  if (q.dim() != 4 || k.dim() != 4 || v.dim() != 4 || element_type(q) < 0 || k.scalar_type() != q.scalar_type() ||
      v.scalar_type() != q.scalar_type())
    return false;
  const int64_t two = c.diff ? 2 : 1, B = q.size(0), Hq = q.size(1) / two, Hkv = k.size(1) / two, Lk = k.size(2), D = q.size(3),
                Dv = v.size(3);
  if (q.numel() == 0 || k.numel() == 0 || v.numel() == 0 || k.size(0) != B || v.size(0) != B || v.size(2) != Lk || k.size(3) != D ||
      q.size(1) % two || k.size(1) % two || Hkv == 0 || Hq % Hkv || v.size(1) != Hkv)
    return false;
  if (c.diff ? !(D == 64 && Dv == 128) : !(D == Dv && (D == 32 || D == 64 || D == 128))) return false;
  if (!addressable(q) || !addressable(k) || !addressable(v)) return false;
  const auto dev = q.device();
  return k.device() == dev && v.device() == dev && dev.index() == c10::hip::current_device();
}

bool bias_fits(const Call& c, int i) {
  const Tensor& b = c.bias[i];
  const int64_t div = c.bias_div[i], B = c.q.size(0), Hq = c.q.size(1) / (c.diff ? 2 : 1);
  if (b.dim() != 4 || b.device() != c.q.device() || div < 1 || B % div || (b.scalar_type() != at::kFloat && b.scalar_type() != c.q.scalar_type()))
    return false;
  const int64_t want[4] = {B / div, Hq, c.q.size(2), c.k.size(2)};
  for (int ax = 0; ax < 4; ++ax)
    if ((b.size(ax) != want[ax] && b.size(ax) != 1) || b.stride(ax) < 0) return false;
  return b.size(3) == 1 || b.stride(3) == 1;
}

bool gate_fits(const Call& c) {
  const Tensor& g = c.gate;
  return g.scalar_type() == c.q.scalar_type() && g.dim() == 4 && g.device() == c.q.device() && g.size(0) == c.q.size(0) &&
         g.size(1) == c.q.size(1) / (c.diff ? 2 : 1) && g.size(2) == c.q.size(2) && g.size(3) == c.v.size(3) && addressable(g);
}

// Whether the shared-bias gradient kernels take a differentiable call with bias operands, a gate or both; puts the shared operand
// first.  `given`: the operands as the caller passed them (c.bias, or c.given_bias).
bool shared_bias_gradients(Call& c, Tensor* given) {
  const int64_t Hq = c.q.size(1), Lq = c.q.size(2), Lk = c.k.size(2), B = c.q.size(0);
  if (c.bias[1].defined() && c.bias[1].size(1) == Hq && c.bias[1].size(2) == Lq && Hq * Lq > 1) {
    std::swap(c.bias[0], c.bias[1]);
    std::swap(c.bias_div[0], c.bias_div[1]);
    if (given != c.bias) std::swap(given[0], given[1]);
  }
  // a batch axis of 1 says that all batch entries share the operand: the gradient kernels write one [Hq, Lq, Lk] per
  // B / divisor, and there is room for one
  if (c.bias[0].defined() && c.bias[0].size(0) == 1) c.bias_div[0] = B;
  fl_attn_params p = {};
  fill(c, p);
  return c.bias[0].defined() && c.bias[0].size(1) == Hq && c.bias[0].size(2) == Lq && c.bias[0].size(3) == Lk &&
         !(c.bias[1].defined() && (given[1].requires_grad() || c.bias[1].size(1) != 1 || c.bias[1].size(2) != 1)) &&
         g_api.shared_bias_bwd_bytes(&p) > 0;
}

// forward(q, k, v, scale, mask_kind, window, prefix, doc_ids, alibi_heads, softcap, biases, gate, diff, lambda, seq_major)
PyObject* py_forward(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 15) {
    PyErr_SetString(PyExc_TypeError, "forward takes 15 positional arguments");
    return nullptr;
  }
  if (!g_api.fwd) Py_RETURN_NONE;
  Call c;
  if (!take_tensor(a[0], c.q) || !take_tensor(a[1], c.k) || !take_tensor(a[2], c.v)) Py_RETURN_NONE;
  if (mode_active()) Py_RETURN_NONE;
  c.diff = a[12] == Py_True;
  c.seq_major = a[14] == Py_True;
  if (!operands_fit(c)) Py_RETURN_NONE;
  const Tensor &q = c.q, &k = c.k, &v = c.v;
  const int64_t B = q.size(0), Lq = q.size(2), Lk = k.size(2);
  const auto dev = q.device();
  if (a[3] == Py_None) {
    c.scale = 1.0 / std::sqrt((double)q.size(3));
  } else {
    c.scale = PyFloat_AsDouble(a[3]);
  }
  c.mask_kind = PyLong_AsLongLong(a[4]);
  c.window = PyLong_AsLongLong(a[5]);
  c.prefix = PyLong_AsLongLong(a[6]);
  c.alibi_heads = PyLong_AsLongLong(a[8]);
  c.softcap = PyFloat_AsDouble(a[9]);
  c.lambda = PyFloat_AsDouble(a[13]);
  if (PyErr_Occurred()) {  // (an argument of another type: the Python path converts it or says what is wrong)
    PyErr_Clear();
    Py_RETURN_NONE;
  }
  constexpr int64_t kInt = INT32_MAX;
  if (std::abs(c.window) > kInt || std::abs(c.prefix) > kInt || B > kInt || Lq > kInt || Lk > kInt) Py_RETURN_NONE;
  if (a[7] != Py_None) {
    if (!take_tensor(a[7], c.doc) || c.doc.scalar_type() != at::kLong || c.doc.dim() != 2 || c.doc.size(1) != Lk ||
        (c.doc.size(0) != B && c.doc.size(0) != 1) || c.doc.stride(1) != 1 || c.doc.device() != dev)
      Py_RETURN_NONE;
  }
  const bool is_doc = c.mask_kind == FL_MASK_DOCUMENT || c.mask_kind == FL_MASK_DOCUMENT_CAUSAL;
  if (is_doc != c.doc.defined()) Py_RETURN_NONE;
  PyObject* biases = a[10];
  if (!PyTuple_Check(biases) && !PyList_Check(biases)) Py_RETURN_NONE;
  const Py_ssize_t nb = PySequence_Fast_GET_SIZE(biases);
  if (nb > 2) Py_RETURN_NONE;
  for (Py_ssize_t i = 0; i < nb; ++i) {
    PyObject* pair = PySequence_Fast_GET_ITEM(biases, i);
    if (!PyTuple_Check(pair) || PyTuple_GET_SIZE(pair) != 2 || !PyLong_Check(PyTuple_GET_ITEM(pair, 1))) Py_RETURN_NONE;
    c.bias_div[i] = PyLong_AsLongLong(PyTuple_GET_ITEM(pair, 1));
    if (!take_tensor(PyTuple_GET_ITEM(pair, 0), c.bias[i]) || !bias_fits(c, i)) Py_RETURN_NONE;
  }
  if (a[11] != Py_None && (!take_tensor(a[11], c.gate) || !gate_fits(c))) Py_RETURN_NONE;
  c.wants_grad = at::GradMode::is_enabled() && (q.requires_grad() || k.requires_grad() || v.requires_grad() ||
                                                (c.gate.defined() && c.gate.requires_grad()) ||
                                                (c.bias[0].defined() && c.bias[0].requires_grad()) ||
                                                (c.bias[1].defined() && c.bias[1].requires_grad()));
  if (c.wants_grad) {
    if (c.diff) Py_RETURN_NONE;
    if (nb || c.gate.defined()) {
      if (!shared_bias_gradients(c, c.bias)) Py_RETURN_NONE;
    } else {
      c.seq_major = false;
    }
  }
  Tensor out = attend(c);
  if (!out.defined()) Py_RETURN_NONE;
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// evoformer(q, k, v, biases, scale, gate): attention over the rows of [*, S, H, D] operands with biases broadcastable to
// [*, H, S, S], as attention_variants.evoformer.attention_reference; None when the call is not of the plain kind.
PyObject* py_evoformer(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 6) {
    PyErr_SetString(PyExc_TypeError, "evoformer takes 6 positional arguments");
    return nullptr;
  }
  if (!g_api.fwd) Py_RETURN_NONE;
  Call c;
  if (!take_tensor(a[0], c.given_q) || !take_tensor(a[1], c.given_k) || !take_tensor(a[2], c.given_v) || mode_active()) Py_RETURN_NONE;
  const Tensor &q = c.given_q, &k = c.given_k, &v = c.given_v;
  if (q.dim() < 4 || k.sizes() != q.sizes() || v.sizes() != q.sizes()) Py_RETURN_NONE;
  const size_t nl = (size_t)q.dim() - 3;
  c.lead.assign(q.sizes().begin(), q.sizes().begin() + nl);
  c.q = heads_first(q, nl);
  c.k = heads_first(k, nl);
  c.v = heads_first(v, nl);
  c.seq_major = true;
  if (!c.q.defined() || !c.k.defined() || !c.v.defined() || !operands_fit(c)) Py_RETURN_NONE;
  c.scale = a[4] == Py_None ? 1.0 / std::sqrt((double)c.q.size(3)) : PyFloat_AsDouble(a[4]);
  if (PyErr_Occurred()) {
    PyErr_Clear();
    Py_RETURN_NONE;
  }
  constexpr int64_t kInt = INT32_MAX;
  if (c.q.size(0) > kInt || c.q.size(2) > kInt) Py_RETURN_NONE;
  c.mask_kind = FL_MASK_NONE;
  PyObject* biases = a[3];
  if (!PyTuple_Check(biases) && !PyList_Check(biases)) Py_RETURN_NONE;
  const Py_ssize_t nb = PySequence_Fast_GET_SIZE(biases);
  if (nb > 2) Py_RETURN_NONE;
  for (Py_ssize_t i = 0; i < nb; ++i) {
    if (!take_tensor(PySequence_Fast_GET_ITEM(biases, i), c.given_bias[i])) Py_RETURN_NONE;
    c.bias[i] = kernel_bias(c.given_bias[i], c.lead, c.q.size(1), c.q.size(2), c.bias_div[i]);
    if (!c.bias[i].defined() || !bias_fits(c, (int)i)) Py_RETURN_NONE;
  }
  if (a[5] != Py_None) {
    if (!take_tensor(a[5], c.given_gate) || c.given_gate.sizes() != v.sizes()) Py_RETURN_NONE;
    c.gate = heads_first(c.given_gate, nl);
    if (!c.gate.defined() || !gate_fits(c)) Py_RETURN_NONE;
  }
  const auto wants = [](const Tensor& t) { return t.defined() && t.requires_grad(); };
  c.wants_grad = at::GradMode::is_enabled() && (wants(q) || wants(k) || wants(v) || wants(c.given_gate) || wants(c.given_bias[0]) ||
                                                wants(c.given_bias[1]));
  if (c.wants_grad && !shared_bias_gradients(c, c.given_bias)) Py_RETURN_NONE;
  Tensor out = attend(c);
  if (!out.defined()) Py_RETURN_NONE;
  return THPVariable_Wrap(c.wants_grad ? std::move(out) : with_lead(out, c.lead));
  END_HANDLE_TH_ERRORS
}

// key_chunks(q, k, v): into how many chunks ops._split_over_keys cuts the keys (0: it does not, operands it cannot judge
// included), and whether the front end should let it
PyObject* py_key_chunks(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 3) {
    PyErr_SetString(PyExc_TypeError, "key_chunks takes three tensors");
    return nullptr;
  }
  Call c;
  int64_t chunks = 0;
  bool better = false;
  if (g_api.fwd && THPVariable_Check(a[0]) && THPVariable_Check(a[1]) && THPVariable_Check(a[2])) {
    const Tensor &q = c.q = THPVariable_Unpack(a[0]), &k = c.k = THPVariable_Unpack(a[1]), &v = c.v = THPVariable_Unpack(a[2]);
    if (element_type(q) >= 0 && q.dim() == 4 && k.dim() == 4 && v.dim() == 4 &&
        q.numel() > 0 && k.numel() > 0 && v.numel() > 0 && k.size(0) == q.size(0) && v.size(0) == q.size(0) && k.size(3) == q.size(3) &&
        v.size(1) == k.size(1) && v.size(2) == k.size(2) && q.size(1) % k.size(1) == 0 && k.stride(3) == 1 && v.stride(3) == 1) {
      fl_attn_params p = {};
      uint64_t bytes;
      fill(c, p);
      const int64_t groups = (int64_t)p.B * p.Hq * ((p.Lq + 127) / 128);
      chunks = key_chunks(p, k, v, groups);
      better = chunks && (!g_api.rows_plan(&p, &bytes) || chunks_beat_rows_kernel(p, groups, chunks));
    }
  }
  return Py_BuildValue("LN", (long long)chunks, PyBool_FromLong(better));
  END_HANDLE_TH_ERRORS
}

// bind(addresses): the C ABI's functions in the order of Api, as integers
PyObject* py_bind(PyObject*, PyObject* const* a, Py_ssize_t n) {
  void* f[kApiFunctions];
  if (n != kApiFunctions) {
    PyErr_SetString(PyExc_TypeError, "bind takes the addresses of ten functions");
    return nullptr;
  }
  for (int i = 0; i < kApiFunctions; ++i) f[i] = PyLong_AsVoidPtr(a[i]);
  if (PyErr_Occurred()) return nullptr;
  g_api.fwd = reinterpret_cast<decltype(g_api.fwd)>(f[0]);
  g_api.bwd = reinterpret_cast<decltype(g_api.bwd)>(f[1]);
  g_api.workspace = reinterpret_cast<decltype(g_api.workspace)>(f[2]);
  g_api.bwd_workspace = reinterpret_cast<decltype(g_api.bwd_workspace)>(f[3]);
  g_api.bwd_split_bytes = reinterpret_cast<decltype(g_api.bwd_split_bytes)>(f[4]);
  g_api.rows_plan = reinterpret_cast<decltype(g_api.rows_plan)>(f[5]);
  g_api.shared_bias_bwd_bytes = reinterpret_cast<decltype(g_api.shared_bias_bwd_bytes)>(f[6]);
  g_api.shared_bias_bwd = reinterpret_cast<decltype(g_api.shared_bias_bwd)>(f[7]);
  g_api.last_error = reinterpret_cast<decltype(g_api.last_error)>(f[8]);
  g_api.fwd_ungated = reinterpret_cast<decltype(g_api.fwd_ungated)>(f[9]);
  Py_RETURN_NONE;
}

PyMethodDef kMethods[] = {
    {"forward", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(&py_forward)), METH_FASTCALL, "Result of the call, or None when it is not of the plain kind."},
    {"evoformer", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(&py_evoformer)), METH_FASTCALL, "Result of an Evoformer call, or None when it is not of the plain kind."},
    {"key_chunks", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(&py_key_chunks)), METH_FASTCALL, "Chunks the keys may be cut into, and whether they should be."},
    {"bind", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(&py_bind)), METH_FASTCALL, "Takes the addresses of the C ABI's functions."},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_host", "Native host path of the attention front ends.", -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

extern "C" __attribute__((visibility("default"))) PyObject* PyInit__host(void) { return PyModule_Create(&kModule); }
