// Native call layer of pope_amd's eager calls: descriptor, workspaces, launch and autograd node of the
// flash attention, the similarity and the polar transform on libpope_hip.so (include/pope_abi.h).
//
// A small call is bound by the host: a (1, 4, 257, 64) training step spent 75-150 us (by host) in
// Python between kernels of 45 us, a similarity step 115-175 us in the custom-op dispatch layers.  The
// Python modules keep the argument checks that raise, the padding and the torch.library ops
// (torch.compile tracing, opcheck); what is here is their forward / backward, with the same
// workspaces, flags and entry points, under torch::autograd::Function.  Nothing is kept between calls.
#include <torch/extension.h>

#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/functions/basic_ops.h>
#include <torch/csrc/jit/frontend/tracer.h>

#include <algorithm>
#include <atomic>
#include <climits>
#include <cstring>

#include "../../include/pope_abi.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

// whether the last flash backward reused its forward's preparation (read by tests)
std::atomic<bool> g_last_bwd_prepared{false};

void check(int status, const char* what) {
  if (status == POPE_OK) return;
  char msg[512];
  pope_last_error(msg, sizeof msg);
  TORCH_CHECK(false, "pope_amd ", what, " failed (status ", status, "): ", msg);
}

size_t workspace_bytes(int op, const pope_desc& d) {
  size_t n = 0;
  check(pope_workspace_bytes(op, &d, &n), "workspace query");
  return n;
}

// torch's caching allocator returns 512-byte aligned blocks
Tensor bytes_like(const Tensor& t, size_t n) {
  return n ? at::empty({(int64_t)n}, t.options().dtype(at::kByte).requires_grad(false)) : Tensor();
}
Tensor fp32_like(const Tensor& t, at::IntArrayRef shape) {
  return at::empty(shape, t.options().dtype(at::kFloat).requires_grad(false));
}

void* data(const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }
void* stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.get_device()).stream(); }
int deterministic_flag() { return at::globalContext().deterministicAlgorithms() ? POPE_FLAG_DETERMINISTIC : 0; }

void strides3(int64_t* dst, const Tensor& t) {
  for (int i = 0; i < 3; ++i) dst[i] = t.stride(i);
}

// (b, h, n) element strides of a freqs table; an extent of 1 broadcasts (stride 0).
void freqs_strides(int64_t* dst, const Tensor& f) {
  const auto st = [&](int64_t i) { return f.size(i) == 1 ? (int64_t)0 : f.stride(i); };
  const int64_t n = f.dim();
  TORCH_CHECK_VALUE(n >= 2 && n <= 4, "freqs must be 2-D, 3-D or 4-D, got ", f.sizes());
  dst[0] = n >= 3 ? st(0) : 0;
  dst[1] = n == 4 ? st(1) : 0;
  dst[2] = st(n - 2);
}

// The gradient of freqs, and its strides for d.  The library clears and fills the positions n < Nk of one table per
// batch and head the descriptor tells apart: any other entry (a longer table, more batches, a broadcast extent)
// stays zero, and a broadcast extent's gradient is summed into its first entry, not written past the tensor
// (grouped heads: more query heads than entries).
Tensor phase_grad(const Tensor& freqs, pope_desc& d) {
  const int64_t n = freqs.dim();
  bool whole = freqs.size(-2) == d.Nk;
  if (n >= 3) whole = whole && freqs.size(0) == (d.f_s[0] ? d.B : 1);
  if (n == 4) whole = whole && freqs.size(1) == (d.f_s[1] ? d.Hq : 1);
  const Tensor g = whole ? fp32_like(freqs, freqs.sizes())
                         : at::zeros(freqs.sizes(), freqs.options().dtype(at::kFloat).requires_grad(false));
  freqs_strides(d.df_s, g);
  for (int i = 0; i < 2; ++i)
    if (d.f_s[i] == 0) d.df_s[i] = 0;
  return g;
}

int dtype_code(const Tensor& t) {
  switch (t.scalar_type()) {
    case at::kFloat: return POPE_F32;
    case at::kHalf: return POPE_F16;
    case at::kBFloat16: return POPE_BF16;
    default: TORCH_CHECK_TYPE(false, "pope_amd: unsupported dtype ", t.scalar_type());
  }
}

pope_desc desc_of(const Tensor& q, const Tensor& k, const Tensor& freqs, const Tensor& bias) {
  pope_desc d{};
  d.B = q.size(0);
  d.Hq = q.size(1);
  d.Nq = q.size(2);
  d.D = q.size(3);
  d.Hk = k.size(1);
  d.Nk = k.size(2);
  d.R = freqs.defined() ? freqs.size(-1) : 0;
  d.dtype = dtype_code(q);
  strides3(d.q_s, q);
  strides3(d.k_s, k);
  if (freqs.defined()) {
    freqs_strides(d.f_s, freqs);
    d.bias_sh = bias.size(0) > 1 ? bias.stride(0) : 0;
  }
  return d;
}

// Whether nothing on this thread traces, records or transforms torch's operators: no torch.jit.trace, no dispatch mode
// (the pre-dispatch ones have a stack of their own) and no functorch transform.  One call in place of four from
// Python: the guard takes 1.2 us for a call's six tensors; with two of these checks, from Python, it took 1.3.
bool untraced() {
  using c10::DispatchKey;
  return !torch::jit::tracer::isTracing() && c10::impl::TorchDispatchModeTLS::stack_len() == 0 &&
         !c10::impl::tls_is_dispatch_key_included(DispatchKey::PreDispatch) &&
         !c10::impl::tls_is_dispatch_key_included(DispatchKey::FuncTorchDynamicLayerFrontMode);
}

// Whether a backward has to run on the torch.library ops: its gradients come from a tracer, a mode or a transform
// (batched gradients, a vectorised Jacobian) that a launch through raw pointers would pass by.
bool on_ops(at::TensorList grads) {
  if (!untraced()) return true;
  for (const Tensor& g : grads)
    if (g.defined() && (!g.has_storage() || g.unsafeGetTensorImpl()->is_python_dispatch())) return true;
  return false;
}

// A registered op of pope_amd (its Python modules are imported before anything here runs).
template <typename Sig>
c10::TypedOperatorHandle<Sig> op(const char* name) {
  return c10::Dispatcher::singleton().findSchemaOrThrow(name, "").typed<Sig>();
}
using Grads4 = std::tuple<Tensor, Tensor, Tensor, Tensor>;
using Grads5 = std::tuple<Tensor, Tensor, Tensor, Tensor, Tensor>;

// Every operand on q's GPU: the kernels read raw pointers.
void check_device(const Tensor& q, std::initializer_list<const Tensor*> ts) {
  TORCH_CHECK(q.is_cuda(), "pope_amd runs on GPU tensors only");
  for (const Tensor* t : ts)
    TORCH_CHECK(!t->defined() || t->device() == q.device(), "pope_amd: operand on ", t->device(), " next to q on ", q.device());
}

// ---------------------------------------------------------------- padded rows

// Columns of a padded tensor: `cols` real ones, the first `split` in place, the others `gap` further on,
// `width` in all; `fill`: element bits of the gap.
struct PadCols {
  int64_t split, gap, cols, width;
  uint32_t fill;
};

// Widths of a call whose head dim D or rotate dim R is no multiple of 8 (pope_amd/_pad.py has the plan
// and the reasons): rotate dims R -> R8, head dims D -> Dp.
struct PadPlan {
  int64_t D, R, R8, Dp;
  PadCols qk(const Tensor& t) const {   // the gap: a logit whose softplus and sigmoid are 0
    const float logit = -1.0e4f;
    uint32_t bits = 0;
    if (t.scalar_type() == at::kFloat) std::memcpy(&bits, &logit, 4);
    else if (t.scalar_type() == at::kHalf) bits = c10::Half(logit).x;
    else bits = c10::BFloat16(logit).x;
    return {R, R8 - R, D, Dp, bits};
  }
  PadCols v() const { return {D, 0, D, Dp, 0}; }
  PadCols phase() const { return {R, 0, R, R8, 0}; }
};

// Every tensor padded or unpadded, in one launch.
variable_list pad_rows(at::TensorList ts, const std::vector<PadCols>& cols, bool pad) {
  std::vector<pope_pad> d(ts.size());
  variable_list out;
  for (size_t i = 0; i < ts.size(); ++i) {
    const Tensor& t = ts[i];
    const PadCols& c = cols[i];
    const int64_t n = t.dim(), lead = n - 1;
    check_device(ts[0], {&t});
    TORCH_CHECK_VALUE(n >= 1 && n <= 4 && t.size(-1) == (pad ? c.cols : c.width), "pope_amd: ", t.sizes(),
                      " does not have rows of ", pad ? c.cols : c.width);
    std::vector<int64_t> shape = t.sizes().vec();
    shape.back() = pad ? c.width : c.cols;
    out.push_back(at::empty(shape, t.options().requires_grad(false)));
    pope_pad& p = d[i];
    p = pope_pad{};
    p.src = t.data_ptr();
    p.dst = out.back().data_ptr();
    for (int64_t j = 0; j < 3; ++j) {
      const int64_t x = lead - 3 + j;   // right-aligned leading dims
      TORCH_CHECK_VALUE(x < 0 || t.size(x) <= INT_MAX, "pope_amd: tensor too large to pad");
      p.shape[j] = x < 0 ? 1 : (int32_t)t.size(x);
      p.src_s[j] = x < 0 ? 0 : t.stride(x);
      p.dst_s[j] = x < 0 ? 0 : out.back().stride(x);
    }
    p.src_s[3] = t.stride(-1);
    p.pad = pad;
    p.elem = (int32_t)t.element_size();
    p.split = (int32_t)c.split;
    p.gap = (int32_t)c.gap;
    p.cols = (int32_t)c.cols;
    p.dst_cols = (int32_t)shape.back();
    p.fill = c.fill;
  }
  check(pope_pad_rows(d.data(), (int)d.size(), stream_of(ts[0])), "padding");
  return out;
}

bool tracked(at::TensorList ts);

// The gradients' move with torch's operators, for backwards on the ops.
Tensor pad_row_ops(const Tensor& t, const PadCols& c, bool pad) {
  const auto part = [&](int64_t from, int64_t n) { return t.narrow(-1, from, n); };
  if (!pad) return at::cat({part(0, c.split), part(c.split + c.gap, c.cols - c.split)}, -1);
  return at::cat({at::constant_pad_nd(part(0, c.split), {0, c.gap}),
                  at::constant_pad_nd(part(c.split, c.cols - c.split), {0, c.width - c.cols - c.gap})}, -1);
}

// Gradients under create_graph: differentiating them again raises, as it does through the torch.library
// ops (whose backward ops have no autograd formula), instead of treating them as constants.
variable_list once_differentiable(variable_list grads, const char* what) {
  if (!at::GradMode::is_enabled()) return grads;
  variable_list in;
  for (const Tensor& g : grads)
    if (g.defined()) in.push_back(g.detach().requires_grad_(true));
  auto err = std::make_shared<torch::autograd::DelayedError>(
      std::string("pope_amd ") + what + ": the gradient is not differentiable a second time", (int64_t)in.size());
  const variable_list out = (*err)(std::move(in));
  size_t i = 0;
  for (Tensor& g : grads)
    if (g.defined()) g = out[i++];
  return grads;
}

// pad_rows under autograd: the gradients take the inverse move (the gap's gradient is dropped, or zero).
// Its inputs are the tensors that need a gradient and its outputs their moved copies, made before, so
// that what needs no gradient (freqs, mostly) stays a constant for the node after this one.
// (mark_non_differentiable would do that too, but compiled autograd asserts that no node has any.)
struct PadFn : torch::autograd::Function<PadFn> {
  static variable_list forward(AutogradContext* ctx, at::TensorList ts, const variable_list& moved,
                               const std::vector<PadCols>& cols, bool pad) {
    std::vector<int64_t> flat;
    for (const PadCols& c : cols) flat.insert(flat.end(), {c.split, c.gap, c.cols, c.width});
    ctx->saved_data["cols"] = flat;
    ctx->saved_data["pad"] = pad;
    ctx->set_materialize_grads(false);
    return moved;
  }

  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const std::vector<int64_t> flat = ctx->saved_data["cols"].toIntVector();
    variable_list ts;
    std::vector<PadCols> cols;
    std::vector<size_t> at_;
    for (size_t i = 0; i < grads.size(); ++i)
      if (grads[i].defined() && ctx->needs_input_grad(i)) {
        ts.push_back(grads[i]);
        cols.push_back({flat[4 * i], flat[4 * i + 1], flat[4 * i + 2], flat[4 * i + 3], 0});
        at_.push_back(i);
      }
    variable_list r(grads.size() + 3);
    if (ts.empty()) return r;
    const bool pad = !ctx->saved_data["pad"].toBool();
    if (on_ops(ts)) {
      for (size_t j = 0; j < ts.size(); ++j) r[at_[j]] = pad_row_ops(ts[j], cols[j], pad);
      return r;
    }
    variable_list out = pad_rows(ts, cols, pad);
    // the node before this one may have marked its gradients as not differentiable: so are the moved ones
    if (std::any_of(ts.begin(), ts.end(), [](const Tensor& t) { return t.requires_grad(); }))
      out = once_differentiable(std::move(out), "padding");
    for (size_t j = 0; j < out.size(); ++j) r[at_[j]] = out[j];
    return r;
  }
};

variable_list padded(at::TensorList ts, const std::vector<PadCols>& cols, bool pad) {
  variable_list out = pad_rows(ts, cols, pad), in, moved;
  std::vector<PadCols> in_cols;
  std::vector<size_t> at_;
  for (size_t i = 0; i < ts.size(); ++i)
    if (tracked(ts[i])) {
      in.push_back(ts[i]);
      moved.push_back(out[i]);
      in_cols.push_back(cols[i]);
      at_.push_back(i);
    }
  if (in.empty()) return out;
  const variable_list r = PadFn::apply(at::TensorList(in), moved, in_cols, pad);
  for (size_t j = 0; j < r.size(); ++j) out[at_[j]] = r[j];
  return out;
}

// ---------------------------------------------------------------- flash attention

Tensor unit_feature(const Tensor& t) { return t.stride(-1) == 1 ? t : t.contiguous(); }

void check_flash(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& freqs, const Tensor& bias,
                 const Tensor& mask) {
  check_device(q, {&k, &v, &freqs, &bias, &mask});
  TORCH_CHECK_VALUE(q.dim() == 4 && k.dim() == 4 && v.dim() == 4, "q, k, v must be 4-D, got ", q.sizes(), ", ", k.sizes(),
                    ", ", v.sizes());
  TORCH_CHECK_VALUE(v.sizes() == k.sizes(), "v ", v.sizes(), " must match k ", k.sizes());
  TORCH_CHECK_VALUE(!mask.defined() || (mask.dim() == 2 && mask.size(0) == q.size(0) && mask.size(1) == k.size(2)), "mask ",
                    mask.defined() ? mask.sizes() : at::IntArrayRef(), " must be (batch, seq_k) = (", q.size(0), ", ", k.size(2), ")");
  for (const Tensor* t : {&k, &v})
    TORCH_CHECK_TYPE(t->scalar_type() == q.scalar_type(), "pope_amd flash: operand of dtype ", t->scalar_type(),
                     " next to q of dtype ", q.scalar_type());
  TORCH_CHECK_VALUE(k.size(0) == q.size(0) && k.size(3) == q.size(3) && k.size(1) > 0 && q.size(1) % k.size(1) == 0,
                    "incompatible q ", q.sizes(), " and k ", k.sizes());
  if (freqs.defined()) {
    TORCH_CHECK_VALUE(freqs.size(-2) >= k.size(2), "freqs has ", freqs.size(-2), " positions, keys need ", k.size(2));
    // fewer batches or heads than the call has would be read past the end (the library refuses per-head tables of grouped heads)
    for (int64_t i = 0; i + 2 < freqs.dim() && i < (q.size(1) == k.size(1) ? 2 : 1); ++i)
      TORCH_CHECK_VALUE(freqs.size(i) == 1 || freqs.size(i) >= q.size(i) || freqs.stride(i) == 0, "freqs has ", freqs.size(i),
                        i ? " heads" : " batches", ", the call ", q.size(i));
    TORCH_CHECK_VALUE(bias.size(-1) == freqs.size(-1) && (bias.size(0) == 1 || bias.size(0) == k.size(1)), "bias ",
                      bias.sizes(), " must be (1 or ", k.size(1), ", ", freqs.size(-1), ")");
  }
}

// decode_head_groups() of the library: whether some power-of-two group of the query heads fits.
bool decode_groups(int64_t Hq, int64_t D) {
  for (int64_t g = 1; g <= Hq; g *= 2)
    if (Hq % g == 0 && Hq / g * D <= 4096) return true;
  return false;
}

// The same decision as hip_pope_flash_attn._decode_eligible (tests/test_decode_gpu.py compares them around the
// shortest caches).
bool decode_eligible(const pope_desc& d, int64_t min_keys) {
  if (d.Nq != 1 || d.causal || (d.Nk < min_keys && (int64_t)d.Nk * d.D < 36 * min_keys) || d.D > 128 || !decode_groups(d.Hq, d.D)) return false;
  if (d.R && (d.f_s[1] != 0 || d.f_s[0] % 4 || d.f_s[2] % 4)) return false;
  return (int64_t)(d.Nk - 1) * std::max(d.k_s[2], d.v_s[2]) + d.D < INT_MAX;
}

// One size for a forward and its backward, which reuses the preparation in it.
size_t flash_workspace_bytes(pope_desc d) {
  d.flags = deterministic_flag();
  return workspace_bytes(d.flags ? POPE_OP_FLASH_BWD : POPE_OP_FLASH_FWD, d);
}

struct FlashOut {
  Tensor o, lse, ws;
};

FlashOut flash_forward(const Tensor& q0, const Tensor& k0, const Tensor& v0, Tensor freqs, const Tensor& bias,
                       const Tensor& mask, bool causal, double scale, int64_t decode_min_keys) {
  const Tensor q = unit_feature(q0), k = unit_feature(k0), v = unit_feature(v0);
  check_flash(q, k, v, freqs, bias, mask);
  FlashOut r;
  r.o = at::empty_like(q);
  r.lse = fp32_like(q, q.sizes().slice(0, 3));
  pope_desc d = desc_of(q, k, freqs, bias);
  d.causal = causal;
  d.softmax_scale = (float)scale;
  strides3(d.v_s, v);
  strides3(d.o_s, r.o);
  if (mask.defined()) d.mask_sb = mask.stride(0);
  const auto* mp = static_cast<const uint8_t*>(data(mask));
  auto* lse = static_cast<float*>(r.lse.data_ptr());
  void* s = stream_of(q);
  if (decode_eligible(d, decode_min_keys)) {
    if (freqs.defined() && reinterpret_cast<uintptr_t>(freqs.data_ptr()) % 16) {
      // a table in memory torch did not allocate: an aligned dense copy, with its strides
      freqs = freqs.clone(at::MemoryFormat::Contiguous);
      freqs_strides(d.f_s, freqs);
    }
    const size_t n = workspace_bytes(POPE_OP_FLASH_DECODE, d);
    const Tensor ws = bytes_like(q, n);
    check(pope_flash_decode(&d, q.data_ptr(), k.data_ptr(), v.data_ptr(), static_cast<const float*>(data(freqs)),
                            static_cast<const float*>(data(bias)), mp, r.o.data_ptr(), lse, data(ws), n, s), "flash decode");
    return r;
  }
  // the workspace holds the preparation the backward reuses and, under deterministic mode, the
  // backward's phase-derivative region after it
  const size_t n = flash_workspace_bytes(d);
  const size_t np = workspace_bytes(POPE_OP_FLASH_FWD_PARTIALS, d);
  r.ws = bytes_like(q, n);
  const Tensor parts = bytes_like(q, np);
  check(pope_flash_fwd_split(&d, q.data_ptr(), k.data_ptr(), v.data_ptr(), static_cast<const float*>(data(freqs)),
                             static_cast<const float*>(data(bias)), mp, r.o.data_ptr(), lse, data(r.ws), n, data(parts), np, s),
        "flash forward");
  return r;
}

Tensor opt(const std::optional<Tensor>& t) { return t.has_value() ? *t : Tensor(); }

struct FlashFn : torch::autograd::Function<FlashFn> {
  // freqs and bias come together, so the node's inputs 3 and 4 are theirs where they exist
  static Tensor forward(AutogradContext* ctx, const Tensor& q, const Tensor& k, const Tensor& v,
                        const std::optional<Tensor>& freqs_, const std::optional<Tensor>& bias_,
                        const std::optional<Tensor>& mask_, bool causal, double scale, int64_t decode_min_keys, bool reuse,
                        int64_t cols) {
    const Tensor freqs = opt(freqs_), bias = opt(bias_), mask = opt(mask_);
    FlashOut r = flash_forward(q, k, v, freqs, bias, mask, causal, scale, decode_min_keys);
    ctx->save_for_backward({q, k, v, freqs, bias, mask, r.o, r.lse, reuse ? r.ws : Tensor()});
    ctx->saved_data["causal"] = causal;
    ctx->saved_data["cols"] = cols;
    ctx->saved_data["scale"] = scale;
    return leading_columns(r.o, cols);
  }

  // The first `cols` columns of o (all: o itself) as an output of the node: no autograd view of o, but with
  // its version counter, so that an in-place change of the output is seen by the saved o.
  static Tensor leading_columns(const Tensor& o, int64_t cols) {
    if (cols == o.size(3)) return o;
    Tensor x;
    {
      at::AutoDispatchBelowADInplaceOrView plain;
      x = o.narrow(3, 0, cols);
    }
    torch::autograd::impl::set_version_counter(x, torch::autograd::impl::version_counter(o));
    return x;
  }

  static variable_list backward_ops(AutogradContext* ctx, const variable_list& sv, Tensor dout) {
    if (const int64_t cols = ctx->saved_data["cols"].toInt(); cols < sv[0].size(3))
      dout = pad_row_ops(dout, {cols, 0, cols, sv[0].size(3), 0}, true);
    const auto maybe = [](const Tensor& t) { return t.defined() ? std::optional<Tensor>(t) : std::nullopt; };
    const bool need_df = sv[3].defined() && ctx->needs_input_grad(3), need_db = sv[4].defined() && ctx->needs_input_grad(4);
    using O = const std::optional<Tensor>&;
    const auto [dq, dk, dv, df, db] =
        op<Grads5(const Tensor&, const Tensor&, const Tensor&, const Tensor&, const Tensor&, const Tensor&, O, O, O, bool,
                  double, bool, bool, O)>("pope_amd::flash_bwd")
            .call(dout, sv[0], sv[1], sv[2], sv[6], sv[7], maybe(sv[3]), maybe(sv[4]), maybe(sv[5]),
                  ctx->saved_data["causal"].toBool(), ctx->saved_data["scale"].toDouble(), need_df, need_db, maybe(sv[8]));
    return {dq, dk, dv, need_df ? df : Tensor(), need_db ? db : Tensor(), Tensor(), Tensor(), Tensor(), Tensor(), Tensor(), Tensor()};
  }

  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const variable_list sv = ctx->get_saved_variables();
    if (on_ops(grads)) return backward_ops(ctx, sv, grads[0]);
    const Tensor q = unit_feature(sv[0]), k = unit_feature(sv[1]), v = unit_feature(sv[2]), freqs = sv[3], bias = sv[4],
                 mask = sv[5], o = unit_feature(sv[6]), fwd_ws = sv[8];
    const Tensor lse = sv[7].contiguous();
    Tensor dout = unit_feature(grads[0]);
    if (dout.scalar_type() != q.scalar_type()) dout = dout.to(q.scalar_type());
    if (const int64_t cols = ctx->saved_data["cols"].toInt(); cols < q.size(3))
      dout = pad_rows({dout}, {{cols, 0, cols, q.size(3), 0}}, true)[0];
    check_flash(q, k, v, freqs, bias, mask);
    TORCH_CHECK_VALUE(dout.sizes() == q.sizes(), "do ", dout.sizes(), " must match q ", q.sizes());
    const bool need_df = freqs.defined() && ctx->needs_input_grad(3);
    const bool need_db = bias.defined() && ctx->needs_input_grad(4);
    const Tensor dq = at::empty_like(q), dk = at::empty_like(k), dv = at::empty_like(v);
    Tensor dfreqs, dbias;
    if (need_db) dbias = fp32_like(bias, bias.sizes());
    pope_desc d = desc_of(q, k, freqs, bias);
    d.causal = ctx->saved_data["causal"].toBool();
    d.softmax_scale = (float)ctx->saved_data["scale"].toDouble();
    strides3(d.v_s, v);
    strides3(d.o_s, o);
    strides3(d.do_s, dout);
    strides3(d.dq_s, dq);
    strides3(d.dk_s, dk);
    strides3(d.dv_s, dv);
    if (need_df) dfreqs = phase_grad(freqs, d);
    if (mask.defined()) d.mask_sb = mask.stride(0);
    d.flags = POPE_FLAG_ZERO_GRADS | deterministic_flag();
    // with the partials the workspace is the forward's
    const size_t n = flash_workspace_bytes(d), np = workspace_bytes(POPE_OP_FLASH_BWD_PARTIALS, d);
    const bool prepared = fwd_ws.defined() && (size_t)fwd_ws.numel() == n;
    g_last_bwd_prepared = prepared;
    if (prepared) d.flags |= POPE_FLAG_PREPARED;
    const Tensor ws = prepared ? fwd_ws : bytes_like(q, n);
    const Tensor parts = bytes_like(q, np);
    check(pope_flash_bwd_split(&d, dout.data_ptr(), q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(),
                               static_cast<const float*>(lse.data_ptr()), static_cast<const float*>(data(freqs)),
                               static_cast<const float*>(data(bias)), static_cast<const uint8_t*>(data(mask)),
                               dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), static_cast<float*>(data(dfreqs)),
                               static_cast<float*>(data(dbias)), data(ws), n, data(parts), np, stream_of(q)),
          "flash backward");
    return {dq, dk, dv, dfreqs, dbias, Tensor(), Tensor(), Tensor(), Tensor(), Tensor(), Tensor()};
  }
};

// Whether a call has to go through the autograd node (which also refuses forward-mode tangents).
bool tracked(at::TensorList ts) {
  for (const Tensor& t : ts)
    if (t.defined() && ((at::GradMode::is_enabled() && t.requires_grad()) || t._fw_grad(0).defined())) return true;
  return false;
}

Tensor flash(const Tensor& q, const Tensor& k, const Tensor& v, const std::optional<Tensor>& freqs,
             const std::optional<Tensor>& bias, const std::optional<Tensor>& mask, bool causal, double scale,
             int64_t decode_min_keys, bool reuse) {
  const Tensor f = opt(freqs), b = opt(bias), m = opt(mask);
  if (!tracked({q, k, v, f, b})) return flash_forward(q, k, v, f, b, m, causal, scale, decode_min_keys).o;
  TORCH_CHECK_VALUE(f.defined() == b.defined(), "freqs and bias come together");
  return FlashFn::apply(q, k, v, freqs, bias, mask, causal, scale, decode_min_keys, reuse, q.size(-1));
}

// The same on unpadded rows: q, k, v, freqs and bias padded in one launch, o's real columns.
Tensor flash_padded(const Tensor& q, const Tensor& k, const Tensor& v, const std::optional<Tensor>& freqs,
                    const std::optional<Tensor>& bias, const std::optional<Tensor>& mask, bool causal, double scale,
                    int64_t decode_min_keys, bool reuse, int64_t R, int64_t R8, int64_t Dp) {
  const Tensor f = opt(freqs), b = opt(bias), m = opt(mask);
  TORCH_CHECK_VALUE(f.defined() == b.defined(), "freqs and bias come together");
  const PadPlan plan{q.size(-1), R, R8, Dp};
  variable_list ts{q, k, v};
  std::vector<PadCols> cols{plan.qk(q), plan.qk(k), plan.v()};
  if (f.defined() && R8 != R) {
    ts.insert(ts.end(), {f, b});
    cols.insert(cols.end(), {plan.phase(), plan.phase()});
  }
  variable_list p = padded(ts, cols, true);
  if (f.defined() && p.size() == 3) p.insert(p.end(), {f, b});
  p.resize(5);
  if (!tracked({p[0], p[1], p[2], p[3], p[4]}))
    return flash_forward(p[0], p[1], p[2], p[3], p[4], m, causal, scale, decode_min_keys).o.narrow(3, 0, plan.D);
  const auto maybe = [](const Tensor& t) { return t.defined() ? std::optional<Tensor>(t) : std::nullopt; };
  return FlashFn::apply(p[0], p[1], p[2], maybe(p[3]), maybe(p[4]), mask, causal, scale, decode_min_keys, reuse, plan.D);
}

// ---------------------------------------------------------------- similarity and polar transform

// Views the kernels read in 16-byte vectors: unit feature stride, other strides multiples of 4
// elements, 16-byte aligned start.
Tensor rows4(Tensor t) {
  const auto off = [](const Tensor& x) { return reinterpret_cast<uintptr_t>(x.data_ptr()) % 16 != 0; };
  bool bad = t.stride(-1) != 1 || off(t);
  for (int64_t i = 0; i + 1 < t.dim(); ++i) bad = bad || t.stride(i) % 4 != 0;
  if (bad) {
    t = t.contiguous();
    if (off(t)) t = t.clone();
  }
  return t;
}

struct SimFn : torch::autograd::Function<SimFn> {
  static Tensor run(const Tensor& q0, const Tensor& k0, const Tensor& freqs, const Tensor& bias, bool split) {
    check_device(q0, {&k0, &freqs, &bias});
    const Tensor q = rows4(q0), k = rows4(k0);
    pope_desc d = desc_of(q, k, freqs, bias);
    d.flags = split ? POPE_FLAG_SPLIT_BF16 : 0;
    const Tensor sim = fp32_like(q, {q.size(0), q.size(1), q.size(2), k.size(2)});
    strides3(d.sim_s, sim);
    const size_t n = workspace_bytes(POPE_OP_SIM_FWD, d);
    const Tensor ws = bytes_like(q, n);
    check(pope_sim_fwd(&d, q.data_ptr(), k.data_ptr(), static_cast<const float*>(freqs.data_ptr()),
                       static_cast<const float*>(bias.data_ptr()), sim.data_ptr(), data(ws), n, stream_of(q)),
          "similarity forward");
    return sim;
  }

  static Tensor forward(AutogradContext* ctx, const Tensor& q, const Tensor& k, const Tensor& freqs, const Tensor& bias,
                        bool split) {
    ctx->save_for_backward({q, k, freqs, bias});
    ctx->saved_data["split"] = split;
    return run(q, k, freqs, bias, split);
  }

  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const variable_list sv = ctx->get_saved_variables();
    const bool need_df = ctx->needs_input_grad(2) && sv[2].size(-1) > 0;
    const bool need_db = ctx->needs_input_grad(3) && sv[3].size(-1) > 0;
    if (on_ops(grads)) {
      const auto [dq, dk, df, db] =
          op<Grads4(const Tensor&, const Tensor&, const Tensor&, const Tensor&, const Tensor&, bool, bool, bool)>("pope_amd::sim_bwd")
              .call(grads[0], sv[0], sv[1], sv[2], sv[3], need_df, need_db, ctx->saved_data["split"].toBool());
      return {dq, dk, need_df ? df : Tensor(), need_db ? db : Tensor(), Tensor()};
    }
    const Tensor q = rows4(sv[0]), k = rows4(sv[1]), freqs = sv[2], bias = sv[3];
    const Tensor dsim = rows4(grads[0].to(at::kFloat));
    TORCH_CHECK_VALUE(dsim.dim() == 4 && dsim.size(0) == q.size(0) && dsim.size(1) == q.size(1) &&
                          dsim.size(2) == q.size(2) && dsim.size(3) == k.size(2), "dsim ", dsim.sizes(), " does not fit the similarity");
    pope_desc d = desc_of(q, k, freqs, bias);
    d.flags = (ctx->saved_data["split"].toBool() ? POPE_FLAG_SPLIT_BF16 : 0) | deterministic_flag() | POPE_FLAG_ZERO_GRADS;
    strides3(d.sim_s, dsim);
    const Tensor dq = at::empty_like(q), dk = at::empty_like(k);
    strides3(d.dq_s, dq);
    strides3(d.dk_s, dk);
    Tensor dfreqs, dbias;
    if (need_df) dfreqs = phase_grad(freqs, d);
    if (need_db) dbias = fp32_like(bias, bias.sizes());
    const size_t n = workspace_bytes(POPE_OP_SIM_BWD, d);
    const Tensor ws = bytes_like(q, n);
    check(pope_sim_bwd(&d, dsim.data_ptr(), q.data_ptr(), k.data_ptr(), static_cast<const float*>(freqs.data_ptr()),
                       static_cast<const float*>(bias.data_ptr()), dq.data_ptr(), dk.data_ptr(),
                       static_cast<float*>(data(dfreqs)), static_cast<float*>(data(dbias)), data(ws), n, stream_of(q)),
          "similarity backward");
    return once_differentiable({dq, dk, dfreqs, dbias, Tensor()}, "similarity");
  }
};

Tensor sim(const Tensor& q, const Tensor& k, const Tensor& freqs, const Tensor& bias, bool split) {
  if (!tracked({q, k, freqs, bias})) return SimFn::run(q, k, freqs, bias, split);
  return SimFn::apply(q, k, freqs, bias, split);
}

// q, k, freqs and bias of a similarity or polar call, padded in one launch.
variable_list pad_operands(const Tensor& q, const Tensor& k, const Tensor& freqs, const Tensor& bias, const PadPlan& plan) {
  if (plan.R == plan.R8) {
    variable_list p = padded({q, k}, {plan.qk(q), plan.qk(k)}, true);
    p.insert(p.end(), {freqs, bias});
    return p;
  }
  return padded({q, k, freqs, bias}, {plan.qk(q), plan.qk(k), plan.phase(), plan.phase()}, true);
}

Tensor sim_padded(const Tensor& q, const Tensor& k, const Tensor& freqs, const Tensor& bias, bool split, int64_t R,
                  int64_t R8, int64_t Dp) {
  const variable_list p = pad_operands(q, k, freqs, bias, {q.size(-1), R, R8, Dp});
  return sim(p[0], p[1], p[2], p[3], split);
}

struct PolarFn : torch::autograd::Function<PolarFn> {
  // fp32 columns per output row: D + R, or D (re, im) pairs
  static int64_t width(const Tensor& q, const Tensor& freqs, bool cplx) {
    return cplx ? 2 * q.size(-1) : q.size(-1) + freqs.size(-1);
  }

  static variable_list run(const Tensor& q0, const Tensor& k0, const Tensor& freqs, const Tensor& bias, bool cplx) {
    check_device(q0, {&k0, &freqs, &bias});
    const Tensor q = rows4(q0), k = rows4(k0);
    pope_desc d = desc_of(q, k, freqs, bias);
    d.flags = cplx ? POPE_FLAG_COMPLEX : 0;
    const int64_t E = width(q, freqs, cplx);
    const Tensor qh = fp32_like(q, {q.size(0), q.size(1), q.size(2), E});
    const Tensor kh = fp32_like(k, {k.size(0), k.size(1), k.size(2), E});
    check(pope_polar_fwd(&d, q.data_ptr(), k.data_ptr(), static_cast<const float*>(freqs.data_ptr()),
                         static_cast<const float*>(bias.data_ptr()), static_cast<float*>(qh.data_ptr()),
                         static_cast<float*>(kh.data_ptr()), stream_of(q)), "polar transform");
    return {qh, kh};
  }

  static variable_list forward(AutogradContext* ctx, const Tensor& q, const Tensor& k, const Tensor& freqs,
                               const Tensor& bias, bool cplx) {
    ctx->save_for_backward({q, k, freqs, bias});
    ctx->saved_data["cplx"] = cplx;
    return run(q, k, freqs, bias, cplx);
  }

  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const variable_list sv = ctx->get_saved_variables();
    const Tensor q = rows4(sv[0]), k = rows4(sv[1]), freqs = sv[2], bias = sv[3];
    const bool cplx = ctx->saved_data["cplx"].toBool();
    const int64_t E = width(q, freqs, cplx);
    const auto grad = [&](const Tensor& g, const Tensor& x) {
      return g.defined() ? g.to(at::kFloat).contiguous()
                         : at::zeros({x.size(0), x.size(1), x.size(2), E}, x.options().dtype(at::kFloat).requires_grad(false));
    };
    const bool need_df = ctx->needs_input_grad(2), need_db = ctx->needs_input_grad(3);
    const bool ops = on_ops(grads);
    const Tensor gq = grad(grads[0], q), gk = grad(grads[1], k);
    if (ops) {
      const auto [dq, dk, df, db] =
          op<Grads4(const Tensor&, const Tensor&, const Tensor&, const Tensor&, const Tensor&, const Tensor&, bool, bool, bool)>(
              "pope_amd::polar_bwd").call(gq, gk, q, k, freqs, bias, need_df, need_db, cplx);
      return {dq, dk, need_df ? df : Tensor(), need_db ? db : Tensor(), Tensor()};
    }
    pope_desc d = desc_of(q, k, freqs, bias);
    d.flags = (cplx ? POPE_FLAG_COMPLEX : 0) | deterministic_flag();
    const Tensor dq = at::empty_like(q), dk = at::empty_like(k);
    strides3(d.dq_s, dq);
    strides3(d.dk_s, dk);
    Tensor dfreqs, dbias;   // accumulated into
    if (need_df) {
      dfreqs = at::zeros(freqs.sizes(), freqs.options().dtype(at::kFloat).requires_grad(false));
      freqs_strides(d.df_s, dfreqs);
    }
    if (need_db) dbias = at::zeros(bias.sizes(), bias.options().dtype(at::kFloat).requires_grad(false));
    const size_t n = workspace_bytes(POPE_OP_POLAR_BWD, d);
    const Tensor ws = bytes_like(q, n);
    check(pope_polar_bwd(&d, static_cast<const float*>(gq.data_ptr()), static_cast<const float*>(gk.data_ptr()),
                         q.data_ptr(), k.data_ptr(), static_cast<const float*>(freqs.data_ptr()),
                         static_cast<const float*>(bias.data_ptr()), dq.data_ptr(), dk.data_ptr(),
                         static_cast<float*>(data(dfreqs)), static_cast<float*>(data(dbias)), data(ws), n, stream_of(q)),
          "polar transform backward");
    return once_differentiable({dq, dk, dfreqs, dbias, Tensor()}, "polar transform");
  }
};

std::pair<Tensor, Tensor> polar(const Tensor& q, const Tensor& k, const Tensor& freqs, const Tensor& bias, bool cplx) {
  const variable_list r =
      tracked({q, k, freqs, bias}) ? PolarFn::apply(q, k, freqs, bias, cplx) : PolarFn::run(q, k, freqs, bias, cplx);
  return {r[0], r[1]};
}

// Real output on unpadded rows: 2 R interleaved (cos, sin) columns, then the D - R pass-through ones.
std::pair<Tensor, Tensor> polar_padded(const Tensor& q, const Tensor& k, const Tensor& freqs, const Tensor& bias, int64_t R,
                                       int64_t R8, int64_t Dp) {
  const int64_t D = q.size(-1);
  const variable_list p = pad_operands(q, k, freqs, bias, {D, R, R8, Dp});
  const auto [qh, kh] = polar(p[0], p[1], p[2], p[3], false);
  const PadCols c{2 * R, 2 * (R8 - R), D + R, Dp + R8, 0};
  const variable_list r = padded({qh, kh}, {c, c}, false);
  return {r[0], r[1]};
}

}  // namespace

PYBIND11_MODULE(_pope_host, m) {
  const auto nogil = py::call_guard<py::gil_scoped_release>();
  m.def("flash", &flash, nogil);
  m.def("flash_padded", &flash_padded, nogil);
  m.def("sim", &sim, nogil);
  m.def("sim_padded", &sim_padded, nogil);
  m.def("polar", &polar, nogil);
  m.def("polar_padded", &polar_padded, nogil);
  m.def("untraced", &untraced);
  m.def("last_bwd_prepared", [] { return g_last_bwd_prepared.load(); });
  m.def("abi_version", [] { return POPE_ABI_VERSION; });
}
