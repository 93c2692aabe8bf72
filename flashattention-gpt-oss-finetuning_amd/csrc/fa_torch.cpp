// fa_torch.cpp - PyTorch binding of the C ABI (include/fa_gfx950.h) for the autograd path.
//
// The per-call host work of the drop-in -- tensor checks, output and workspace allocation (the
// caching allocator), the current HIP stream, filling fa_fwd_params / fa_bwd_params and the
// launch -- in C++, so a forward + backward costs a few microseconds of host time instead of
// the tens that per-field ctypes marshalling takes.  Every FLOP still runs in libfa_gfx950.so;
// this module only calls the C ABI.  swda / swda_sinks / swda_varlen are the autograd functions themselves
// in C++ (forward, saved tensors, backward), which the functional forms of the Python package call.
//
// Error behaviour matches the ctypes path (_ops.py): tensors not on a GPU -> RuntimeError,
// unsupported dtype or shape -> ValueError, a C ABI status -> ValueError (argument) or
// RuntimeError (launch), with fa_strerror's text.
#include <torch/extension.h>

#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPGraphsC10Utils.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/jit/frontend/tracer.h>

#include <stdexcept>
#include <string>

#include "../../include/fa_gfx950.h"

namespace {

int32_t dtype_code(const at::Tensor& t) {
  if (t.scalar_type() == at::kBFloat16) return FA_DTYPE_BF16;
  if (t.scalar_type() == at::kHalf) return FA_DTYPE_F16;
  if (t.scalar_type() == at::kFloat) return FA_DTYPE_F32;
  throw std::invalid_argument("q has dtype " + std::string(c10::toString(t.scalar_type())) +
                              "; supported dtypes are bfloat16, float16 and float32");
}

void check(const std::vector<std::pair<const at::Tensor*, const char*>>& ts, bool dim4 = true) {
  const at::Tensor& first = *ts[0].first;
  if (!first.is_cuda())
    throw std::runtime_error(std::string(ts[0].second) + " is on " + first.device().str() +
                             ": the gfx950 attention kernels need GPU tensors (there is no CPU implementation)");
  dtype_code(first);
  for (const auto& [t, name] : ts) {
    if (dim4 && t->dim() != 4) throw std::invalid_argument(std::string(name) + " must be 4-D [B, H, L, D]");
    if (t->device() != first.device())
      throw std::runtime_error(std::string(name) + " is on " + t->device().str() + " but " + ts[0].second +
                               " is on " + first.device().str());
    if (t->scalar_type() != first.scalar_type())
      throw std::invalid_argument(std::string(name) + " has a different dtype than " + ts[0].second);
  }
}

// Inputs the kernels cannot read directly (head-dim stride != 1, strides not whole multiples of
// 16 bytes, base not 16-byte aligned) are copied to a contiguous layout first.
at::Tensor kernel_ready(const at::Tensor& t) {
  const auto st = t.strides();
  const int64_t m = 16 / int64_t(t.element_size()) - 1;
  const auto misaligned = [&](const at::Tensor& x) { return (reinterpret_cast<uintptr_t>(x.data_ptr()) & 15) != 0; };
  if (st[3] != 1 || (st[0] & m) || (st[1] & m) || (st[2] & m) || misaligned(t)) {
    at::Tensor c = t.contiguous();
    if (misaligned(c)) c = c.clone(at::MemoryFormat::Contiguous);
    return c;
  }
  return t;
}

void strides3(int64_t dst[3], const at::Tensor& t) {
  dst[0] = t.stride(0);
  dst[1] = t.stride(1);
  dst[2] = t.stride(2);
}

int32_t clamp_i32(int64_t x) {
  return x < INT32_MIN ? INT32_MIN : (x > INT32_MAX ? INT32_MAX : int32_t(x));
}

void raise_for_status(int rc, const char* what) {
  if (rc == FA_OK) return;
  const std::string msg = std::string(what) + ": " + fa_strerror(rc);
  if (rc == FA_ERR_LAUNCH) throw std::runtime_error(msg);
  throw std::invalid_argument(msg);
}

void* current_stream(const at::Tensor& t) {
  return c10::hip::getCurrentHIPStream(t.device().index()).stream();
}

// Is the call recorded or transformed instead of computed on plain tensors (torch.jit tracing, dispatch modes as
// make_fx's and FakeTensorMode, functorch's transforms, forward-mode AD)?  What a C ABI call writes is
// invisible to all of them: a trace would keep the allocation of its outputs only.
bool transformed(std::initializer_list<const at::Tensor*> ts) {
  if (torch::jit::tracer::isTracing() || c10::impl::TorchDispatchModeTLS::any_modes_set() ||
      c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode))
    return true;
  for (const at::Tensor* t : ts)
    if (t->key_set().has(c10::DispatchKey::Python) || t->_fw_grad(0).defined()) return true;
  return false;
}

// Learned sink logits as the C ABI takes them: float32 [Hq], contiguous, on q's device.
at::Tensor sinks_ready(const at::Tensor& sinks, int64_t Hq, const at::Tensor& q) {
  if (sinks.dim() != 1 || sinks.size(0) != Hq)
    throw std::invalid_argument("sinks must have shape [" + std::to_string(Hq) +
                                "] (one logit per query head)");
  if (sinks.device() != q.device())
    throw std::runtime_error("sinks is on " + sinks.device().str() + " but q is on " + q.device().str());
  return sinks.to(at::kFloat).contiguous();
}

// forward: returns (o, lse) for q [B,Hq,L,D], k/v [B,Hkv,L,D]; o has q's memory layout (as
// torch.empty_like(q) in the reference, flash_attention_gpt_oss.py:356).  With learned sink
// logits (float32-convertible [Hq]) it calls fa_fwd_sinks.
std::vector<at::Tensor> fwd(const at::Tensor& q_in, const at::Tensor& k_in, const at::Tensor& v_in, int64_t window,
                            int64_t sink, double scale, const c10::optional<at::Tensor>& sinks_in) {
  check({{&q_in, "q"}, {&k_in, "k"}, {&v_in, "v"}});
  const c10::DeviceGuard guard(q_in.device());
  const at::Tensor q = kernel_ready(q_in), k = kernel_ready(k_in), v = kernel_ready(v_in);
  const int64_t B = q.size(0), Hq = q.size(1), L = q.size(2), D = q.size(3);
  const at::Tensor sinks = sinks_in.has_value() ? sinks_ready(*sinks_in, Hq, q) : at::Tensor();
  at::Tensor o = at::empty_like(q);
  at::Tensor lse = at::empty({B, Hq, L}, q.options().dtype(at::kFloat));
  fa_fwd_params p{};
  p.q = q.data_ptr();
  p.k = k.data_ptr();
  p.v = v.data_ptr();
  p.o = o.data_ptr();
  p.lse = lse.data_ptr<float>();
  strides3(p.q_stride, q);
  strides3(p.k_stride, k);
  strides3(p.v_stride, v);
  strides3(p.o_stride, o);
  p.lse_stride[0] = lse.stride(0);
  p.lse_stride[1] = lse.stride(1);
  p.lse_stride[2] = lse.stride(2);
  p.batch = clamp_i32(B);
  p.heads_q = clamp_i32(Hq);
  p.heads_kv = clamp_i32(k.size(1));
  p.seqlen = clamp_i32(L);
  p.head_dim = clamp_i32(D);
  p.window = clamp_i32(window);
  p.sink = clamp_i32(sink);
  p.softmax_scale = float(scale);
  p.dtype = dtype_code(q);
  if (sinks.defined())
    raise_for_status(fa_fwd_sinks(&p, sinks.data_ptr<float>(), current_stream(q)), "fa_fwd_sinks");
  else
    raise_for_status(fa_fwd(&p, current_stream(q)), "fa_fwd");
  return {o, lse};
}

// backward: returns (dq, dk, dv) in the input dtype and the layouts of q, k, v; with learned
// sink logits, (dq, dk, dv, dsinks) through fa_bwd_sinks, dsinks float32 [Hq]
std::vector<at::Tensor> bwd(const at::Tensor& q_in, const at::Tensor& k_in, const at::Tensor& v_in,
                            const at::Tensor& o_in, const at::Tensor& lse, const at::Tensor& do_in, int64_t window,
                            int64_t sink, double scale, const c10::optional<at::Tensor>& sinks_in) {
  check({{&q_in, "q"}, {&k_in, "k"}, {&v_in, "v"}, {&o_in, "o"}, {&do_in, "do"}});
  const c10::DeviceGuard guard(q_in.device());
  const at::Tensor q = kernel_ready(q_in), k = kernel_ready(k_in), v = kernel_ready(v_in);
  const at::Tensor o = kernel_ready(o_in), dout = kernel_ready(do_in);
  const int64_t B = q.size(0), Hq = q.size(1), L = q.size(2), D = q.size(3), Hkv = k.size(1);
  const at::Tensor sinks = sinks_in.has_value() ? sinks_ready(*sinks_in, Hq, q) : at::Tensor();
  at::Tensor dq = at::empty_like(q);
  at::Tensor dk = at::empty_like(k);
  at::Tensor dv = at::empty_like(v);
  const size_t ws_bytes = fa_bwd_full_workspace_bytes(clamp_i32(B), clamp_i32(Hq), clamp_i32(Hkv), clamp_i32(L),
                                                      clamp_i32(D), clamp_i32(window), clamp_i32(sink), dtype_code(q), -1);
  at::Tensor ws = at::empty({int64_t(ws_bytes > 256 ? ws_bytes : 256)}, q.options().dtype(at::kByte));
  fa_bwd_params p{};
  p.q = q.data_ptr();
  p.k = k.data_ptr();
  p.v = v.data_ptr();
  p.o = o.data_ptr();
  p.dout = dout.data_ptr();
  p.lse = lse.data_ptr<float>();
  p.dq = dq.data_ptr();
  p.dk = dk.data_ptr();
  p.dv = dv.data_ptr();
  strides3(p.q_stride, q);
  strides3(p.k_stride, k);
  strides3(p.v_stride, v);
  strides3(p.o_stride, o);
  strides3(p.do_stride, dout);
  p.lse_stride[0] = lse.stride(0);
  p.lse_stride[1] = lse.stride(1);
  p.lse_stride[2] = lse.stride(2);
  strides3(p.dq_stride, dq);
  strides3(p.dk_stride, dk);
  strides3(p.dv_stride, dv);
  p.batch = clamp_i32(B);
  p.heads_q = clamp_i32(Hq);
  p.heads_kv = clamp_i32(Hkv);
  p.seqlen = clamp_i32(L);
  p.head_dim = clamp_i32(D);
  p.window = clamp_i32(window);
  p.sink = clamp_i32(sink);
  p.softmax_scale = float(scale);
  p.dtype = dtype_code(q);
  if (sinks.defined()) {
    at::Tensor dsinks = at::empty({Hq}, q.options().dtype(at::kFloat));
    raise_for_status(fa_bwd_sinks(&p, sinks.data_ptr<float>(), dsinks.data_ptr<float>(), ws.data_ptr(),
                                  size_t(ws.numel()), current_stream(q)),
                     "fa_bwd_sinks");
    return {dq, dk, dv, dsinks};
  }
  raise_for_status(fa_bwd(&p, ws.data_ptr(), size_t(ws.numel()), current_stream(q)), "fa_bwd");
  return {dq, dk, dv};
}

// The autograd function of flash_attention_gpt_oss.py:340-438 (FlashSWDAWithSink) in C++: the
// forward saves (q, k, v, o, lse) and the window / sink / scale, the backward returns dq, dk, dv
// and no gradient for the other four arguments.  The autograd engine runs this backward on its
// device thread without taking the Python interpreter lock, so a training step spends no Python
// time in the backward; the computation is the same fa_fwd / fa_bwd calls as fwd() / bwd().
struct SwdaFunction : public torch::autograd::Function<SwdaFunction> {
  static at::Tensor forward(torch::autograd::AutogradContext* ctx, const at::Tensor& q, const at::Tensor& k,
                            const at::Tensor& v, int64_t window, int64_t sink, double scale) {
    std::vector<at::Tensor> r = fwd(q, k, v, window, sink, scale, c10::nullopt);
    ctx->save_for_backward({q, k, v, r[0], r[1]});
    ctx->saved_data["window"] = window;
    ctx->saved_data["sink"] = sink;
    ctx->saved_data["scale"] = scale;
    return r[0];
  }

  static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx,
                                                 torch::autograd::variable_list grads) {
    const torch::autograd::variable_list s = ctx->get_saved_variables();
    std::vector<at::Tensor> g = bwd(s[0], s[1], s[2], s[3], s[4], grads[0], ctx->saved_data["window"].toInt(),
                                    ctx->saved_data["sink"].toInt(), ctx->saved_data["scale"].toDouble(), c10::nullopt);
    return {g[0], g[1], g[2], at::Tensor(), at::Tensor(), at::Tensor()};
  }
};

// The same with GPT-OSS learned sink logits (sinks [Hq]): the backward also returns d sinks, in
// the dtype of sinks.
struct SwdaSinksFunction : public torch::autograd::Function<SwdaSinksFunction> {
  static at::Tensor forward(torch::autograd::AutogradContext* ctx, const at::Tensor& q, const at::Tensor& k,
                            const at::Tensor& v, const at::Tensor& sinks, int64_t window, int64_t sink, double scale) {
    std::vector<at::Tensor> r = fwd(q, k, v, window, sink, scale, sinks);
    ctx->save_for_backward({q, k, v, r[0], r[1], sinks});
    ctx->saved_data["window"] = window;
    ctx->saved_data["sink"] = sink;
    ctx->saved_data["scale"] = scale;
    return r[0];
  }

  static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx,
                                                 torch::autograd::variable_list grads) {
    const torch::autograd::variable_list s = ctx->get_saved_variables();
    std::vector<at::Tensor> g = bwd(s[0], s[1], s[2], s[3], s[4], grads[0], ctx->saved_data["window"].toInt(),
                                    ctx->saved_data["sink"].toInt(), ctx->saved_data["scale"].toDouble(), s[5]);
    return {g[0], g[1], g[2], g[3].to(s[5].scalar_type()), at::Tensor(), at::Tensor(), at::Tensor()};
  }
};

// The autograd functions' forwards; None for a transformed call, which the Python functions take (torch.jit traces
// those as a call, forward-mode AD and functorch refuse them by name).
c10::optional<at::Tensor> swda(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, int64_t window,
                               int64_t sink, double scale) {
  if (transformed({&q, &k, &v})) return c10::nullopt;
  return SwdaFunction::apply(q, k, v, window, sink, scale);
}

c10::optional<at::Tensor> swda_sinks(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v,
                                     const at::Tensor& sinks, int64_t window, int64_t sink, double scale) {
  if (transformed({&q, &k, &v, &sinks})) return c10::nullopt;
  return SwdaSinksFunction::apply(q, k, v, sinks, window, sink, scale);
}

// ---- packed batches ---------------------------------------------------------------------------
// [total, H, D] tensors on one GPU with one supported dtype, all with q's rows and head dim (the kernels
// bound every row they touch by q's row count).
void check_packed(const std::vector<std::pair<const at::Tensor*, const char*>>& ts) {
  const at::Tensor& q = *ts[0].first;
  const auto shape = [](const at::Tensor& t) {
    std::string r = "(";
    for (int64_t i = 0; i < t.dim(); ++i) r += (i ? ", " : "") + std::to_string(t.size(i));
    return r + (t.dim() == 1 ? ",)" : ")");
  };
  for (const auto& [t, name] : ts)
    if (t->dim() != 3)
      throw std::invalid_argument(std::string(name) + " must be 3-D [total, H, D], got shape " + shape(*t));
  check(ts, false);
  for (const auto& [t, name] : ts)
    if (t->size(0) != q.size(0) || t->size(2) != q.size(2))
      throw std::invalid_argument(std::string(name) + " has shape " + shape(*t) + "; packed tensors need " +
                                  std::to_string(q.size(0)) + " rows and head dim " + std::to_string(q.size(2)));
}

// A packed [total, H, D] tensor as the [1, H, total, D] view the C ABI describes (the batch stride is not
// used there), copied where the kernels cannot read it.  `in_place`: the caller leaves its rows where they are,
// at strides that it did not choose, so they are also copied where a sequence of that many rows spans more
// than the kernels' 32-bit offsets.
at::Tensor as_bhld(const at::Tensor& t, int64_t in_place = 0) {
  const int64_t span = ((in_place - 1) * t.stride(0) + t.size(2)) * int64_t(t.element_size());
  const at::Tensor x = in_place > 0 && span >= (int64_t(1) << 31) ? t.contiguous() : t;
  return kernel_ready(x.permute({1, 0, 2}).unsqueeze(0));
}

// The sequences of a packed batch: offsets [B + 1], or starts [B] with lengths.
struct Sequences {
  at::Tensor cu, lens;
  int64_t max_seqlen, token_rows;
  int64_t batch() const { return cu.size(0) - (lens.defined() ? 0 : 1); }
  const int32_t* cu_ptr() const { return cu.data_ptr<int32_t>(); }
  int64_t in_place() const { return lens.defined() ? max_seqlen : 0; }
  const int32_t* lens_ptr() const { return lens.defined() ? lens.data_ptr<int32_t>() : nullptr; }
};

Sequences sequences(const at::Tensor& q, const at::Tensor& cu, const at::Tensor& lens, int64_t max_seqlen,
                    int64_t token_rows) {
  for (const at::Tensor* t : {&cu, &lens})
    if (t->defined() && (t->device() != q.device() || t->scalar_type() != at::kInt || t->dim() != 1 || !t->is_contiguous()))
      throw std::invalid_argument("sequence offsets must be a contiguous 1-D int32 tensor on q's device");
  if (cu.size(0) < (lens.defined() ? 1 : 2) || (lens.defined() && lens.size(0) != cu.size(0)))
    throw std::invalid_argument("sequence offsets must hold at least one sequence, and as many lengths as starts");
  return Sequences{cu, lens, max_seqlen, lens.defined() ? token_rows : q.size(0)};
}

// (o [total, Hq, D], lse float32 [Hq, total])
std::vector<at::Tensor> fwd_packed(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, const Sequences& sq,
                                   int64_t window, int64_t sink, double scale, const at::Tensor& sinks_in) {
  check_packed({{&q, "q"}, {&k, "k"}, {&v, "v"}});
  const c10::DeviceGuard guard(q.device());
  const int64_t total = q.size(0), Hq = q.size(1), D = q.size(2);
  const int64_t ip = sq.in_place();
  const at::Tensor qv = as_bhld(q, ip), kv = as_bhld(k, ip), vv = as_bhld(v, ip);
  const at::Tensor sinks = sinks_in.defined() ? sinks_ready(sinks_in, Hq, q) : at::Tensor();
  at::Tensor o = at::empty({total, Hq, D}, q.options());
  at::Tensor lse = at::empty({Hq, total}, q.options().dtype(at::kFloat));
  const at::Tensor ov = o.permute({1, 0, 2}).unsqueeze(0);
  fa_fwd_params p{};
  p.q = qv.data_ptr();
  p.k = kv.data_ptr();
  p.v = vv.data_ptr();
  p.o = o.data_ptr();
  p.lse = lse.data_ptr<float>();
  strides3(p.q_stride, qv);
  strides3(p.k_stride, kv);
  strides3(p.v_stride, vv);
  strides3(p.o_stride, ov);
  p.lse_stride[1] = lse.stride(0);
  p.lse_stride[2] = lse.stride(1);
  p.batch = clamp_i32(sq.batch());
  p.heads_q = clamp_i32(Hq);
  p.heads_kv = clamp_i32(k.size(1));
  p.seqlen = clamp_i32(sq.max_seqlen);
  p.head_dim = clamp_i32(D);
  p.window = clamp_i32(window);
  p.sink = clamp_i32(sink);
  p.softmax_scale = float(scale);
  p.dtype = dtype_code(q);
  const float* sk = sinks.defined() ? sinks.data_ptr<float>() : nullptr;
  if (sq.lens.defined())
    raise_for_status(fa_fwd_ranges(&p, sq.cu_ptr(), sq.lens_ptr(), clamp_i32(total), clamp_i32(sq.token_rows), sk,
                                   current_stream(q)),
                     "fa_fwd_ranges");
  else
    raise_for_status(fa_fwd_varlen(&p, sq.cu_ptr(), clamp_i32(total), sk, current_stream(q)), "fa_fwd_varlen");
  return {o, lse};
}

// (dq, dk, dv packed like q, k, v, and with sinks dsinks float32 [Hq])
std::vector<at::Tensor> bwd_packed(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, const at::Tensor& o,
                                   const at::Tensor& lse, const at::Tensor& dout, const Sequences& sq, int64_t window,
                                   int64_t sink, double scale, const at::Tensor& sinks_in) {
  check_packed({{&q, "q"}, {&k, "k"}, {&v, "v"}, {&o, "o"}, {&dout, "do"}});
  const c10::DeviceGuard guard(q.device());
  const int64_t total = q.size(0), Hq = q.size(1), D = q.size(2), Hkv = k.size(1);
  const int64_t ip = sq.in_place();
  const at::Tensor qv = as_bhld(q, ip), kv = as_bhld(k, ip), vv = as_bhld(v, ip), ov = as_bhld(o), dov = as_bhld(dout, ip);
  const at::Tensor sinks = sinks_in.defined() ? sinks_ready(sinks_in, Hq, q) : at::Tensor();
  at::Tensor dq = at::empty({total, Hq, D}, q.options());
  at::Tensor dk = at::empty({total, Hkv, D}, q.options());
  at::Tensor dv = at::empty({total, Hkv, D}, q.options());
  at::Tensor dsinks = sinks.defined() ? at::empty({Hq}, q.options().dtype(at::kFloat)) : at::Tensor();
  fa_bwd_params p{};
  p.q = qv.data_ptr();
  p.k = kv.data_ptr();
  p.v = vv.data_ptr();
  p.o = ov.data_ptr();
  p.dout = dov.data_ptr();
  p.lse = lse.data_ptr<float>();
  p.dq = dq.data_ptr();
  p.dk = dk.data_ptr();
  p.dv = dv.data_ptr();
  strides3(p.q_stride, qv);
  strides3(p.k_stride, kv);
  strides3(p.v_stride, vv);
  strides3(p.o_stride, ov);
  strides3(p.do_stride, dov);
  p.lse_stride[1] = lse.stride(0);
  p.lse_stride[2] = lse.stride(1);
  for (int64_t* st : {p.dq_stride, p.dk_stride, p.dv_stride}) {
    st[1] = D;
    st[2] = (st == p.dq_stride ? Hq : Hkv) * D;
  }
  p.batch = clamp_i32(sq.batch());
  p.heads_q = clamp_i32(Hq);
  p.heads_kv = clamp_i32(Hkv);
  p.seqlen = clamp_i32(sq.max_seqlen);
  p.head_dim = clamp_i32(D);
  p.window = clamp_i32(window);
  p.sink = clamp_i32(sink);
  p.softmax_scale = float(scale);
  p.dtype = dtype_code(q);
  const size_t ws_bytes = fa_bwd_full_workspace_bytes(p.batch, p.heads_q, p.heads_kv, p.seqlen, p.head_dim, p.window,
                                                      p.sink, p.dtype, clamp_i32(sq.token_rows));
  at::Tensor ws = at::empty({int64_t(ws_bytes > 256 ? ws_bytes : 256)}, q.options().dtype(at::kByte));
  const float* sk = sinks.defined() ? sinks.data_ptr<float>() : nullptr;
  float* dsk = sinks.defined() ? dsinks.data_ptr<float>() : nullptr;
  if (sq.lens.defined())
    raise_for_status(fa_bwd_ranges(&p, sq.cu_ptr(), sq.lens_ptr(), clamp_i32(total), clamp_i32(sq.token_rows), sk, dsk,
                                   ws.data_ptr(), size_t(ws.numel()), current_stream(q)),
                     "fa_bwd_ranges");
  else
    raise_for_status(fa_bwd_varlen(&p, sq.cu_ptr(), clamp_i32(total), sk, dsk, ws.data_ptr(), size_t(ws.numel()),
                                   current_stream(q)),
                     "fa_bwd_varlen");
  return {dq, dk, dv, dsinks};
}

// FlashSWDAWithSinkVarlen in C++: the forward saves (q, k, v, o, lse, offsets[, lengths][, sinks]), the
// backward returns dq, dk, dv and, with sinks, d sinks in their dtype.
struct SwdaVarlenFunction : public torch::autograd::Function<SwdaVarlenFunction> {
  static at::Tensor forward(torch::autograd::AutogradContext* ctx, const at::Tensor& q, const at::Tensor& k,
                            const at::Tensor& v, const at::Tensor& cu, const c10::optional<at::Tensor>& lens_in,
                            int64_t max_seqlen, int64_t token_rows, int64_t window, int64_t sink, double scale,
                            const c10::optional<at::Tensor>& sinks_in) {
    const at::Tensor lens = lens_in.has_value() ? *lens_in : at::Tensor();
    const at::Tensor sinks = sinks_in.has_value() ? *sinks_in : at::Tensor();
    std::vector<at::Tensor> r =
        fwd_packed(q, k, v, sequences(q, cu, lens, max_seqlen, token_rows), window, sink, scale, sinks);
    ctx->save_for_backward({q, k, v, r[0], r[1], cu, lens, sinks});
    ctx->saved_data["max_seqlen"] = max_seqlen;
    ctx->saved_data["token_rows"] = token_rows;
    ctx->saved_data["window"] = window;
    ctx->saved_data["sink"] = sink;
    ctx->saved_data["scale"] = scale;
    return r[0];
  }

  static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx,
                                                 torch::autograd::variable_list grads) {
    const torch::autograd::variable_list s = ctx->get_saved_variables();
    const Sequences sq = sequences(s[0], s[5], s[6], ctx->saved_data["max_seqlen"].toInt(),
                                   ctx->saved_data["token_rows"].toInt());
    std::vector<at::Tensor> g = bwd_packed(s[0], s[1], s[2], s[3], s[4], grads[0], sq, ctx->saved_data["window"].toInt(),
                                           ctx->saved_data["sink"].toInt(), ctx->saved_data["scale"].toDouble(), s[7]);
    const at::Tensor none;
    return {g[0], g[1], g[2], none, none, none, none, none, none, none,
            s[7].defined() ? g[3].to(s[7].scalar_type()) : none};
  }
};

c10::optional<at::Tensor> swda_varlen(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v,
                                      const at::Tensor& cu, const c10::optional<at::Tensor>& lens, int64_t max_seqlen,
                                      int64_t token_rows, int64_t window, int64_t sink, double scale,
                                      const c10::optional<at::Tensor>& sinks) {
  if (transformed({&q, &k, &v, sinks.has_value() ? &*sinks : &q})) return c10::nullopt;
  return SwdaVarlenFunction::apply(q, k, v, cu, lens, max_seqlen, token_rows, window, sink, scale, sinks);
}

// Per-tensor e4m3 quantisation of a GPU tensor (quantize_fp8 in attention.py): (x8, descale), x8 with x's
// strides; without a given descale it is max |x| / 448.  The host waits for the maximum only: the codes
// are written by a kernel behind it that reads the maximum on the device.  Returns None for tensors
// the kernels do not take (other dtypes, strides with gaps, unaligned or empty) and in transformed calls.
py::object quantize_fp8(const at::Tensor& x_in, c10::optional<double> descale) {
  if (transformed({&x_in})) return py::none();
  const at::Tensor x = x_in.detach();
  const auto st = x.scalar_type();
  const int dtype = st == at::kBFloat16 ? FA_DTYPE_BF16 : st == at::kHalf ? FA_DTYPE_F16 : st == at::kFloat ? FA_DTYPE_F32 : 0;
  if (!x.is_cuda() || dtype == 0 || x.numel() == 0 || !x.is_non_overlapping_and_dense() ||
      (reinterpret_cast<uintptr_t>(x.data_ptr()) & 15) != 0)
    return py::none();
  const c10::DeviceGuard guard(x.device());
  at::Tensor x8 = at::empty_like(x, x.options().dtype(at::kFloat8_e4m3fn));
  void* stream = current_stream(x);
  if (descale.has_value()) {
    raise_for_status(fa_quantize_fp8(x.data_ptr(), dtype, x.numel(), x8.data_ptr(), *descale, stream),
                     "fa_quantize_fp8");
    return py::make_tuple(x8, *descale);
  }
  if (c10::hip::currentStreamCaptureStatusMayInitCtx() != c10::hip::CaptureStatus::None)
    raise_for_status(FA_ERR_LAUNCH, "fa_quantize_fp8_amax under graph capture, where the host cannot read the maximum");
  at::Tensor parts = at::empty({FA_AMAX_PARTS}, x.options().dtype(at::kFloat));
  at::Tensor host = at::empty({FA_AMAX_PARTS}, at::TensorOptions().dtype(at::kFloat).pinned_memory(true));
  float amax = 0.f;
  int rc;
  {
    py::gil_scoped_release nogil;
    rc = fa_quantize_fp8_amax(x.data_ptr(), dtype, x.numel(), x8.data_ptr(), parts.data_ptr<float>(),
                              host.data_ptr<float>(), &amax, stream);
  }
  raise_for_status(rc, "fa_quantize_fp8_amax");
  return py::make_tuple(x8, amax > 0.f ? double(amax) / 448.0 : 1.0);
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.def("swda", &swda,
        "autograd forward of causal sliding-window + sink attention: (q, k, v, window, sink, scale) -> o or None",
        py::arg("q"), py::arg("k"), py::arg("v"), py::arg("window"), py::arg("sink"), py::arg("scale"));
  m.def("swda_sinks", &swda_sinks,
        "autograd forward with learned sink logits: (q, k, v, sinks, window, sink, scale) -> o or None", py::arg("q"),
        py::arg("k"), py::arg("v"), py::arg("sinks"), py::arg("window"), py::arg("sink"), py::arg("scale"));
  m.def("swda_varlen", &swda_varlen,
        "autograd forward of a packed batch: (q, k, v, cu_seqlens or starts, lens, max_seqlen, token_rows, window, sink, "
        "scale, sinks=None) -> o or None",
        py::arg("q"), py::arg("k"), py::arg("v"), py::arg("cu"), py::arg("lens"), py::arg("max_seqlen"),
        py::arg("token_rows"), py::arg("window"), py::arg("sink"), py::arg("scale"), py::arg("sinks") = py::none());
  m.def("quantize_fp8", &quantize_fp8, "per-tensor e4m3 quantisation: (x, descale=None) -> (x8, descale) or None",
        py::arg("x"), py::arg("descale") = py::none());
  m.doc() = "PyTorch binding of libfa_gfx950.so (fa_fwd / fa_bwd)";
  m.def("fwd", &fwd, "forward: (q, k, v, window, sink, scale, sinks=None) -> (o, lse)", py::arg("q"), py::arg("k"),
        py::arg("v"), py::arg("window"), py::arg("sink"), py::arg("scale"), py::arg("sinks") = py::none());
  m.def("bwd", &bwd, "backward: (q, k, v, o, lse, do, window, sink, scale, sinks=None) -> (dq, dk, dv[, dsinks])",
        py::arg("q"), py::arg("k"), py::arg("v"), py::arg("o"), py::arg("lse"), py::arg("do"), py::arg("window"),
        py::arg("sink"), py::arg("scale"), py::arg("sinks") = py::none());
}
