// Host side of the op wrappers in C++ (module fxgpu._host): the buffers a call needs are
// allocated from torch's caching allocator and its kernels launched through the C ABI in one
// call from Python, on torch's current stream.  The autograd functions stay in Python
// (fxlm/*.py, fxgpu/fused_linear.py) and call these from their forward and backward.
//
// Why: a small layer's kernels take 5-15 us each, and the same work done from Python took
// longer: about 1.3 us per allocation, 5 per ctypes call with a dozen arguments, and the
// checks and views between them.  A function that takes a checked tensor returns nothing
// (None) when a check fails: the Python wrapper then goes through its own checks, which
// raise the error or make the aligned copy.
#include <torch/extension.h>
#include <torch/csrc/utils/pybind.h>
#include <c10/hip/HIPStream.h>

#include <initializer_list>
#include <tuple>
#include <vector>

#include "../../include/fx_abi.h"
#include "fx_internal.h"

namespace {

using at::Tensor;
using OptT = std::optional<Tensor>;

void* stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.get_device()).stream(); }
uint16_t* bf(const Tensor& t) { return static_cast<uint16_t*>(t.data_ptr()); }
uint16_t* bf(const OptT& t) { return t.has_value() ? bf(*t) : nullptr; }
float* f32(const Tensor& t) { return static_cast<float*>(t.data_ptr()); }
bool aligned(const Tensor& t) { return (reinterpret_cast<uintptr_t>(t.data_ptr()) & 15) == 0; }
bool is_bf(const Tensor& t) { return t.scalar_type() == at::kBFloat16; }
at::TensorOptions as_f32(const Tensor& t) { return t.options().dtype(at::kFloat); }

// the C ABI's return code as the Python wrappers report it (fxgpu.abi.call)
void check(int rc, const char* name) {
    if (rc == 0) return;
    const std::string msg = fx_last_error();
    if (rc == FX_EINVAL) throw py::value_error(msg);
    throw std::runtime_error(std::string(name) + " failed: hipError=" + std::to_string(rc) + " (" + msg + ")");
}

const Tensor* given(const Tensor& t) { return &t; }
const Tensor* given(const OptT& t) { return t.has_value() ? &*t : nullptr; }

// Every tensor whose pointer a kernel gets lies on the GPU of the first: a host pointer, or another
// GPU's, is refused here and never launched with
template <class... Rest>
void same_gpu(const Tensor& a, const Rest&... rest) {
    if (!a.is_cuda()) throw std::runtime_error("expected all tensors to be on one GPU, got " + a.device().str());
    for (const Tensor* t : std::initializer_list<const Tensor*>{given(rest)...})
        if (t && t->device() != a.device())
            throw std::runtime_error("expected all tensors to be on one GPU, got " + a.device().str() + " and " +
                                     t->device().str());
}

// ---- RMSNorm ---------------------------------------------------------------------------

bool norm_ok(const Tensor& x, const Tensor& w) {
    if (!is_bf(x) || !is_bf(w) || !x.is_cuda() || !w.is_cuda() || x.dim() < 1) return false;
    const int64_t D = x.size(-1);
    return w.dim() == 1 && w.size(0) == D && D >= 8 && D % 8 == 0 && D <= 8192 && x.is_contiguous() &&
           w.is_contiguous() && aligned(x) && aligned(w);
}

// (y, rstd), or None when x or w need a check or a copy
std::optional<std::tuple<Tensor, Tensor>> norm_fwd(const Tensor& x, const Tensor& w, double eps) {
    if (!norm_ok(x, w)) return std::nullopt;
    same_gpu(x, w);
    const int64_t D = x.size(-1), N = x.numel() / D;
    Tensor y = at::empty(x.sizes(), x.options());
    Tensor rstd = at::empty({N}, as_f32(x));
    check(fx_rms_norm_fwd(bf(x), bf(w), bf(y), f32(rstd), N, (int32_t)D, (float)eps, stream_of(x)), "fx_rms_norm_fwd");
    return std::make_tuple(y, rstd);
}

// (s, y, rstd) for s = x + r
std::optional<std::tuple<Tensor, Tensor, Tensor>> norm_add_fwd(const Tensor& x, const Tensor& r, const Tensor& w,
                                                               double eps) {
    if (!norm_ok(x, w) || r.sizes() != x.sizes() || !is_bf(r) || !r.is_cuda() || !r.is_contiguous() || !aligned(r))
        return std::nullopt;
    same_gpu(x, r, w);
    const int64_t D = x.size(-1), N = x.numel() / D;
    Tensor s = at::empty(x.sizes(), x.options());
    Tensor y = at::empty(x.sizes(), x.options());
    Tensor rstd = at::empty({N}, as_f32(x));
    check(fx_rms_norm_fwd_add(bf(x), bf(r), bf(w), bf(s), bf(y), f32(rstd), N, (int32_t)D, (float)eps, stream_of(x)),
          "fx_rms_norm_fwd_add");
    return std::make_tuple(s, y, rstd);
}

// a gradient as the kernels read it: contiguous, 16-byte aligned, bf16
Tensor grad_rows(const Tensor& g) {
    Tensor t = g.contiguous();
    if (!aligned(t)) t = t.clone();
    if (!is_bf(t)) t = t.to(at::kBFloat16);
    return t;
}

// (dx shaped like x, dw); dx += dres in the same pass when given
std::tuple<Tensor, Tensor> norm_bwd(const Tensor& x, const Tensor& dy, const Tensor& w, const Tensor& rstd,
                                    const OptT& dres) {
    same_gpu(x, dy, w, rstd, dres);
    const int64_t D = x.size(-1), N = x.numel() / D;
    const Tensor g = grad_rows(dy);
    Tensor dx = at::empty(x.sizes(), x.options());
    Tensor dw = at::empty({D}, w.options());
    // fp32 dw, then the kernel's workspace
    const int64_t nwork = fx_rms_norm_bwd_workspace(N, (int32_t)D) / 4, d4 = (D + 3) / 4 * 4;
    Tensor buf = at::empty({d4 + (nwork < 1 ? 1 : nwork)}, as_f32(x));
    float* dw32 = f32(buf);
    if (dres.has_value()) {
        const Tensor r = grad_rows(*dres);
        check(fx_rms_norm_bwd_add(bf(x), bf(g), bf(r), bf(w), f32(rstd), bf(dx), dw32, bf(dw), dw32 + d4, N, (int32_t)D,
                                  stream_of(x)),
              "fx_rms_norm_bwd_add");
    } else {
        check(fx_rms_norm_bwd(bf(x), bf(g), bf(w), f32(rstd), bf(dx), dw32, bf(dw), dw32 + d4, N, (int32_t)D,
                              stream_of(x)),
              "fx_rms_norm_bwd");
    }
    return std::make_tuple(dx, dw);
}

// ---- attention -------------------------------------------------------------------------

bool attn_ok(const Tensor& t) {
    return is_bf(t) && t.is_cuda() && t.stride(-1) == 1 && t.stride(0) % 8 == 0 && t.stride(1) % 8 == 0 &&
           t.stride(2) % 8 == 0 && aligned(t);
}

// q, k, v as the three slices of one (B, T, 3, H, Dh) tensor
fxAttnArgs packed_args(const Tensor& qkv, bool causal, double scale) {
    fxAttnArgs a{};
    a.q = bf(qkv);
    a.k = a.q + qkv.stride(2);
    a.v = a.k + qkv.stride(2);
    a.qsb = a.ksb = a.vsb = qkv.stride(0);
    a.qst = a.kst = a.vst = qkv.stride(1);
    a.qsh = a.ksh = a.vsh = qkv.stride(3);
    a.B = (int32_t)qkv.size(0);
    a.T = (int32_t)qkv.size(1);
    a.H = (int32_t)qkv.size(3);
    a.D = (int32_t)qkv.size(4);
    a.scale = (float)scale;
    a.causal = causal;
    return a;
}

fxAttnArgs split_args(const Tensor& q, const Tensor& k, const Tensor& v, bool causal, double scale) {
    fxAttnArgs a{};
    a.q = bf(q);
    a.k = bf(k);
    a.v = bf(v);
    a.qsb = q.stride(0), a.qst = q.stride(1), a.qsh = q.stride(2);
    a.ksb = k.stride(0), a.kst = k.stride(1), a.ksh = k.stride(2);
    a.vsb = v.stride(0), a.vst = v.stride(1), a.vsh = v.stride(2);
    a.B = (int32_t)q.size(0);
    a.T = (int32_t)q.size(1);
    a.H = (int32_t)q.size(2);
    a.D = (int32_t)q.size(3);
    a.scale = (float)scale;
    a.causal = causal;
    return a;
}

std::tuple<Tensor, Tensor> attn_run_fwd(fxAttnArgs& a, const Tensor& like) {
    Tensor o = at::empty({a.B, a.T, a.H, a.D}, like.options());
    Tensor lse = at::empty({a.B, a.H, a.T}, as_f32(like));
    a.o_out = bf(o);
    a.lse_out = f32(lse);
    check(fx_attn_fwd(&a, stream_of(like)), "fx_attn_fwd");
    return std::make_tuple(o, lse);
}

// (o, lse), or None when a check of q, k, v fails
std::optional<std::tuple<Tensor, Tensor>> attn_fwd(const Tensor& q, const Tensor& k, const Tensor& v, bool causal,
                                                   double scale) {
    if (q.dim() != 4 || k.sizes() != q.sizes() || v.sizes() != q.sizes()) return std::nullopt;
    const int64_t Dh = q.size(3);
    if ((Dh != 64 && Dh != 128) || q.numel() < 1 || q.numel() >= (int64_t)1 << 31 || !attn_ok(q) || !attn_ok(k) ||
        !attn_ok(v))
        return std::nullopt;
    same_gpu(q, k, v);
    fxAttnArgs a = split_args(q, k, v, causal, scale);
    return attn_run_fwd(a, q);
}

std::optional<std::tuple<Tensor, Tensor>> attn_fwd_qkv(const Tensor& qkv, bool causal, double scale) {
    if (qkv.dim() != 5 || qkv.size(2) != 3 || !qkv.is_contiguous() || !is_bf(qkv) || !qkv.is_cuda() || !aligned(qkv))
        return std::nullopt;
    const int64_t Dh = qkv.size(4);
    if ((Dh != 64 && Dh != 128) || qkv.numel() < 1 || qkv.numel() / 3 >= (int64_t)1 << 31) return std::nullopt;
    fxAttnArgs a = packed_args(qkv, causal, scale);
    return attn_run_fwd(a, qkv);
}

void attn_run_bwd(fxAttnArgs& a, const Tensor& o, const Tensor& lse, const Tensor& dout) {
    Tensor d = dout.contiguous();
    if (!is_bf(d)) d = d.to(at::kBFloat16);
    Tensor delta = at::empty({a.B, a.H, a.T}, lse.options());
    a.o = bf(o);
    a.dout = bf(d);
    a.lse = f32(lse);
    a.delta = f32(delta);
    check(fx_attn_bwd(&a, stream_of(o)), "fx_attn_bwd");
}

std::tuple<Tensor, Tensor, Tensor> attn_bwd(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& o,
                                            const Tensor& lse, const Tensor& dout, bool causal, double scale) {
    same_gpu(q, k, v, o, lse, dout);
    fxAttnArgs a = split_args(q, k, v, causal, scale);
    Tensor dq = at::empty(q.sizes(), q.options()), dk = at::empty(q.sizes(), q.options()),
           dv = at::empty(q.sizes(), q.options());
    a.dq = bf(dq);
    a.dk = bf(dk);
    a.dv = bf(dv);
    const int64_t sh = a.D, st = sh * a.H, sb = st * a.T;
    a.dqb = a.dkb = a.dvb = sb;
    a.dqt = a.dkt = a.dvt = st;
    a.dqh = a.dkh = a.dvh = sh;
    attn_run_bwd(a, o, lse, dout);
    return std::make_tuple(dq, dk, dv);
}

Tensor attn_bwd_qkv(const Tensor& qkv, const Tensor& o, const Tensor& lse, const Tensor& dout, bool causal,
                    double scale) {
    same_gpu(qkv, o, lse, dout);
    fxAttnArgs a = packed_args(qkv, causal, scale);
    Tensor dqkv = at::empty(qkv.sizes(), qkv.options());
    a.dq = bf(dqkv);
    a.dk = a.dq + dqkv.stride(2);
    a.dv = a.dk + dqkv.stride(2);
    a.dqb = a.dkb = a.dvb = dqkv.stride(0);
    a.dqt = a.dkt = a.dvt = dqkv.stride(1);
    a.dqh = a.dkh = a.dvh = dqkv.stride(3);
    attn_run_bwd(a, o, lse, dout);
    return dqkv;
}

// ---- linear layers ---------------------------------------------------------------------

// rows as the GEMM kernels read them: unit stride, 16-byte aligned starts, none overlapping another
// (an expanded row, sliding windows)
bool rows_ok(const Tensor& r) {
    return r.stride(1) == 1 && r.stride(0) % 8 == 0 && (r.size(0) <= 1 || r.stride(0) >= r.size(1)) && aligned(r);
}

// t as a (rows, cols) view with such rows, or a copy of it
Tensor rows(const Tensor& t) {
    Tensor r = t.dim() == 2 ? t : t.reshape({-1, t.size(-1)});
    if (!rows_ok(r)) r = r.contiguous();
    if (!aligned(r)) r = r.clone();   // contiguous, but not where it starts
    // one row, whose stride may be anything
    if (r.size(0) == 1 && r.stride(0) != r.size(1)) r = r.reshape({r.size(1)}).unsqueeze(0);
    return r;
}

// y = act(x2 w^T + bias), and h (the pre-activation, act 2: the GELU derivative) when wanted
std::tuple<Tensor, OptT> linear_fwd(const Tensor& x2, const Tensor& w, const OptT& bias, int64_t act, bool want_h) {
    same_gpu(x2, w, bias);
    const int64_t M = x2.size(0), K = x2.size(1), N = w.size(0);
    Tensor y = at::empty({M, N}, x2.options());
    OptT h;
    if (want_h) h = at::empty({M, N}, x2.options());
    check(fx_linear_fwd(bf(x2), x2.stride(0), nullptr, 0, 0, bf(w), bf(bias), bf(y), bf(h), nullptr, M, N, K, (int32_t)act,
                        stream_of(x2)),
          "fx_linear_fwd");
    return std::make_tuple(y, h);
}

// (out, Xg or None), or None when a check of the gather's inputs fails
std::optional<std::tuple<Tensor, OptT>> gather_fwd(const Tensor& X, const Tensor& idx, const Tensor& w, const Tensor& b,
                                                   bool want_xg) {
    if (X.dim() != 2 || w.dim() != 2 || b.dim() != 1 || idx.dim() != 1) return std::nullopt;
    const int64_t F = X.size(1), K = w.size(1), N = w.size(0), B = idx.size(0);
    if (F < 8 || F % 8 || K % F || b.size(0) != N || !is_bf(X) || !is_bf(w) || !is_bf(b) || idx.scalar_type() != at::kInt ||
        !X.is_cuda() || !idx.is_cuda() || !w.is_cuda() || !b.is_cuda() || !X.is_contiguous() || !idx.is_contiguous() ||
        !w.is_contiguous() || !b.is_contiguous())
        return std::nullopt;
    same_gpu(X, idx, w, b);
    Tensor out = at::empty({B, N}, X.options());
    OptT xg;
    if (want_xg) xg = at::empty({B, K}, X.options());
    check(fx_linear_fwd(bf(X), F, static_cast<int32_t*>(idx.data_ptr()), F, X.size(0), bf(w), bf(b), bf(out), nullptr,
                        bf(xg), B, N, K, 0, stream_of(X)),
          "fx_linear_fwd");
    return std::make_tuple(out, xg);
}

// dW = dy^T x
Tensor wgrad(const Tensor& dy, const Tensor& x) {
    if (!is_bf(dy) || !is_bf(x)) throw py::type_error("dy and x must be bfloat16");
    if (!dy.is_cuda() || !x.is_cuda()) throw py::type_error("dy and x must be cuda tensors");
    same_gpu(dy, x);
    const Tensor dy2 = rows(dy), x2 = rows(x);
    if (dy2.size(0) != x2.size(0))
        throw py::value_error("dy has " + std::to_string(dy2.size(0)) + " rows, x has " + std::to_string(x2.size(0)));
    const int64_t T = dy2.size(0), N = dy2.size(1), K = x2.size(1);
    if (N % 8 || K % 8) return at::mm(dy2.t(), x2);
    Tensor dW = at::empty({N, K}, x2.options());
    const int64_t nbytes = fx_linear_wgrad_workspace(N, K, T);
    Tensor work;
    if (nbytes) work = at::empty({(nbytes + 3) / 4}, as_f32(x2));
    check(fx_linear_wgrad(bf(dy2), dy2.stride(0), bf(x2), x2.stride(0), bf(dW), K, nbytes ? f32(work) : nullptr, N, K, T,
                          stream_of(x2)),
          "fx_linear_wgrad");
    return dW;
}

// dx = dy2 w (times g), or None when a layout check fails.  whole: a shape of fx_linear_dgrad
OptT dgrad(const Tensor& dy2, const Tensor& w, const OptT& g, bool whole) {
    if (!dy2.is_cuda()) return std::nullopt;
    same_gpu(dy2, w, g);
    if (!w.is_contiguous() || !aligned(w) || !rows_ok(dy2) || dy2.stride(0) < dy2.size(1) ||
        !is_bf(dy2) || !is_bf(w) || (g.has_value() && (!g->is_contiguous() || !aligned(*g) || !is_bf(*g))))
        return std::nullopt;
    const int64_t M = dy2.size(0), K = dy2.size(1), N = w.size(1);
    Tensor dx = at::empty({M, N}, dy2.options());
    if (whole) {
        if (g.has_value())
            check(fx_linear_dgrad_gate(bf(dy2), dy2.stride(0), bf(w), N, bf(*g), bf(dx), N, M, N, K, stream_of(dy2)),
                  "fx_linear_dgrad_gate");
        else
            check(fx_linear_dgrad(bf(dy2), dy2.stride(0), bf(w), N, nullptr, bf(dx), N, M, N, K, stream_of(dy2)),
                  "fx_linear_dgrad");
        return dx;
    }
    const int64_t nbytes = fx::input_grad_workspace(M, N, K, g.has_value());
    Tensor work;
    if (nbytes) work = at::empty({nbytes / 4}, as_f32(dy2));
    check(fx::input_grad(bf(dy2), dy2.stride(0), bf(w), bf(g), bf(dx), nbytes ? f32(work) : nullptr, M, N, K,
                         stream_of(dy2)),
          "input_grad");
    return dx;
}

// db = the column sums of g (rows, cols) in g's type
Tensor column_sums(const Tensor& g) {
    const int64_t R = g.size(0), C = g.size(1);
    if (!is_bf(g) || !g.is_cuda() || !g.is_contiguous() || !aligned(g) || R < 1 || R > 64 * 65535 || C < 8 || C % 8)
        return g.sum(0);
    Tensor out = at::empty({C}, g.options());
    Tensor work = at::empty({fx::column_sums_workspace(R, C) / 4}, as_f32(g));
    check(fx::column_sums(bf(g), R, C, f32(work), bf(out), stream_of(g)), "column_sums");
    return out;
}

// ---- cross-entropy ---------------------------------------------------------------------

// device scalars (1 / n_valid, that times the gradient scale)
std::tuple<Tensor, Tensor> ce_inv_nvalid(const Tensor& target, int64_t ignore, const OptT& gs, double gs_value) {
    same_gpu(target);
    const auto o = target.options().dtype(at::kFloat);
    Tensor inv_n = at::empty({}, o), mul = at::empty({}, o), g;
    if (gs.has_value()) g = gs->detach().to(target.device(), at::kFloat).reshape({});
    check(fx_ce_inv_nvalid(static_cast<int64_t*>(target.data_ptr()), target.numel(), ignore, gs.has_value() ? f32(g) : nullptr,
                           (float)gs_value, f32(inv_n), f32(mul), stream_of(target)),
          "fx_ce_inv_nvalid");
    return std::make_tuple(inv_n, mul);
}

void ce_rows(const Tensor& logits, const Tensor& target, const OptT& grad, const Tensor& row_loss, const Tensor& mul,
             int64_t ignore) {
    same_gpu(logits, target, grad, row_loss, mul);
    fxCEArgs a{};
    a.logits = bf(logits);
    a.target = static_cast<int64_t*>(target.data_ptr());
    a.grad = bf(grad);
    a.row_loss = f32(row_loss);
    a.mul = f32(mul);
    a.N = logits.size(0);
    a.V = logits.size(1);
    a.ld = logits.stride(0);
    a.ldg = grad.has_value() ? grad->stride(0) : a.V;
    a.ignore_index = ignore;
    check(fx_ce_fwd_grad(&a, stream_of(logits)), "fx_ce_fwd_grad");
}

Tensor ce_finalize(const Tensor& row_loss, const Tensor& inv_n) {
    same_gpu(row_loss, inv_n);
    Tensor loss = at::empty({}, row_loss.options());
    check(fx_ce_loss_finalize(f32(row_loss), row_loss.numel(), f32(inv_n), f32(loss), stream_of(row_loss)),
          "fx_ce_loss_finalize");
    return loss;
}

// (loss, dlogits or None) of checked logits and targets, or None when a check fails
std::optional<std::tuple<Tensor, OptT>> ce_fwd(const Tensor& logits, const Tensor& target, int64_t ignore, bool want_grad) {
    if (!is_bf(logits) || !logits.is_cuda() || !target.is_cuda() || !logits.is_contiguous() || !target.is_contiguous() ||
        target.scalar_type() != at::kLong || logits.dim() != 2 || target.dim() != 1 || target.size(0) != logits.size(0))
        return std::nullopt;
    auto [inv_n, mul] = ce_inv_nvalid(target, ignore, std::nullopt, 1.0);
    Tensor row_loss = at::empty({logits.size(0)}, as_f32(logits));
    OptT grad;
    if (want_grad) grad = at::empty(logits.sizes(), logits.options());
    ce_rows(logits, target, grad, row_loss, mul, ignore);
    return std::make_tuple(ce_finalize(row_loss, inv_n), grad);
}

void ce_scale_grad(const Tensor& grad, const Tensor& g32, const Tensor& applied, int64_t src) {
    same_gpu(grad, g32, applied);
    check(fx_ce_scale_grad(bf(grad), grad.numel(), f32(g32), f32(applied), (int32_t)src, stream_of(grad)),
          "fx_ce_scale_grad");
}

void ce_lin_scale_inplace(const Tensor& dW, const Tensor& dx, const Tensor& g32, const OptT& gs, double inv) {
    same_gpu(dW, dx, g32, gs);
    check(fx_ce_lin_grad_scale_inplace(bf(dW), dW.numel(), bf(dx), dx.numel(), f32(g32), gs.has_value() ? f32(*gs) : nullptr,
                                       (float)inv, stream_of(dx)),
          "fx_ce_lin_grad_scale_inplace");
}

// ---- a decode step's ends ----------------------------------------------------------------

// the step's inputs into a graph's static buffers; false: not tensors the kernel takes
bool decode_inputs(const Tensor& tok, int64_t pos, const Tensor& tok_out, const Tensor& pos_out, const Tensor& lens) {
    if (tok.scalar_type() != at::kLong || !tok.is_contiguous() || tok.device() != tok_out.device() ||
        tok.sizes() != tok_out.sizes())
        return false;
    same_gpu(tok_out, pos_out, lens);
    check(fx::decode_inputs(static_cast<int64_t*>(tok.data_ptr()), tok.numel(), pos, static_cast<int64_t*>(tok_out.data_ptr()),
                            static_cast<int64_t*>(pos_out.data_ptr()), static_cast<int32_t*>(lens.data_ptr()),
                            stream_of(tok)),
          "decode_inputs");
    return true;
}

// E[tok] + P[pos] as (B, 1, D), or None when a check fails
OptT decode_embed(const Tensor& tok, const Tensor& pos, const Tensor& E, const Tensor& P) {
    if (tok.dim() != 1 || tok.scalar_type() != at::kLong || !tok.is_contiguous() || !tok.is_cuda() || tok.numel() < 1 ||
        pos.numel() != 1 || pos.scalar_type() != at::kLong || !pos.is_cuda() || !is_bf(E) || !is_bf(P) || !E.is_cuda() ||
        !P.is_cuda() || E.dim() != 2 || P.dim() != 2 || E.size(1) != P.size(1) || E.size(1) % 8 || E.size(1) < 8 ||
        !E.is_contiguous() || !P.is_contiguous() || !aligned(E) || !aligned(P))
        return std::nullopt;
    same_gpu(tok, pos, E, P);
    const int64_t B = tok.numel(), D = E.size(1);
    Tensor x = at::empty({B, 1, D}, E.options());
    check(fx::decode_embed(static_cast<int64_t*>(tok.data_ptr()), static_cast<int64_t*>(pos.data_ptr()), bf(E), E.size(0), bf(P),
                           P.size(0), bf(x), B, D, stream_of(E)),
          "decode_embed");
    return x;
}

// norm(x) W^T as fp32 for x (B, D) rows, or None when a check fails
OptT few_rows_logits(const Tensor& x, const Tensor& w, const Tensor& norm_w, double eps) {
    if (x.dim() != 2 || w.dim() != 2 || norm_w.dim() != 1 || !is_bf(x) || !is_bf(w) || !is_bf(norm_w) || !x.is_cuda() ||
        !w.is_cuda() || !norm_w.is_cuda() || x.size(0) < 1 || x.size(0) > 64 || w.size(1) != x.size(1) ||
        norm_w.size(0) != x.size(1) || x.size(1) % 8 || x.stride(1) != 1 || x.stride(0) % 8 || !w.is_contiguous() ||
        !norm_w.is_contiguous() || !aligned(x) || !aligned(w) || !aligned(norm_w))
        return std::nullopt;
    same_gpu(x, w, norm_w);
    Tensor out = at::empty({x.size(0), w.size(0)}, as_f32(x));
    check(fx::few_rows_logits(bf(x), x.stride(0), bf(w), bf(norm_w), (float)eps, f32(out), x.size(0), w.size(0), x.size(1),
                              stream_of(x)),
          "few_rows_logits");
    return out;
}

// ---- optimiser -------------------------------------------------------------------------

// The flat layout of FlatAdamW: per parameter its offset, size and weight-decay flag.
struct FlatLayout {
    std::vector<int64_t> off, n;
    std::vector<int32_t> wd;
};

// One optimiser step over the parameters that have a gradient.  t: master, m, v, flat16, step,
// found_inf, grad norm, scale, growth.  h: lr, beta1, beta2, eps, weight decay, max norm,
// growth interval.  Returns the workspace (grown when too small) and -1, or the index of a
// parameter whose gradient is not bf16 (-2 - index: not 16-byte aligned), nothing launched.
std::tuple<Tensor, int64_t> adamw_step(const FlatLayout& f, const std::vector<Tensor>& params, const std::vector<Tensor>& t,
                                       const std::vector<double>& h, Tensor work) {
    std::vector<Tensor> keep;   // contiguous copies, alive until the launches are queued
    std::vector<fxTensorList> lists;
    for (size_t i = 0; i < params.size(); ++i) {
        Tensor g = params[i].grad();
        if (!g.defined()) continue;
        same_gpu(t[0], g);
        if (!is_bf(g)) return std::make_tuple(work, (int64_t)i);
        if (!g.is_contiguous()) {
            g = g.contiguous();
            keep.push_back(g);
        }
        if (!aligned(g)) return std::make_tuple(work, -2 - (int64_t)i);
        if (lists.empty() || lists.back().count == FX_ADAMW_MAX_TENSORS) {
            lists.emplace_back();
            lists.back().count = 0;
        }
        fxTensorList& l = lists.back();
        l.g[l.count] = bf(g);
        l.off[l.count] = f.off[i];
        l.n[l.count] = f.n[i];
        l.wd[l.count] = f.wd[i];
        ++l.count;
    }
    for (const Tensor& s : t) same_gpu(t[0], s);
    const int32_t nl = (int32_t)lists.size();
    if (lists.empty()) lists.emplace_back();   // a list to point to
    const int64_t need = fx_adamw_workspace(lists.data(), nl) / 4;
    if (work.numel() < need) work = at::empty({need}, t[0].options());
    fxAdamWState s{};
    s.master = f32(t[0]);
    s.m = f32(t[1]);
    s.v = f32(t[2]);
    s.p16 = bf(t[3]);
    s.step = static_cast<int32_t*>(t[4].data_ptr());
    s.found_inf = f32(t[5]);
    s.grad_norm = f32(t[6]);
    s.scale = f32(t[7]);
    s.growth = static_cast<int32_t*>(t[8].data_ptr());
    s.work = f32(work);
    s.lr = (float)h[0];
    s.beta1 = (float)h[1];
    s.beta2 = (float)h[2];
    s.eps = (float)h[3];
    s.weight_decay = (float)h[4];
    s.max_grad_norm = (float)h[5];
    s.growth_factor = 2.f;
    s.backoff_factor = 0.5f;
    s.growth_interval = (int32_t)h[6];
    check(fx_adamw_step(&s, lists.data(), nl, stream_of(t[0])), "fx_adamw_step");
    return std::make_tuple(work, (int64_t)-1);
}

}  // namespace

// every function: torch's exceptions (out of memory among them) reach Python as themselves, and other
// Python threads run during the call, as during a ctypes call: an allocation that reaches the driver
// or a launch into a full queue may wait.  So none of them calls Python or keeps state.
#define FX_DEF(name) m.def(#name, torch::wrap_pybind_function_no_gil(name))

PYBIND11_MODULE(_host, m) {
    FX_DEF(norm_fwd);
    FX_DEF(norm_add_fwd);
    FX_DEF(norm_bwd);
    FX_DEF(attn_fwd);
    FX_DEF(attn_fwd_qkv);
    FX_DEF(attn_bwd);
    FX_DEF(attn_bwd_qkv);
    FX_DEF(rows);
    FX_DEF(linear_fwd);
    FX_DEF(gather_fwd);
    FX_DEF(wgrad);
    FX_DEF(dgrad);
    FX_DEF(column_sums);
    FX_DEF(decode_inputs);
    FX_DEF(decode_embed);
    FX_DEF(few_rows_logits);
    FX_DEF(ce_inv_nvalid);
    FX_DEF(ce_rows);
    FX_DEF(ce_finalize);
    FX_DEF(ce_fwd);
    FX_DEF(ce_scale_grad);
    FX_DEF(ce_lin_scale_inplace);
    py::class_<FlatLayout>(m, "FlatLayout")
        .def(py::init([](std::vector<int64_t> off, std::vector<int64_t> n, std::vector<int32_t> wd) {
            return FlatLayout{std::move(off), std::move(n), std::move(wd)};
        }));
    FX_DEF(adamw_step);
}
