// The eager host path of the package's hot calls: argument checks, allocations,
// GEMM calls, native launches and autograd nodes in C++, behind a Python module.
//
// A block's training step is about 30 launches of a few microseconds each at
// small sizes; enqueued from Python through registered ops it took 735 us of host
// time for 283 us of GPU work (8 x 200 positions of the default model's widths in
// fp32), and takes about 390 us from here. The prefill of one prompt of 117
// positions at the 110M widths went 238 -> 143 us (now 154, with copies of the
// session's matrices), a decode position of the default model 244 -> 171 us.
// Everything here evaluates what kernel.py's implementations evaluate, with the
// same native calls in the same order, and without the interpreter's lock; a call
// that is not a plain eager one, or that they would refuse, returns None and is
// left to them: tracing, functorch transforms, forward-mode tangents, tensor
// subclasses, disagreeing shapes, other dtypes and devices.
#include <ATen/ATen.h>
#include <ATen/core/dispatch/Dispatcher.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>
#include <torch/csrc/utils/pybind.h>

#include <optional>
#include <string>
#include <vector>

#include "../../include/ulm_fm.h"

namespace py = pybind11;
using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

namespace {

constexpr float kLogWMin = -7.f, kLogWMax = 12.f;   // kernel.py's LOG_W_MIN, LOG_W_MAX (model.py:75)

void check(const char *name, int status) {
    if (status != ULM_OK)
        throw std::runtime_error(std::string(name) + " failed with status " + std::to_string(status) + ": " + ulm_last_error());
}

int code(at::ScalarType t) {
    switch (t) {
    case at::kFloat: return ULM_F32;
    case at::kBFloat16: return ULM_BF16;
    case at::kHalf: return ULM_F16;
    default: throw py::type_error("unsupported dtype; expected float32, bfloat16 or float16");
    }
}
bool has_code(const Tensor &t) {
    return t.scalar_type() == at::kFloat || t.scalar_type() == at::kBFloat16 || t.scalar_type() == at::kHalf;
}

void *stream_of(const Tensor &t) { return c10::hip::getCurrentHIPStream(t.get_device()).stream(); }

Tensor f32c(const Tensor &t) { return (t.scalar_type() == at::kFloat ? t : t.to(at::kFloat)).contiguous(); }
const float *fp(const Tensor &t) { return t.defined() ? static_cast<const float *>(t.data_ptr()) : nullptr; }
float *fpm(const Tensor &t) { return static_cast<float *>(t.data_ptr()); }

// the current device's tensors of a call
struct Maker {
    at::TensorOptions opt;
    explicit Maker(const Tensor &like) : opt(at::TensorOptions().device(like.device())) {}
    Tensor operator()(at::IntArrayRef shape, at::ScalarType dt = at::kFloat) const { return at::empty(shape, opt.dtype(dt)); }
    Tensor bytes(size_t n) const { return at::empty({static_cast<int64_t>(std::max<size_t>(n, 1))}, opt.dtype(at::kByte)); }
};

// keys of tensors, and of the thread, that only the Python implementations know how to meet
const c10::DispatchKeySet kNotPlain({c10::DispatchKey::FuncTorchGradWrapper, c10::DispatchKey::FuncTorchBatched,
                                     c10::DispatchKey::FuncTorchVmapMode, c10::DispatchKey::Functionalize,
                                     c10::DispatchKey::Batched, c10::DispatchKey::VmapMode,
                                     c10::DispatchKey::Python, c10::DispatchKey::PythonTLSSnapshot,
                                     c10::DispatchKey::Negative, c10::DispatchKey::Conjugate,
                                     c10::DispatchKey::ZeroTensor, c10::DispatchKey::Named});

bool plain_thread() {
    return !c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode) &&
           !c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::Python) &&
           !c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::Functionalize) && !torch::jit::tracer::isTracing();
}

// Whether a node's backward may launch on these gradients and saved tensors by
// itself. Not where the backward is to be differentiated (create_graph), or where
// a gradient, or what a saved-tensor hook gave back, is a batch of tensors or
// another that only a dispatch can meet: the registered backward op serves those
// as it does for a traced call, and has no derivative of its own, so that a
// second one raises.
bool launches(const variable_list &grads, const variable_list &saved) {
    bool ok = !at::GradMode::is_enabled() && plain_thread();
    for (const variable_list *list : {&grads, &saved})
        for (const Tensor &t : *list) {
            if (!t.defined()) continue;
            TORCH_CHECK(t.device() == saved[0].device(), "tensors on different devices: ", saved[0].device(), " and ", t.device());
            ok = ok && !t.key_set().has_any(kNotPlain) && t.layout() == at::kStrided;
        }
    return ok;
}

template <class F> auto registered(const char *name) {
    return c10::Dispatcher::singleton().findSchemaOrThrow(name, "").typed<F>();
}

// f() without the interpreter's lock: launches, library GEMMs and the allocator may wait, and other threads run
template <class F> auto unlocked(F f) {
    py::gil_scoped_release release;
    return f();
}

// a Tensor or Parameter proper (no subclass), strided, on a GPU, floating, with no tangent; undefined otherwise
Tensor plain(const py::handle &h) {
    if (!THPVariable_CheckExact(h.ptr())) return {};
    const Tensor &t = THPVariable_Unpack(h.ptr());
    if (!t.defined() || !t.is_cuda() || t.layout() != at::kStrided || !at::isFloatingType(t.scalar_type()) ||
        t.key_set().has_any(kNotPlain) || t._fw_grad(0).defined())
        return {};
    return t;
}

// ---- unified_memory

struct FM : torch::autograd::Function<FM> {
    static variable_list forward(AutogradContext *ctx, const Tensor &r, const Tensor &v, const Tensor &g, const Tensor &w) {
        at::AutoDispatchBelowAutograd guard;
        const int B = r.size(0), T = r.size(1), A = r.size(2), D = v.size(2), vdt = code(v.scalar_type());
        const Maker make(r);
        const Tensor r32 = f32c(r), vc = v.contiguous(), g1 = f32c(g), w32 = f32c(w);
        const Tensor q = make({B, T, A}), fast = make({B, T, D}, v.scalar_type());
        const size_t sb = ulm_fm_saved_bytes(B, T, A, D, vdt), wb = ulm_fm_fwd_workspace_bytes(B, T, A, D, vdt);
        const Tensor saved = at::empty({static_cast<int64_t>(sb)}, make.opt.dtype(at::kByte)), ws = make.bytes(wb);
        check("ulm_fm_fwd", ulm_fm_fwd(fp(r32), vc.data_ptr(), vdt, fp(g1), fp(w32), fpm(q), fast.data_ptr(), vdt,
                                       saved.data_ptr(), sb, ws.data_ptr(), wb, B, T, A, D, stream_of(r)));
        ctx->save_for_backward({r, g, w, saved});
        ctx->saved_data["vdt"] = static_cast<int64_t>(v.scalar_type());
        ctx->saved_data["D"] = static_cast<int64_t>(D);
        ctx->set_materialize_grads(false);
        return {q, fast};
    }
    static variable_list backward(AutogradContext *ctx, variable_list grads) {
        const auto sv = ctx->get_saved_variables();
        const Tensor &r = sv[0], &g = sv[1], &w = sv[2], &saved = sv[3];
        const Tensor dq = grads[0];
        Tensor dfast = grads[1];
        if (!dq.defined() && !dfast.defined()) return {Tensor(), Tensor(), Tensor(), Tensor()};
        const int B = r.size(0), T = r.size(1), A = r.size(2), D = ctx->saved_data["D"].toInt();
        const auto vt = static_cast<at::ScalarType>(ctx->saved_data["vdt"].toInt());
        const int vdt = code(vt);
        const Maker make(r);
        if (!launches(grads, sv)) {
            using F = std::tuple<Tensor, Tensor, Tensor, Tensor>(const Tensor &, const Tensor &, const Tensor &, const Tensor &,
                                                                 at::ScalarType, const std::optional<Tensor> &, const Tensor &);
            if (!dfast.defined()) dfast = at::zeros({B, T, D}, make.opt.dtype(at::kFloat));
            const auto [dr, dv, dg, dw] = registered<F>("ulm::fm_bwd").call(
                r, g, w, saved, vt, dq.defined() ? std::optional<Tensor>(dq) : std::nullopt, dfast);
            return {dr, dv, dg.reshape(g.sizes()), dw};
        }
        at::AutoDispatchBelowAutograd guard;
        dfast = dfast.defined() ? dfast.contiguous() : at::zeros({B, T, D}, make.opt.dtype(at::kFloat));
        const int ddt = code(dfast.scalar_type());
        const Tensor r32 = f32c(r), g1 = f32c(g), w32 = f32c(w), dqo = dq.defined() ? f32c(dq) : dq;
        const Tensor dr = make({B, T, A}), dv = make({B, T, D}, dfast.scalar_type()), dg = make({1}), dw = make({A});
        const size_t sb = saved.numel(), wb = ulm_fm_bwd_workspace_bytes(B, T, A, D, ddt, sb, vdt);
        const Tensor ws = make.bytes(wb);
        check("ulm_fm_bwd", ulm_fm_bwd(fp(r32), fp(g1), fp(w32), saved.data_ptr(), sb, vdt, dfast.data_ptr(), ddt, fp(dqo),
                                       fpm(dr), dv.data_ptr(), ddt, fpm(dg), fpm(dw), ws.data_ptr(), wb, B, T, A, D,
                                       stream_of(r)));
        return {dr, dv, dg.reshape(g.sizes()), dw};
    }
};

py::object memory(const py::handle &r_, const py::handle &v_, const py::handle &g_, const py::handle &w_) {
    if (!plain_thread()) return py::none();
    const Tensor r = plain(r_), v = plain(v_), g = plain(g_), w = plain(w_);
    if (!r.defined() || !v.defined() || !g.defined() || !w.defined() || r.dim() != 3 || v.dim() != 3 ||
        r.size(0) != v.size(0) || r.size(1) != v.size(1) || r.numel() == 0 || v.numel() == 0 || w.dim() != 1 ||
        w.size(0) != r.size(2) || g.numel() != 1 || !has_code(v))
        return py::none();
    for (const Tensor *t : {&v, &g, &w})
        if (t->device() != r.device()) return py::none();
    const auto out = unlocked([&] { return FM::apply(r, v, g, w); });
    return py::make_tuple(py::cast(out[0]), py::cast(out[1]));
}

// ---- one UnifiedBlock

Tensor gemm(const Tensor &a, const Tensor &b, at::ScalarType out) {
    return a.scalar_type() == out ? at::mm(a, b) : at::mm(a, b, out);
}

Tensor wgrad(const Tensor &a_, const Tensor &b_, void *s) {
    const int K = a_.size(0), N1 = a_.size(1), N2 = b_.size(1);
    if (a_.scalar_type() != at::kBFloat16 || b_.scalar_type() != at::kBFloat16 || N1 % 8 || N2 % 8)
        return gemm(a_.t(), b_, at::kFloat);
    const Tensor a = a_.contiguous(), b = b_.contiguous();
    const Maker make(a);
    const Tensor c = make({N1, N2});
    const size_t wb = ulm_wgrad_workspace_bytes(K, N1, N2);
    const Tensor ws = make.bytes(wb);
    check("ulm_wgrad", ulm_wgrad(a.data_ptr(), b.data_ptr(), fpm(c), K, N1, N2, ws.data_ptr(), wb, s));
    return c;
}

void addmm_(Tensor &c, const Tensor &a, const Tensor &b) {
    if (a.scalar_type() == c.scalar_type()) at::addmm_out(c, c, a, b);
    else at::addmm_out(c, c, a, b, c.scalar_type());
}

Tensor cast(const Tensor &t, at::ScalarType dt) { return (t.scalar_type() == dt ? t : t.to(dt)).contiguous(); }

// what the forward and the prefill of a block share, up to the fast memory
struct Block {
    int B, T, D, A, Kc, cd;
    int64_t M;
    at::ScalarType cdt;
    void *s;
    Maker make;
    Tensor x32, mw, h, u, rstd, pre, v, b32, le, denom, g1, w32;

    Block(const Tensor &x, const Tensor &norm_w, const Tensor &conv_w, const Tensor &key_w, const std::optional<Tensor> &key_b,
          const Tensor &log_eps, const Tensor &val_w, const Tensor &mu_w, const Tensor &log_rate, const Tensor &log_w,
          double eps, at::ScalarType cdt_)
        : B(x.size(0)), T(x.size(1)), D(x.size(2)), A(key_w.size(0)), Kc(conv_w.size(-1)), cd(code(cdt_)),
          M(static_cast<int64_t>(B) * T), cdt(cdt_), s(stream_of(x)), make(x) {
        x32 = x.contiguous();
        const Tensor nw = f32c(norm_w), cw = f32c(conv_w);
        h = make({B, T, D}, cdt);
        u = make({B, T, D}, cdt);
        rstd = make({B, T});
        check("ulm_norm_conv_fwd", ulm_norm_conv_fwd(x32.data_ptr(), ULM_F32, fp(nw), fp(cw), Kc, static_cast<float>(eps),
                                                     h.data_ptr(), cd, u.data_ptr(), cd, fpm(rstd), B, T, D, s));
        const Tensor kw = cast(key_w, cdt), vw = cast(val_w, cdt);
        mw = cast(mu_w, cdt);
        pre = at::mm(u.view({M, D}), kw.t());
        v = at::mm(h.view({M, D}), vw.t());
        if (key_b) b32 = f32c(*key_b);
        le = f32c(log_eps);
        denom = make({M});
        check("ulm_addr_fwd", ulm_addr_fwd(pre.data_ptr(), cd, fp(b32), fp(le), nullptr, fpm(denom), M, A, s));
        const Tensor lr = f32c(log_rate), lw = f32c(log_w);
        g1 = make({1});
        w32 = make({A});
        check("ulm_block_params", ulm_block_params(fp(lr), fp(lw), kLogWMin, kLogWMax, A, fpm(g1), fpm(w32), s));
    }
};

struct BlockFn : torch::autograd::Function<BlockFn> {
    static Tensor forward(AutogradContext *ctx, const Tensor &x, const Tensor &norm_w, const Tensor &conv_w,
                          const Tensor &key_w, const std::optional<Tensor> &key_b, const Tensor &log_eps,
                          const Tensor &val_w, const Tensor &mu_w, const Tensor &log_rate, const Tensor &log_w, double eps,
                          int64_t cdt) {
        at::AutoDispatchBelowAutograd guard;
        // the GEMM dtypes are explicit: autocast must not re-cast them
        c10::impl::ExcludeDispatchKeyGuard no_autocast(c10::autocast_dispatch_keyset);
        Block k(x, norm_w, conv_w, key_w, key_b, log_eps, val_w, mu_w, log_rate, log_w, eps,
                static_cast<at::ScalarType>(cdt));
        const size_t sb = ulm_fm_saved_bytes(k.B, k.T, k.A, k.D, k.cd);
        const size_t wb = ulm_block_fm_fwd_workspace_bytes(k.B, k.T, k.A, k.D);
        const Tensor saved = at::empty({static_cast<int64_t>(sb)}, k.make.opt.dtype(at::kByte));
        const Tensor qw = k.make({k.M, k.A}, k.cdt);
        Tensor y = k.make({k.M, k.D});
        {
            const Tensor ws = k.make.bytes(wb);
            check("ulm_block_fm_fwd",
                  ulm_block_fm_fwd(k.pre.data_ptr(), k.cd, fp(k.b32), fp(k.denom), k.v.data_ptr(), k.cd, fp(k.g1),
                                   fp(k.w32), qw.data_ptr(), k.cd, fp(k.x32), fpm(y), saved.data_ptr(), sb, ws.data_ptr(),
                                   wb, k.B, k.T, k.A, k.D, k.s));
        }
        k.v.reset();
        addmm_(y, qw, k.mw.t());
        ctx->save_for_backward({x, norm_w, conv_w, key_w, key_b.value_or(Tensor()), log_eps, val_w, mu_w, log_rate, log_w,
                                k.rstd, k.h, k.u, k.pre, k.denom, k.g1, k.w32, saved, qw});
        ctx->saved_data["cdt"] = cdt;
        ctx->set_materialize_grads(false);
        return y.view({k.B, k.T, k.D});
    }

    static variable_list backward(AutogradContext *ctx, variable_list grads) {
        variable_list out(12);
        if (!grads[0].defined()) return out;
        const auto sv = ctx->get_saved_variables();
        const Tensor &x = sv[0], &norm_w = sv[1], &conv_w = sv[2], &key_w = sv[3], &key_b = sv[4], &log_eps = sv[5],
                     &val_w = sv[6], &mu_w = sv[7], &log_rate = sv[8], &log_w = sv[9], &rstd = sv[10], &h = sv[11],
                     &u = sv[12], &pre = sv[13], &denom = sv[14], &g1 = sv[15], &w32 = sv[16], &saved = sv[17],
                     &qw = sv[18];
        if (!launches(grads, sv)) {
            using T1 = const Tensor &;
            using F = std::tuple<Tensor, Tensor, Tensor, Tensor, Tensor, Tensor, Tensor, Tensor, Tensor, Tensor>(
                T1, T1, T1, T1, T1, const std::optional<Tensor> &, T1, T1, T1, T1, T1, T1, T1, T1, T1, T1, T1, T1, T1, T1,
                at::ScalarType);
            const std::optional<Tensor> bias = key_b.defined() ? std::optional<Tensor>(key_b) : std::nullopt;
            auto [dx, dnw, dcw, dkey, dbias, dle, dval, dmu, dlr, dlw] = registered<F>("ulm::block_bwd").call(
                grads[0], x, norm_w, conv_w, key_w, bias, log_eps, val_w, mu_w, log_rate, log_w, rstd, h, u, pre, denom, g1,
                w32, saved, qw, static_cast<at::ScalarType>(ctx->saved_data["cdt"].toInt()));
            return {dx, dnw, dcw, dkey, bias ? dbias : Tensor(), dle, dval, dmu, dlr, dlw, Tensor(), Tensor()};
        }
        at::AutoDispatchBelowAutograd guard;
        c10::impl::ExcludeDispatchKeyGuard no_autocast(c10::autocast_dispatch_keyset);
        const auto cdt = static_cast<at::ScalarType>(ctx->saved_data["cdt"].toInt());
        const int B = x.size(0), T = x.size(1), D = x.size(2), A = key_w.size(0), Kc = conv_w.size(-1), cd = code(cdt);
        const int64_t M = static_cast<int64_t>(B) * T;
        void *s = stream_of(x);
        const Maker make(x);
        const Tensor x32 = x.contiguous(), nw = f32c(norm_w), cw = f32c(conv_w);
        const Tensor kw = cast(key_w, cdt), vw = cast(val_w, cdt), mw = cast(mu_w, cdt);
        const Tensor b32 = key_b.defined() ? f32c(key_b) : key_b;
        const Tensor le = f32c(log_eps), lr = f32c(log_rate), lw = f32c(log_w), dout = f32c(grads[0]);
        Tensor d16 = dout;
        if (cdt != at::kFloat) {
            d16 = make({B, T, D}, cdt);
            check("ulm_cast", ulm_cast(dout.data_ptr(), ULM_F32, d16.data_ptr(), cd, M * D, s));
        }
        const Tensor d2 = d16.view({M, D});
        Tensor dqw = at::mm(d2, mw);   // d(w q) = dout mu
        const Tensor dmu = wgrad(d2, qw, s);
        Tensor dr = make({M, A});
        const Tensor dv = make({M, D}, cdt), dg = make({1}), dw = make({A});
        {
            const size_t wb = ulm_fm_bwd_workspace_bytes(B, T, A, D, cd, saved.numel(), cd);
            const Tensor ws = make.bytes(wb);
            check("ulm_block_fm_bwd",
                  ulm_block_fm_bwd(pre.data_ptr(), cd, fp(b32), fp(denom), fp(g1), fp(w32), saved.data_ptr(), saved.numel(),
                                   cd, d16.data_ptr(), cd, dqw.data_ptr(), cd, fpm(dr), dv.data_ptr(), cd, fpm(dg), fpm(dw),
                                   ws.data_ptr(), wb, B, T, A, D, s));
        }
        dqw.reset();
        const Tensor dlr = make({1}), dlw = make({A});
        check("ulm_block_params_bwd",
              ulm_block_params_bwd(fp(lr), fp(lw), kLogWMin, kLogWMax, fp(dg), fp(dw), A, fpm(dlr), fpm(dlw), s));
        const Tensor dpre = at::empty_like(pre), dle = make({1});
        const Tensor dbias = key_b.defined() ? make({A}) : Tensor();
        {
            const size_t wb = ulm_addr_bwd_workspace_bytes(M, A);
            const Tensor ws = make.bytes(wb);
            check("ulm_addr_bwd", ulm_addr_bwd(pre.data_ptr(), cd, fp(b32), fp(le), nullptr, fp(denom), fp(dr),
                                               dpre.data_ptr(), dbias.defined() ? fpm(dbias) : nullptr, fpm(dle),
                                               ws.data_ptr(), wb, M, A, s));
        }
        dr.reset();
        const Tensor du = gemm(dpre, kw, at::kFloat), dkey = wgrad(dpre, u.view({M, D}), s);
        const Tensor dhv = gemm(dv, vw, at::kFloat), dval = wgrad(dv, h.view({M, D}), s);
        const Tensor dx = make({B, T, D}), dnw = make({D}), dcw = make({D, Kc});
        const size_t wb = ulm_norm_conv_bwd_workspace_bytes(B, T, D, Kc);
        if (wb == 0) throw py::value_error("ulm_norm_conv_bwd: unsupported D=" + std::to_string(D));
        const Tensor ws = make.bytes(wb);
        check("ulm_norm_conv_bwd",
              ulm_norm_conv_bwd(x32.data_ptr(), ULM_F32, fp(rstd), fp(nw), fp(cw), Kc, du.data_ptr(), ULM_F32, dhv.data_ptr(),
                                ULM_F32, fp(dout), fpm(dx), fpm(dnw), fpm(dcw), ws.data_ptr(), wb, B, T, D, s));
        return {dx, dnw, dcw.view(conv_w.sizes()), dkey, dbias, dle.reshape(log_eps.sizes()), dval, dmu,
                dlr.reshape(log_rate.sizes()), dlw, Tensor(), Tensor()};
    }
};

// the arguments of a block's forward or prefill, or ok false where the Python implementation decides
struct BlockArgs {
    Tensor x, norm_w, conv_w, key_w, log_eps, val_w, mu_w, log_rate, log_w;
    std::optional<Tensor> key_b;
    bool ok = false;

    explicit BlockArgs(const py::args &a) {
        if (a.size() != 10 || !plain_thread()) return;
        Tensor *to[] = {&x, &norm_w, &conv_w, &key_w, nullptr, &log_eps, &val_w, &mu_w, &log_rate, &log_w};
        for (int i = 0; i < 10; ++i) {
            if (i == 4 && a[4].is_none()) continue;
            const Tensor t = plain(a[i]);
            if (!t.defined() || (i > 0 && t.device() != x.device())) return;
            if (i == 4) key_b = t;
            else *to[i] = t;
        }
        if (x.dim() != 3 || x.scalar_type() != at::kFloat || x.numel() == 0 || key_w.dim() != 2 || key_w.size(0) == 0 ||
            mu_w.dim() != 2 || val_w.dim() != 2 || conv_w.dim() < 1)
            return;
        const int64_t D = x.size(2), A = key_w.size(0), Kc = conv_w.size(-1);
        if (key_w.size(1) != D || mu_w.size(0) != D || mu_w.size(1) != A || val_w.size(0) != D || val_w.size(1) != D ||
            log_w.dim() != 1 || log_w.size(0) != A || log_rate.numel() != 1 || log_eps.numel() != 1 || Kc < 1 || Kc > 8 ||
            conv_w.numel() != D * Kc || norm_w.numel() != D || (key_b && key_b->numel() != A))
            return;
        ok = true;
    }
};

bool gemm_dtype(at::ScalarType dt) { return dt == at::kFloat || dt == at::kBFloat16 || dt == at::kHalf; }

py::object block(double eps, at::ScalarType cdt, const py::args &args) {
    const BlockArgs a(args);
    if (!a.ok || !gemm_dtype(cdt)) return py::none();
    return py::cast(unlocked([&] {
        return BlockFn::apply(a.x, a.norm_w, a.conv_w, a.key_w, a.key_b, a.log_eps, a.val_w, a.mu_w, a.log_rate, a.log_w, eps,
                              static_cast<int64_t>(cdt));
    }));
}

// (out, S, c, r_prev, conv window, g, w) of kernel.block_prefill and UnifiedBlock.prefill; under no_grad
std::vector<Tensor> prefill_of(const BlockArgs &a, double eps, at::ScalarType cdt, size_t wb) {
    const int B = a.x.size(0), T = a.x.size(1), D = a.x.size(2), A = a.key_w.size(0);
    at::NoGradGuard no_grad;
    at::AutoDispatchBelowAutograd guard;
    c10::impl::ExcludeDispatchKeyGuard no_autocast(c10::autocast_dispatch_keyset);
    Block k(a.x, a.norm_w, a.conv_w, a.key_w, a.key_b, a.log_eps, a.val_w, a.mu_w, a.log_rate, a.log_w, eps, cdt);
    k.u.reset();
    const Tensor qw = k.make({k.M, A}, cdt), S = k.make({B, D, A}), c = k.make({B, A});
    Tensor y = k.make({k.M, D});
    {
        const Tensor ws = k.make.bytes(wb);
        check("ulm_block_fm_prefill",
              ulm_block_fm_prefill(k.pre.data_ptr(), k.cd, fp(k.b32), fp(k.denom), k.v.data_ptr(), k.cd, fp(k.g1), fp(k.w32),
                                   qw.data_ptr(), k.cd, fp(k.x32), fpm(y), fpm(S), fpm(c), ws.data_ptr(), wb, B, T, A, D, k.s));
    }
    k.v.reset();
    addmm_(y, qw, k.mw.t());
    // the address at the last position, the decode state's r_prev
    const Tensor last = k.pre.view({B, T, A}).select(1, T - 1).contiguous(), r_prev = k.make({B, A}), dn = k.make({B});
    check("ulm_addr_fwd", ulm_addr_fwd(last.data_ptr(), k.cd, fp(k.b32), fp(k.le), fpm(r_prev), fpm(dn), B, A, k.s));
    // the conv window: the last (up to) taps - 1 normalised inputs, oldest first
    const int kw = k.Kc - 1, n = std::min(kw, T);
    Tensor buf = n < kw ? at::zeros({B, D, kw}, k.make.opt.dtype(at::kFloat)) : k.make({B, D, kw});
    if (n > 0) buf.narrow(2, kw - n, n).copy_(k.h.narrow(1, T - n, n).transpose(1, 2));
    return {y.view({B, T, D}), S, c, r_prev, buf, k.g1, k.w32};
}

py::object prefill(double eps, at::ScalarType cdt, const py::args &args) {
    const BlockArgs a(args);
    if (!a.ok || !gemm_dtype(cdt)) return py::none();
    const size_t wb = ulm_block_fm_prefill_workspace_bytes(a.x.size(0), a.x.size(1), a.key_w.size(0), a.x.size(2), code(cdt));
    if (wb == 0) return py::none();
    return py::tuple(py::cast(unlocked([&] { return prefill_of(a, eps, cdt, wb); })));
}

// fp32 copies of tensors, one allocation and one launch, or None (UnifiedBlock._step_params' matrices)
py::object copies(const py::args &args) {
    if (!plain_thread()) return py::none();
    std::vector<Tensor> mats;
    for (const auto &a : args) {
        mats.push_back(plain(a));
        if (!mats.back().defined()) return py::none();
    }
    return py::cast(unlocked([&] {
        at::NoGradGuard no_grad;
        at::AutoDispatchBelowAutograd guard;
        std::vector<Tensor> flat, out;
        for (const Tensor &t : mats) flat.push_back(f32c(t).view(-1));
        const Tensor all = at::cat(flat);
        int64_t from = 0;
        for (const Tensor &t : mats) {
            out.push_back(all.narrow(0, from, t.numel()).view(t.sizes()));
            from += t.numel();
        }
        return out;
    }));
}

// ---- decode positions (kernel.decode_step)

// the state dicts' keys, made once
struct Keys {
    py::str params, np, state[6], param[9];
    Keys() : params("params"), np("np") {
        const char *s[] = {"buf", "S", "c", "r_prev", "pv", "pr"};
        const char *p[] = {"norm_w", "conv_w", "key_w", "key_b", "log_eps", "val_w", "mu_w", "w", "g"};
        for (int i = 0; i < 6; ++i) state[i] = py::str(s[i]);
        for (int i = 0; i < 9; ++i) param[i] = py::str(p[i]);
    }
};

py::object decode_step(const py::handle &x_, const py::list &states, const py::list &eps) {
    static const Keys &keys = *new Keys;   // outlives the interpreter's own teardown
    if (!plain_thread() || states.size() == 0 || eps.size() != states.size()) return py::none();
    const Tensor x = plain(x_);
    if (!x.defined() || x.dim() != 2 || x.scalar_type() != at::kFloat || !x.is_contiguous() || x.numel() == 0)
        return py::none();
    const int64_t N = x.size(0), D = x.size(1), J = ulm_decode_max_pending();
    int64_t A = 0, Kc = 0;
    size_t wb = 0;
    std::vector<ulm_decode_layer> layers(states.size());
    for (size_t i = 0; i < layers.size(); ++i) {
        if (!py::isinstance<py::dict>(states[i])) return py::none();
        PyObject *s = py::handle(states[i]).ptr(), *p = PyDict_GetItem(s, keys.params.ptr());
        if (!p || !PyDict_Check(p)) return py::none();
        auto get = [&](PyObject *d, const py::str &key) -> const at::TensorImpl * {
            PyObject *o = PyDict_GetItem(d, key.ptr());
            if (!o || !THPVariable_CheckExact(o)) return nullptr;
            const Tensor &t = THPVariable_Unpack(o);
            return t.defined() && t.is_cuda() && t.scalar_type() == at::kFloat && t.device() == x.device() &&
                           t.layout() == at::kStrided && t.is_contiguous() && !t.key_set().has_any(kNotPlain)
                       ? t.unsafeGetTensorImpl()
                       : nullptr;
        };
        if (i == 0) {
            const at::TensorImpl *S = get(s, keys.state[1]), *cw = get(p, keys.param[1]);
            if (!S || S->dim() != 3 || !cw || cw->dim() != 2) return py::none();
            A = S->size(2);
            Kc = cw->size(1);
            wb = ulm_decode_step_workspace_bytes(N, D, A, Kc);
            if (wb == 0) return py::none();
        }
        const std::vector<int64_t> shapes[15] = {{D}, {D, Kc}, {A, D}, {A}, {1}, {D, D}, {D, A}, {A}, {1},
                                                 {N, D, Kc - 1}, {N, D, A}, {N, A}, {N, A}, {J, N, D}, {J, N, A}};
        void *at[15];
        for (int j = 0; j < 15; ++j) {
            const at::TensorImpl *t = j < 9 ? get(p, keys.param[j]) : get(s, keys.state[j - 9]);
            if (!t || t->sizes() != at::IntArrayRef(shapes[j])) return py::none();
            at[j] = const_cast<void *>(t->data());
            // mu_w, w, S, c, r_prev, pr: 16-byte accesses
            if ((j == 6 || j == 7 || (j >= 10 && j <= 12) || j == 14) && reinterpret_cast<uintptr_t>(at[j]) % 16) return py::none();
        }
        PyObject *m = PyDict_GetItem(s, keys.np.ptr());
        const long held = m && PyLong_Check(m) ? PyLong_AsLong(m) : -1;
        if (held < 0 || held >= J) return py::none();
        auto f = [&](int j) { return static_cast<float *>(at[j]); };
        layers[i] = ulm_decode_layer{f(0), f(1), f(2), f(3), f(4), f(5), f(6), f(7), f(8), f(9), f(10), f(11), f(12), f(13),
                                     f(14), eps[i].cast<double>(), held};
    }
    const Tensor out = unlocked([&] {
        at::NoGradGuard no_grad;
        const Tensor y = at::empty_like(x), ws = Maker(x).bytes(wb);
        check("ulm_decode_step", ulm_decode_step(layers.data(), layers.size(), fp(x), fpm(y), ws.data_ptr(), wb, N, D, A, Kc,
                                                 stream_of(x)));
        return y;
    });
    for (size_t i = 0; i < layers.size(); ++i)
        states[i][keys.np] = py::int_((layers[i].pending + 1) % J);
    return py::cast(out);
}

}  // namespace

PYBIND11_MODULE(ulm_host, m) {
    m.def("memory", &memory);
    m.def("block", &block);
    m.def("prefill", &prefill);
    m.def("copies", &copies);
    m.def("decode_step", &decode_step);
}
