// The operators as torch::autograd::Function, over the C ABI of librwkv_hip.so: what the Python classes of rwkv_cuda_amd/*.py
// run.  Everything the reference's wrapper classes do on the host (checks, allocations, saved tensors, the launches of one
// direction) happens here in one call from Python and one from the autograd engine, which needs no interpreter for it: for the
// small shapes the host is what a step waits for.  With the classes in Python and the library called through ctypes, wkv4 B4 T512
// C768, forward + backward, took 147 us, of which the GPU worked 27; it takes 72 (most of it torch.autograd.grad and the hand-over
// to the engine's thread).  rwkv7 B1 T16 C2048, forward: 33 -> 9 us.
#include <torch/extension.h>
#include <ATen/hip/impl/HIPGuardImplMasqueradingAsCUDA.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>

#include "rwkv_hip.h"

namespace py = pybind11;

namespace {

using torch::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::Function;
using torch::autograd::variable_list;
using Guard = c10::hip::HIPGuardMasqueradingAsCUDA;

constexpr auto BF = torch::kBFloat16;
constexpr auto F32 = torch::kFloat32;
constexpr int64_t HEAD = 64, MAX_HEAD = 128, CHUNK7 = 16;

// the reference's wrappers use bare asserts (e.g. wkv6_state/run.py:84-100): an AssertionError keeps that contract.  Only
// called from the forwards, which run under the interpreter's lock.
void require(bool cond, const std::string& msg) {
    if (cond) return;
    PyErr_SetString(PyExc_AssertionError, msg.c_str());
    throw py::error_already_set();
}
std::string str(c10::ScalarType t) { return std::string("torch.") + (t == BF ? "bfloat16" : (t == F32 ? "float32" : c10::toString(t))); }
// one device, one dtype, contiguous
void check(std::initializer_list<std::pair<const Tensor*, const char*>> ts, c10::ScalarType dt, const Tensor& first) {
    for (const auto& t : ts) {
        const Tensor& x = *t.first;
        if (x.is_cuda() && x.scalar_type() == dt && x.is_contiguous() && x.device() == first.device()) continue;
        const std::string n = t.second;
        require(x.is_cuda() && first.is_cuda(), "tensors must live on a HIP device: there is no CPU path");
        require(x.scalar_type() == dt, n + ".dtype must be " + str(dt) + ", got " + str(x.scalar_type()));
        require(x.is_contiguous(), n + " must be contiguous");
        require(false, n + " is on " + x.device().str() + ", expected " + first.device().str());
    }
}
void check_head(int64_t C, int64_t H) {
    require(H > 0 && C % H == 0 && C / H <= MAX_HEAD, "C must be a multiple of H with a head size of at most 128");
}
// the package's own error type, in either direction: the engine's threads, which run the backwards, do not hold the interpreter's lock
[[noreturn]] void fail(const std::string& msg) {
    const py::gil_scoped_acquire lock;
    PyErr_SetString(py::module_::import("rwkv_cuda_amd._lib").attr("RwkvHipError").ptr(), msg.c_str());
    throw py::error_already_set();
}
// sizes as the C ABI takes them
int i32(int64_t x) {
    if (x <= 0 || x > std::numeric_limits<int>::max()) fail("size " + std::to_string(x) + " is outside 1 .. 2147483647");
    return static_cast<int>(x);
}
struct Dims { int B, T, C, H; };
Dims dims(int64_t B, int64_t T, int64_t C, int64_t H) { return {i32(B), i32(T), i32(C), i32(H)}; }

void* stream_of(const Tensor& t) { return static_cast<void*>(c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(t.device().index()).stream()); }
void ok(int status) {
    if (status == RWKV_OK) return;
    std::string msg = "librwkv_hip: status " + std::to_string(status) + ": " + rwkv_strerror(status);
    if (status == RWKV_ERR_LAUNCH) msg += " (hipError " + std::to_string(rwkv_last_hip_error()) + ")";
    fail(msg);
}

// typed pointers; an undefined tensor is NULL
struct Ptr {
    void* p;
    template <class T> operator T*() const { return static_cast<T*>(p); }
};
Ptr P(const Tensor& t) { return {t.defined() ? t.data_ptr() : nullptr}; }
Tensor bytes(const Tensor& like, size_t n) { return at::empty({static_cast<int64_t>(n)}, like.options().dtype(torch::kUInt8)); }
bool wants_grad(std::initializer_list<const Tensor*> ts) {
    if (!c10::GradMode::is_enabled()) return false;
    for (const Tensor* t : ts) if (t->requires_grad()) return true;
    return false;
}
void put(AutogradContext* ctx, std::initializer_list<std::pair<const char*, int64_t>> xs) { for (const auto& x : xs) ctx->saved_data[x.first] = x.second; }
int64_t get(AutogradContext* ctx, const char* n) { return ctx->saved_data[n].toInt(); }
Dims get_dims(AutogradContext* ctx) { return dims(get(ctx, "B"), get(ctx, "T"), get(ctx, "C"), get(ctx, "H")); }
const Tensor NONE;

// --------------------------------------------------------------------------------------------- wkv (wkv/run.py:89-117)
struct Wkv4 : Function<Wkv4> {
    static Tensor forward(AutogradContext* ctx, int64_t B, int64_t T, int64_t C, const Tensor& w_, const Tensor& u_, const Tensor& k_, const Tensor& v_) {
        const Tensor w = w_.contiguous(), u = u_.contiguous(), k = k_.contiguous(), v = v_.contiguous();
        check({{&w, "w"}, {&u, "u"}, {&k, "k"}, {&v, "v"}}, F32, w);
        require(k.numel() == B * T * C && v.numel() == k.numel() && w.numel() == C && u.numel() == C, "shape mismatch");
        const Guard guard(w.device());
        Tensor y = at::empty({B, T, C}, k.options());
        // w = -exp(w) of the reference wrapper (:95) happens inside the kernels
        ok(rwkv_wkv4raw_forward(stream_of(w), i32(B), i32(T), i32(C), P(w), P(u), P(k), P(v), P(y)));
        ctx->save_for_backward({w, u, k, v});
        put(ctx, {{"B", B}, {"T", T}, {"C", C}});
        return y;
    }
    static variable_list backward(AutogradContext* ctx, variable_list g) {
        const auto s = ctx->get_saved_variables();
        const Tensor &w = s[0], &u = s[1], &k = s[2], &v = s[3], gy = g[0].contiguous();
        const int B = i32(get(ctx, "B")), T = i32(get(ctx, "T")), C = i32(get(ctx, "C"));
        const Guard guard(w.device());
        Tensor gw = at::empty({C}, w.options()), gu = at::empty({C}, w.options());      // summed over the batch by the library (:115-116)
        Tensor gk = at::empty({B, T, C}, w.options()), gv = at::empty({B, T, C}, w.options());
        const size_t n = rwkv_wkv4raw_backward_workspace_bytes(B, T, C);
        Tensor ws = bytes(w, n);
        ok(rwkv_wkv4raw_backward(stream_of(w), B, T, C, P(w), P(u), P(k), P(v), P(gy), P(gw), P(gu), P(gk), P(gv), P(ws), n));
        return {NONE, NONE, NONE, gw, gu, gk, gv};
    }
};
Tensor wkv4_op(int64_t B, int64_t T, int64_t C, const Tensor& w, const Tensor& u, const Tensor& k, const Tensor& v) { return Wkv4::apply(B, T, C, w, u, k, v); }

// --------------------------------------------------------------------------------------------- depthwise_conv1d (run.py:76-102)
constexpr int64_t T_MAX = 4096;
struct TimeX : Function<TimeX> {
    static Tensor forward(AutogradContext* ctx, const Tensor& w_, const Tensor& k_, int64_t B, int64_t C, int64_t T, double eps) {
        require(T % 4 == 0 && T <= T_MAX, "require T % 4 == 0 and T <= T_MAX");
        const Tensor w = w_.contiguous(), k = k_.contiguous();
        check({{&w, "w"}, {&k, "k"}}, F32, w);
        require(w.numel() == C * T && k.numel() == B * C * T, "shape mismatch");
        const Guard guard(w.device());
        Tensor x = at::empty({B, C, T}, k.options());
        ok(rwkv_timex_forward(stream_of(w), P(w), P(k), P(x), static_cast<float>(eps), i32(B), i32(C), i32(T)));
        ctx->save_for_backward({w, k});
        put(ctx, {{"B", B}, {"T", T}, {"C", C}});
        return x;
    }
    static variable_list backward(AutogradContext* ctx, variable_list g) {
        const auto s = ctx->get_saved_variables();
        const Tensor &w = s[0], &k = s[1], gx = g[0].contiguous();
        const int B = i32(get(ctx, "B")), T = i32(get(ctx, "T")), C = i32(get(ctx, "C"));
        const Guard guard(w.device());
        Tensor gk = at::empty({B, C, T}, k.options()), gw = at::empty({C, T}, k.options());      // the sum over the batch of run.py:102 happens in the library
        const size_t n = rwkv_timex_backward_ws_bytes(B, C, T);
        const Tensor ws = n > 0 ? bytes(k, n) : Tensor();
        ok(rwkv_timex_backward_ws(stream_of(w), P(w), P(k), P(gx), P(gw), P(gk), B, C, T, P(ws), n));
        return {gw, gk, NONE, NONE, NONE, NONE};
    }
};
Tensor timex_op(const Tensor& w, const Tensor& k, int64_t B, int64_t C, int64_t T, double eps) { return TimeX::apply(w, k, B, C, T, eps); }

// --------------------------------------------------------------------------------------------- wkv5, fp32 (wkv5/run.py:469-504)
struct Wkv5F32 : Function<Wkv5F32> {
    static Tensor forward(AutogradContext* ctx, int64_t B, int64_t T, int64_t C, int64_t H, const Tensor& r, const Tensor& k, const Tensor& v,
                          const Tensor& w, const Tensor& u, int64_t flags, bool grad) {
        check({{&r, "r"}, {&k, "k"}, {&v, "v"}, {&w, "w"}, {&u, "u"}}, F32, r);
        check_head(C, H);
        require(r.numel() == B * T * C && k.numel() == r.numel() && v.numel() == r.numel() && w.numel() == C && u.numel() == C, "shape mismatch");
        const Guard guard(r.device());
        const Dims d = dims(B, T, C, H);
        Tensor y = at::empty({B, T, C}, r.options());
        // head size 64: the raw decay and the sums over the batch (:482-483,:497-501) are the library's; other head sizes, and
        // the sequential kernels on request, sit behind the reference's own signature
        const bool chunked = C == H * HEAD && !(flags & RWKV_FLAG_SWEEPS);
        if (chunked) {
            const size_t n = grad ? rwkv_wkv5f32s_saved_bytes(d.B, d.T, d.C, d.H) : 0;
            const Tensor saved = grad ? bytes(r, n) : Tensor();
            const size_t nw = rwkv_wkv5f32s_forward_workspace_bytes(d.B, d.T, d.C, d.H);
            const Tensor ws = nw > 0 ? bytes(r, nw) : Tensor();
            ok(rwkv_wkv5f32s_forward_ws(stream_of(r), d.B, d.T, d.C, d.H, P(r), P(k), P(v), P(w), P(u), P(y), P(saved), n, P(ws), nw));
            if (grad) ctx->save_for_backward({r, k, v, w, u, saved});
        } else {
            const Tensor ew = w.exp().neg_(), eew = ew.exp();
            ok(rwkv_wkv5f32_forward(stream_of(r), d.B, d.T, d.C, d.H, P(r), P(k), P(v), P(eew), P(u), P(y)));
            if (grad) ctx->save_for_backward({r, k, v, w, u, eew, ew});
        }
        put(ctx, {{"B", B}, {"T", T}, {"C", C}, {"H", H}, {"chunked", chunked}});
        return y;
    }
    static variable_list backward(AutogradContext* ctx, variable_list g) {
        const auto s = ctx->get_saved_variables();
        const Tensor &r = s[0], &k = s[1], &v = s[2], &w = s[3], &u = s[4], gy = g[0].contiguous();
        const Dims d = get_dims(ctx);
        const Guard guard(r.device());
        const auto o = r.options();
        Tensor gr = at::empty({d.B, d.T, d.C}, o), gk = at::empty({d.B, d.T, d.C}, o), gv = at::empty({d.B, d.T, d.C}, o), gw, gu;
        if (get(ctx, "chunked")) {
            const Tensor& saved = s[5];
            gw = at::empty(w.sizes(), o); gu = at::empty(u.sizes(), o);
            const size_t n = rwkv_wkv5f32s_backward_workspace_bytes(d.B, d.T, d.C, d.H);
            Tensor ws = bytes(r, n);
            ok(rwkv_wkv5f32s_backward(stream_of(r), d.B, d.T, d.C, d.H, P(r), P(k), P(v), P(w), P(u), P(gy), P(gr), P(gk), P(gv), P(gw), P(gu),
                                      P(saved), saved.numel(), P(ws), n));
        } else {
            Tensor pw = at::empty({d.B, d.C}, o), pu = at::empty({d.B, d.C}, o);
            ok(rwkv_wkv5f32_backward(stream_of(r), d.B, d.T, d.C, d.H, P(r), P(k), P(v), P(s[5]), P(s[6]), P(u), P(gy), P(gr), P(gk), P(gv), P(pw), P(pu)));
            gw = pw.sum(0).view(w.sizes()); gu = pu.sum(0).view(u.sizes());
        }
        return {NONE, NONE, NONE, NONE, gr, gk, gv, gw, gu, NONE, NONE};
    }
};
Tensor wkv5_f32_op(int64_t B, int64_t T, int64_t C, int64_t H, const Tensor& r, const Tensor& k, const Tensor& v, const Tensor& w, const Tensor& u, int64_t flags) {
    return Wkv5F32::apply(B, T, C, H, r, k, v, w, u, flags, wants_grad({&r, &k, &v, &w, &u}));
}

// --------------------------------------------------------------------------------------------- wkv5a, fp32 (wkv5a/run.py:100-154)
struct Wkv5A : Function<Wkv5A> {
    static Tensor forward(AutogradContext* ctx, const Tensor& r, const Tensor& k, const Tensor& v, const Tensor& w1, const Tensor& u1,
                          const Tensor& w2, const Tensor& u2, int64_t flags, bool grad) {
        check({{&r, "r"}, {&k, "k"}, {&v, "v"}, {&w1, "w1"}, {&u1, "u1"}, {&w2, "w2"}, {&u2, "u2"}}, F32, r);
        require(r.dim() == 3 && w1.dim() == 2, "r,k,v are [B,T,C]; w1,u1,w2,u2 are [H,N]");
        const int64_t B = r.size(0), T = r.size(1), C = r.size(2), H = w1.size(0);
        require(H > 0 && C % H == 0 && w1.size(1) == C / H && C / H <= MAX_HEAD, "w1 is [H, C/H] with a head size of at most 128");
        require(k.sizes() == r.sizes() && v.sizes() == r.sizes(), "shape mismatch");
        require(u1.sizes() == w1.sizes() && w2.sizes() == w1.sizes() && u2.sizes() == w1.sizes(), "shape mismatch");
        const Guard guard(r.device());
        const Dims d = dims(B, T, C, H);
        Tensor y = at::empty({B, T, C}, r.options());
        const bool chunked = C == H * HEAD && !(flags & RWKV_FLAG_SWEEPS);
        if (chunked) {
            const size_t n = grad ? rwkv_wkv5as_saved_bytes(d.B, d.T, d.C, d.H) : 0;
            const Tensor saved = grad ? bytes(r, n) : Tensor();
            const size_t nw = rwkv_wkv5as_forward_workspace_bytes(d.B, d.T, d.C, d.H);
            const Tensor ws = nw > 0 ? bytes(r, nw) : Tensor();
            ok(rwkv_wkv5as_forward_ws(stream_of(r), d.B, d.T, d.C, d.H, P(r), P(k), P(v), P(w1), P(u1), P(w2), P(u2), P(y), P(saved), n, P(ws), nw));
            if (grad) ctx->save_for_backward({r, k, v, w1, u1, w2, u2, saved});
        } else {
            const Tensor ew1 = w1.exp().neg_(), eew1 = ew1.exp(), ew2 = w2.exp().neg_(), eew2 = ew2.exp();
            ok(rwkv_wkv5a_forward(stream_of(r), d.B, d.T, d.C, d.H, P(r), P(k), P(v), P(eew1), P(u1), P(eew2), P(u2), P(y)));
            if (grad) ctx->save_for_backward({r, k, v, w1, u1, w2, u2, eew1, ew1, eew2, ew2});
        }
        put(ctx, {{"B", B}, {"T", T}, {"C", C}, {"H", H}, {"chunked", chunked}});
        return y;
    }
    static variable_list backward(AutogradContext* ctx, variable_list g) {
        const auto s = ctx->get_saved_variables();
        const Tensor &r = s[0], &k = s[1], &v = s[2], &w1 = s[3], &u1 = s[4], &w2 = s[5], &u2 = s[6], gy = g[0].contiguous();
        const Dims d = get_dims(ctx);
        const Guard guard(r.device());
        const auto o = r.options();
        Tensor gr = at::empty({d.B, d.T, d.C}, o), gk = at::empty({d.B, d.T, d.C}, o), gv = at::empty({d.B, d.T, d.C}, o);
        Tensor gp[4];                                     // w1, u1, w2, u2
        if (get(ctx, "chunked")) {
            const Tensor& saved = s[7];
            for (Tensor& x : gp) x = at::empty(w1.sizes(), o);                      // summed over the batch by the library (:150-153)
            const size_t n = rwkv_wkv5as_backward_workspace_bytes(d.B, d.T, d.C, d.H);
            Tensor ws = bytes(r, n);
            ok(rwkv_wkv5as_backward(stream_of(r), d.B, d.T, d.C, d.H, P(r), P(k), P(v), P(w1), P(u1), P(w2), P(u2), P(gy), P(gr), P(gk), P(gv),
                                    P(gp[0]), P(gp[1]), P(gp[2]), P(gp[3]), P(saved), saved.numel(), P(ws), n));
        } else {
            for (Tensor& x : gp) x = at::empty({d.B, d.C}, o);
            ok(rwkv_wkv5a_backward(stream_of(r), d.B, d.T, d.C, d.H, P(r), P(k), P(v), P(s[7]), P(s[8]), P(u1), P(s[9]), P(s[10]), P(u2), P(gy),
                                   P(gr), P(gk), P(gv), P(gp[0]), P(gp[1]), P(gp[2]), P(gp[3])));
            for (Tensor& x : gp) x = x.sum(0).view(w1.sizes());
        }
        return {gr, gk, gv, gp[0], gp[1], gp[2], gp[3], NONE, NONE};
    }
};
Tensor wkv5a_op(const Tensor& r, const Tensor& k, const Tensor& v, const Tensor& w1, const Tensor& u1, const Tensor& w2, const Tensor& u2, int64_t flags) {
    return Wkv5A::apply(r, k, v, w1, u1, w2, u2, flags, wants_grad({&r, &k, &v, &w1, &u1, &w2, &u2}));
}

// --------------------------------------------------------------------------------------------- wkv5, bf16 (wkv5_bf16/run.py:44-88)
struct Wkv5Bf16 : Function<Wkv5Bf16> {
    static Tensor forward(AutogradContext* ctx, int64_t B, int64_t T, int64_t C, int64_t H, const Tensor& r, const Tensor& k, const Tensor& v,
                          const Tensor& w, const Tensor& u, int64_t flags, bool grad) {
        check({{&r, "r"}, {&k, "k"}, {&v, "v"}, {&w, "w"}, {&u, "u"}}, BF, r);
        check_head(C, H);
        require(r.numel() == B * T * C && k.numel() == r.numel() && v.numel() == r.numel() && w.numel() == C && u.numel() == C, "shape mismatch");
        const Guard guard(r.device());
        const Dims d = dims(B, T, C, H);
        // ew = -exp(w.float()), eew = exp(ew) (:63-64) are made by the library into `decay` = [eew | ew]
        Tensor decay = at::empty({2 * C}, r.options().dtype(F32)), y = at::empty({B, T, C}, r.options());
        const bool whole = C == H * MAX_HEAD && flags == 0;
        const size_t n = C == H * HEAD || whole ? rwkv_wkv5s_saved_bytes(d.B, d.T, d.C, d.H) : 0;
        if (n > 0) {
            // head sizes 64 and 128: one forward and one reverse sweep; the forward keeps the state entering every 64th token
            // (at 128 only if a backward can follow)
            const bool keep = grad || !whole;
            const Tensor saved = keep ? bytes(r, n) : Tensor();
            const size_t nw = rwkv_wkv5s_blocks_workspace_bytes(d.B, d.T, d.C, d.H, 0);
            const Tensor ws = nw > 0 ? bytes(r, nw) : Tensor();
            ok(rwkv_wkv5s_forward_ws(stream_of(r), d.B, d.T, d.C, d.H, P(r), P(k), P(v), P(w), P(u), P(y), P(decay), P(saved), keep ? n : 0, P(ws), nw, flags));
            if (keep) ctx->save_for_backward({r, k, v, decay, u, w, saved});
        } else {
            // heads of 128 channels with options run as four heads of 64 whose fp32 terms need scratch; every other size needs none
            const size_t nf = rwkv_wkv5_forward_workspace_bytes(d.B, d.T, d.C, d.H);
            Tensor ws = bytes(r, nf < 16 ? 16 : nf);
            ok(rwkv_wkv5raw_forward_ws(stream_of(r), d.B, d.T, d.C, d.H, P(r), P(k), P(v), P(w), P(u), P(y), P(decay), P(ws), nf, flags));
            ctx->save_for_backward({r, k, v, decay, u});
        }
        put(ctx, {{"B", B}, {"T", T}, {"C", C}, {"H", H}, {"flags", flags}});
        return y;
    }
    static variable_list backward(AutogradContext* ctx, variable_list g) {
        const auto s = ctx->get_saved_variables();
        const Tensor &r = s[0], &k = s[1], &v = s[2], &decay = s[3], &u = s[4], gy = g[0].contiguous();
        const Dims d = get_dims(ctx);
        const unsigned flags = static_cast<unsigned>(get(ctx, "flags"));
        const Guard guard(r.device());
        const auto o = r.options();
        Tensor gr = at::empty({d.B, d.T, d.C}, o), gk = at::empty({d.B, d.T, d.C}, o), gv = at::empty({d.B, d.T, d.C}, o);
        Tensor gw = at::empty({d.H, d.C / d.H}, o), gu = at::empty({d.H, d.C / d.H}, o);       // summed over the batch by the library (:86-87)
        if (s.size() > 5) {
            const Tensor &w = s[5], &saved = s[6];
            // (at head size 128 without options the per-batch rows of gw and gu are all, and what blocks of time take)
            const size_t nb = rwkv_wkv5s_blocks_workspace_bytes(d.B, d.T, d.C, d.H, 1);
            const size_t n = nb > 0 ? nb : d.C == d.H * MAX_HEAD ? 4 * static_cast<size_t>(d.B) * d.C : rwkv_wkv5s_backward_workspace_bytes(d.B, d.T, d.C, d.H);
            Tensor ws = bytes(r, n);
            ok(rwkv_wkv5s_backward(stream_of(r), d.B, d.T, d.C, d.H, P(r), P(k), P(v), P(w), P(decay), P(u), P(gy), P(gr), P(gk), P(gv), P(gw), P(gu),
                                   P(saved), saved.numel(), P(ws), n, flags));
        } else {
            const size_t n = rwkv_wkv5raw_backward_workspace_bytes(d.B, d.T, d.C, d.H);
            Tensor ws = bytes(r, n);
            ok(rwkv_wkv5raw_backward(stream_of(r), d.B, d.T, d.C, d.H, P(r), P(k), P(v), P(decay), P(u), P(gy), P(gr), P(gk), P(gv), P(gw), P(gu),
                                     P(ws), n, flags));
        }
        return {NONE, NONE, NONE, NONE, gr, gk, gv, gw, gu, NONE, NONE};
    }
};
Tensor wkv5_bf16_op(int64_t B, int64_t T, int64_t C, int64_t H, const Tensor& r, const Tensor& k, const Tensor& v, const Tensor& w, const Tensor& u, int64_t flags) {
    return Wkv5Bf16::apply(B, T, C, H, r, k, v, w, u, flags, wants_grad({&r, &k, &v, &w, &u}));
}

// ------------------------------------------------------- wkv6 and wkv6_state, bf16 (wkv6/run.py:128-170, wkv6_state/run.py:80-124)
// (s: the initial state, undefined for wkv6; the saved variables are taken once: hooks on them run per taking, and a checkpoint
// refuses a second one)
variable_list wkv6_grads(AutogradContext* ctx, const Tensor& gy_, bool state) {
    const auto s = ctx->get_saved_variables();
    const Tensor &r = s[0], &k = s[1], &v = s[2], &w = s[3], &u = s[4], &saved = s[5], s0 = state ? s[6] : Tensor(), gy = gy_.contiguous();
    const Dims d = get_dims(ctx);
    const Guard guard(r.device());
    const auto o = r.options();
    Tensor gr = at::empty({d.B, d.T, d.C}, o), gk = at::empty({d.B, d.T, d.C}, o), gv = at::empty({d.B, d.T, d.C}, o), gw = at::empty({d.B, d.T, d.C}, o);
    const int64_t N = d.C / d.H;
    Tensor gu = at::empty({d.H, N}, o), gs = s0.defined() ? at::empty({d.B, d.H, N, N}, o) : Tensor();    // gu summed over the batch by the library (:169, :123)
    const size_t n = rwkv_wkv6f_backward_saved_workspace_bytes(d.B, d.T, d.C, d.H);
    Tensor ws = bytes(r, n);
    ok(rwkv_wkv6f_backward_saved(stream_of(r), d.B, d.T, d.C, d.H, P(r), P(k), P(v), P(w), P(u), P(s0), P(gy), P(gr), P(gk), P(gv), P(gw), P(gu), P(gs),
                                 saved.numel() > 0 ? P(saved) : Ptr{nullptr}, saved.numel(), P(ws), n, static_cast<unsigned>(get(ctx, "flags"))));
    return {NONE, NONE, NONE, NONE, gr, gk, gv, gw, gu, gs, NONE};
}
Tensor wkv6_run(AutogradContext* ctx, int64_t B, int64_t T, int64_t C, int64_t H, const Tensor& r, const Tensor& k, const Tensor& v, const Tensor& w,
                const Tensor& u, const Tensor& s, int64_t flags) {
    check({{&r, "r"}, {&k, "k"}, {&v, "v"}, {&w, "w"}, {&u, "u"}}, BF, r);
    check_head(C, H);
    require(r.numel() == B * T * C && k.numel() == r.numel() && v.numel() == r.numel() && w.numel() == r.numel() && u.numel() == C, "shape mismatch");
    const Guard guard(r.device());
    const Dims d = dims(B, T, C, H);
    Tensor y = at::empty({B, T, C}, r.options());
    // the forward keeps the state entering every 64th token for the backward's single reverse sweep (no bytes for head sizes
    // and options that take the two-sweep kernels)
    const size_t n = rwkv_wkv6f_saved_bytes(d.B, d.T, d.C, d.H);
    Tensor saved = bytes(r, n);
    ok(rwkv_wkv6f_forward(stream_of(r), d.B, d.T, d.C, d.H, P(r), P(k), P(v), P(w), P(u), P(s), P(y), n > 0 ? P(saved) : Ptr{nullptr}, n,
                          static_cast<unsigned>(flags)));
    if (s.defined()) ctx->save_for_backward({r, k, v, w, u, saved, s});
    else ctx->save_for_backward({r, k, v, w, u, saved});
    put(ctx, {{"B", B}, {"T", T}, {"C", C}, {"H", H}, {"flags", flags}});
    return y;
}
struct Wkv6 : Function<Wkv6> {
    static Tensor forward(AutogradContext* ctx, int64_t B, int64_t T, int64_t C, int64_t H, const Tensor& r, const Tensor& k, const Tensor& v,
                          const Tensor& w, const Tensor& u, int64_t flags) {
        return wkv6_run(ctx, B, T, C, H, r, k, v, w, u, NONE, flags);
    }
    static variable_list backward(AutogradContext* ctx, variable_list g) {
        variable_list x = wkv6_grads(ctx, g[0], false);
        x.erase(x.begin() + 9);
        return x;
    }
};
struct Wkv6State : Function<Wkv6State> {
    static Tensor forward(AutogradContext* ctx, int64_t B, int64_t T, int64_t C, int64_t H, const Tensor& r, const Tensor& k, const Tensor& v,
                          const Tensor& w, const Tensor& u, const Tensor& s, int64_t flags) {
        check({{&s, "s"}}, BF, r);
        check_head(C, H);
        require(s.numel() == B * C * (C / H), "shape mismatch");
        return wkv6_run(ctx, B, T, C, H, r, k, v, w, u, s, flags);
    }
    static variable_list backward(AutogradContext* ctx, variable_list g) { return wkv6_grads(ctx, g[0], true); }
};
Tensor wkv6_op(int64_t B, int64_t T, int64_t C, int64_t H, const Tensor& r, const Tensor& k, const Tensor& v, const Tensor& w, const Tensor& u, int64_t flags) {
    return Wkv6::apply(B, T, C, H, r, k, v, w, u, flags);
}
Tensor wkv6_state_op(int64_t B, int64_t T, int64_t C, int64_t H, const Tensor& r, const Tensor& k, const Tensor& v, const Tensor& w, const Tensor& u,
                  const Tensor& s, int64_t flags) {
    return Wkv6State::apply(B, T, C, H, r, k, v, w, u, s, flags);
}

// --------------------------------------------- rwkv7 clamp-w (rwkv7_cuda_benchmark_state_passing.py:75-103, _state.py:75-102, .py:76-100)
// One body for the three siblings: s0 may be undefined (no state), passing = the final state is an output too.  r is
// [B,T,H*64] (flat: the functions) or [B,T,H,64] (the classes), the others either (the same memory); y has the shape of r, with
// `passing` always [B,T,H*64].  The checkpoint tensors `s` and `sa` are scratch
// whose layout belongs to the library.  The backward must run with the flags of the forward (the kernel families lay `s` out
// differently), so they ride on the context.
variable_list rwkv7_run(AutogradContext* ctx, const Tensor& s0, const Tensor& r, const Tensor& w, const Tensor& k, const Tensor& v, const Tensor& a,
                        const Tensor& b, int64_t flags, bool passing, bool flat, bool grad) {
    const auto dt = r.scalar_type();
    require(dt == BF || dt == F32, "r.dtype must be bfloat16 or float32, got " + str(dt));
    require(r.dim() == (flat ? 3 : 4), flat ? "r must be [B,T,H*64]" : "r must be [B,T,H,64]");
    require(flat ? r.size(2) % HEAD == 0 : r.size(3) == HEAD, "head size must be 64");
    const int64_t B = r.size(0), T = r.size(1), H = flat ? r.size(2) / HEAD : r.size(2);
    require(T % CHUNK7 == 0, "T must be a multiple of CHUNK_LEN");
    check({{&r, "r"}, {&w, "w"}, {&k, "k"}, {&v, "v"}, {&a, "a"}, {&b, "b"}}, dt, r);
    for (const Tensor* x : {&w, &k, &v, &a, &b}) require(x->numel() == r.numel(), "shape mismatch");
    if (s0.defined()) {
        check({{&s0, "s0"}}, F32, r);
        require(s0.sizes() == at::IntArrayRef({B, H, HEAD, HEAD}), "s0 must be [B,H,N,N] on the same device");
    }
    const Guard guard(r.device());
    const int b_ = i32(B), t_ = i32(T), h_ = i32(H);
    const auto f32 = r.options().dtype(F32);
    Tensor y = flat || passing ? at::empty({B, T, H * HEAD}, r.options()) : at::empty({B, T, H, HEAD}, r.options());
    Tensor sT = passing ? at::empty({B, H, HEAD, HEAD}, f32) : Tensor();
    void* st = stream_of(r);
    const bool sweeps = flags & RWKV_FLAG_SWEEPS;
    const size_t n = sweeps ? 0 : rwkv7_workspace_bytes(b_, t_, h_, 0);
    const Tensor ws = n > 0 ? bytes(r, n) : Tensor();
    if (!grad && !sweeps) {
        // no backward can follow: nothing is kept for one
        ok(rwkv7_forward_ws(st, b_, t_, h_, dt == F32, P(s0), P(r), P(w), P(k), P(v), P(a), P(b), P(y), P(sT), nullptr, nullptr, P(ws), n));
        if (passing) return {y, sT};
        return {y};
    }
    Tensor s = at::empty({B, H, T / CHUNK7, HEAD, HEAD}, f32), sa = at::empty({B, T, H, HEAD}, f32);
    if (!sweeps)
        ok(rwkv7_forward_ws(st, b_, t_, h_, dt == F32, P(s0), P(r), P(w), P(k), P(v), P(a), P(b), P(y), P(sT), P(s), P(sa), P(ws), n));
    else if (dt == BF)
        ok(rwkv7_statepassing_forward_ex(st, b_, t_, h_, P(s0), P(r), P(w), P(k), P(v), P(a), P(b), P(y), P(sT), P(s), P(sa), static_cast<unsigned>(flags)));
    else
        ok(rwkv7_statepassing_forward_f32_ex(st, b_, t_, h_, P(s0), P(r), P(w), P(k), P(v), P(a), P(b), P(y), P(sT), P(s), P(sa), static_cast<unsigned>(flags)));
    ctx->save_for_backward({r, w, k, v, a, b, s, sa});
    put(ctx, {{"B", B}, {"T", T}, {"H", H}, {"flags", flags}});
    if (passing) return {y, sT};
    return {y};
}
// ds0 (undefined without a state), dr, dw, dk, dv, da, db; dsT undefined: no gradient comes back for a final state
variable_list rwkv7_grads(AutogradContext* ctx, const Tensor& dy_, const Tensor& dsT_, bool state) {
    const auto x = ctx->get_saved_variables();
    const Tensor &r = x[0], &w = x[1], &k = x[2], &v = x[3], &a = x[4], &b = x[5], &s = x[6], &sa = x[7];
    const Tensor dy = dy_.contiguous(), dsT = dsT_.defined() ? dsT_.contiguous() : Tensor();
    const int B = i32(get(ctx, "B")), T = i32(get(ctx, "T")), H = i32(get(ctx, "H"));
    const Guard guard(r.device());
    Tensor ds0 = state ? at::empty({B, H, HEAD, HEAD}, r.options().dtype(F32)) : Tensor(), d[6];
    for (int i = 0; i < 6; ++i) d[i] = at::empty(x[i].sizes(), r.options());       // (each input may have come in either shape)
    void* st = stream_of(r);
    if (!(get(ctx, "flags") & RWKV_FLAG_SWEEPS)) {
        const size_t n = rwkv7_workspace_bytes(B, T, H, 1);
        const Tensor ws = n > 0 ? bytes(r, n) : Tensor();
        ok(rwkv7_backward_ws(st, B, T, H, r.scalar_type() == F32, P(r), P(w), P(k), P(v), P(a), P(b), P(dy), P(dsT), P(s), P(sa), P(ds0), P(d[0]), P(d[1]),
                             P(d[2]), P(d[3]), P(d[4]), P(d[5]), P(ws), n));
    } else if (r.scalar_type() == BF)
        ok(rwkv7_statepassing_backward_ex(st, B, T, H, P(r), P(w), P(k), P(v), P(a), P(b), P(dy), P(dsT), P(s), P(sa), P(ds0), P(d[0]), P(d[1]), P(d[2]),
                                          P(d[3]), P(d[4]), P(d[5]), static_cast<unsigned>(get(ctx, "flags"))));
    else
        ok(rwkv7_statepassing_backward_f32_ex(st, B, T, H, P(r), P(w), P(k), P(v), P(a), P(b), P(dy), P(dsT), P(s), P(sa), P(ds0), P(d[0]), P(d[1]), P(d[2]),
                                              P(d[3]), P(d[4]), P(d[5]), static_cast<unsigned>(get(ctx, "flags"))));
    return {ds0, d[0], d[1], d[2], d[3], d[4], d[5], NONE, NONE};
}
struct Rwkv7Passing : Function<Rwkv7Passing> {
    static variable_list forward(AutogradContext* ctx, const Tensor& s0, const Tensor& r, const Tensor& w, const Tensor& k, const Tensor& v, const Tensor& a,
                                 const Tensor& b, int64_t flags, bool flat, bool grad) { return rwkv7_run(ctx, s0, r, w, k, v, a, b, flags, true, flat, grad); }
    static variable_list backward(AutogradContext* ctx, variable_list g) { variable_list x = rwkv7_grads(ctx, g[0], g[1], true); x.push_back(NONE); return x; }
};
struct Rwkv7State : Function<Rwkv7State> {
    static variable_list forward(AutogradContext* ctx, const Tensor& s0, const Tensor& r, const Tensor& w, const Tensor& k, const Tensor& v, const Tensor& a,
                                 const Tensor& b, int64_t flags, bool flat, bool grad) { return rwkv7_run(ctx, s0, r, w, k, v, a, b, flags, false, flat, grad); }
    static variable_list backward(AutogradContext* ctx, variable_list g) { variable_list x = rwkv7_grads(ctx, g[0], NONE, true); x.push_back(NONE); return x; }
};
struct Rwkv7 : Function<Rwkv7> {
    static variable_list forward(AutogradContext* ctx, const Tensor& r, const Tensor& w, const Tensor& k, const Tensor& v, const Tensor& a, const Tensor& b,
                                 int64_t flags, bool flat, bool grad) { return rwkv7_run(ctx, NONE, r, w, k, v, a, b, flags, false, flat, grad); }
    static variable_list backward(AutogradContext* ctx, variable_list g) {
        variable_list x = rwkv7_grads(ctx, g[0], NONE, false);
        x.erase(x.begin());
        x.push_back(NONE);
        return x;
    }
};
std::tuple<Tensor, Tensor> rwkv7_passing_op(const Tensor& s0, const Tensor& r, const Tensor& w, const Tensor& k, const Tensor& v, const Tensor& a, const Tensor& b, int64_t flags, bool flat) {
    variable_list o = Rwkv7Passing::apply(s0, r, w, k, v, a, b, flags, flat, wants_grad({&s0, &r, &w, &k, &v, &a, &b}));
    return {o[0], o[1]};
}
Tensor rwkv7_state_op(const Tensor& s0, const Tensor& r, const Tensor& w, const Tensor& k, const Tensor& v, const Tensor& a, const Tensor& b, int64_t flags, bool flat) {
    return Rwkv7State::apply(s0, r, w, k, v, a, b, flags, flat, wants_grad({&s0, &r, &w, &k, &v, &a, &b}))[0];
}
Tensor rwkv7_op(const Tensor& r, const Tensor& w, const Tensor& k, const Tensor& v, const Tensor& a, const Tensor& b, int64_t flags, bool flat) {
    return Rwkv7::apply(r, w, k, v, a, b, flags, flat, wants_grad({&r, &w, &k, &v, &a, &b}))[0];
}

}  // namespace

void bind_autograd(py::module_& m) {
    auto ops = m.def_submodule("ops");
    ops.def("wkv4", &wkv4_op);
    ops.def("timex", &timex_op);
    ops.def("wkv5_f32", &wkv5_f32_op);
    ops.def("wkv5a", &wkv5a_op);
    ops.def("wkv5_bf16", &wkv5_bf16_op);
    ops.def("wkv6", &wkv6_op);
    ops.def("wkv6_state", &wkv6_state_op);
    ops.def("rwkv7_passing", &rwkv7_passing_op);
    ops.def("rwkv7_state", &rwkv7_state_op);
    ops.def("rwkv7", &rwkv7_op);
}
