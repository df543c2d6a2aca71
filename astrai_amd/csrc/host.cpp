// The everyday calls of the Python adapters in one native step each: what the operands are, the outputs and scratch, torch's
// current stream, the library call. An eager Linear of a few tokens spends more time on these than on the card. A call, with
// attribute reads, allocations and ctypes in Python / here / its kernels alone (us): int8, 16 tokens through 4096 x 11008
// weights 15.3 / 11.9 / 11.6; fp8 21.5 / 16 / 15.4; 128-block fp8, 4 tokens, 7168 x 2048 21.8 / 14.7 / 8.3; paged decode, 4 x
// 500 keys 13.6 / 9.8 / 9.4; attention of 100 dense tokens 12.4 / 7.0 / 6.5; an fp8 training step of 256 tokens, 2048 x 2048
// 152 / 122; of 300 tokens, 2048 x 3072, whose bf16 backward is one call too, 81 / 61. A function returns None where a call is not the plain case that it checks for; the adapter then takes its own
// path, which says what is wrong or makes it right. Only exact torch.Tensor / Parameter objects are plain: subclasses see
// the operations that they would see without this module.
#include "host.h"

#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/record_function.h>
#include <c10/core/GradMode.h>
#include <c10/core/impl/LocalDispatchKeySet.h>

#include "../../include/astrai_w8a8.h"

namespace {

constexpr int64_t kAmaxPartials = ASTRAI_W8A8_AMAX_PARTIALS;   // floats of one operand's maxima

// a step: one fp32 value on the device
bool step_ok(const Tensor* t, c10::Device dev) {
    return !t || (t->scalar_type() == at::kFloat && t->device() == dev && t->numel() == 1);
}

Tensor bytes(int64_t n, c10::Device dev) { return at::empty({n}, at::TensorOptions().device(dev).dtype(at::kByte)); }

PyObject* failed(int rc) {
    PyErr_Format(PyExc_RuntimeError, "astrai_w8a8 error %d: %s", rc, astrai_w8a8_last_error());
    return nullptr;
}

// linear_int8(x, wq, sw, bias)
PyObject* linear_int8(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
    HANDLE_TH_ERRORS
    const Tensor *x, *wq, *sw, *bias;
    if (n_args != 4 || !(x = tensor_of(a[0])) || !(wq = tensor_of(a[1])) || !(sw = tensor_of(a[2])) || !optional(a[3], bias) ||
        !x->is_cuda() || x->dim() < 1 || wq->dim() != 2)
        Py_RETURN_NONE;
    const auto dev = x->device();
    const int64_t k = x->size(-1), n = wq->size(0);
    if (k % 16 || !x->numel() || !n || wq->size(1) != k || !plain(*x, at::kBFloat16, dev) || !plain(*wq, at::kChar, dev) ||
        !plain(*sw, at::kFloat, dev) || sw->numel() != n || (bias && (!plain(*bias, at::kBFloat16, dev) || bias->numel() != n)))
        Py_RETURN_NONE;
    const int64_t m = x->numel() / k;
    const c10::DeviceGuard guard(dev);
    const Tensor codes = bytes(m * (k + 4), dev);   // codes, then a step per row
    Tensor out = output(*x, n, at::kBFloat16);
    auto* const at = static_cast<uint8_t*>(codes.data_ptr());
    const int rc = unlocked([&] {
        return astrai_w8a8_linear_int8_bf16(x->data_ptr(), wq->data_ptr(), sw->data_ptr<float>(), ptr(bias), at,
                                            reinterpret_cast<float*>(at + m * k), out.data_ptr(), m, n, k, stream_of(dev));
    });
    return rc ? failed(rc) : THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// bf16 on one GPU as the kernels read them, rows of x as wide as w.size(inner)
bool fp8_operands(const Tensor& x, const Tensor& w, const Tensor* bias, int64_t inner) {
    if (!x.is_cuda() || x.dim() < 1 || w.dim() != 2 || x.size(-1) != w.size(inner) || x.size(-1) % 16 || !x.numel() || !w.numel())
        return false;
    const auto dev = x.device();
    return plain16(x, at::kBFloat16, dev) && plain16(w, at::kBFloat16, dev) &&
           (!bias || (bias->dim() == 1 && bias->size(0) == w.size(0) && plain16(*bias, at::kBFloat16, dev)));
}

// linear_fp8_operands(x, w, bias, inner)
PyObject* linear_fp8_operands(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
    HANDLE_TH_ERRORS
    const Tensor *x, *w, *bias;
    int64_t inner;
    if (n_args != 4 || !(x = tensor_of(a[0])) || !(w = tensor_of(a[1])) || !optional(a[2], bias) || !whole(a[3], inner) ||
        inner < 0 || inner > 1)
        Py_RETURN_NONE;
    return PyBool_FromLong(fp8_operands(*x, *w, bias, inner));
    END_HANDLE_TH_ERRORS
}

struct Ring {
    const Tensor* hist = nullptr;
    int64_t idx = 0;
    bool read(PyObject* h, PyObject* i, c10::Device dev) {
        return optional(h, hist) && whole(i, idx) && (!hist || plain(*hist, at::kFloat, dev));
    }
    float* at() const { return hist ? hist->data_ptr<float>() : nullptr; }
    int len() const { return hist ? (int)hist->numel() : 0; }
};

// linear_fp8(x, w, bias, codes, x_step, w_step, x_hist, x_idx, w_hist, w_idx, fmt, fmax, pow2_margin)
PyObject* linear_fp8(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
    HANDLE_TH_ERRORS
    const Tensor *x, *w, *bias, *codes, *sx, *sw;
    Ring rx, rw;
    int64_t fmt;
    double fmax, margin;
    if (n_args != 13 || !(x = tensor_of(a[0])) || !(w = tensor_of(a[1])) || !optional(a[2], bias) || !optional(a[3], codes) ||
        !optional(a[4], sx) || !optional(a[5], sw) || !fp8_operands(*x, *w, bias, 1))
        Py_RETURN_NONE;
    const auto dev = x->device();
    if (!rx.read(a[6], a[7], dev) || !rw.read(a[8], a[9], dev) || !whole(a[10], fmt) || !real(a[11], fmax) || !real(a[12], margin) ||
        !step_ok(sx, dev) || !step_ok(sw, dev) || (codes && (codes->device() != dev || codes->numel() != w->numel())))
        Py_RETURN_NONE;
    const int64_t n = w->size(0), k = w->size(1), m = x->numel() / k;
    const bool measure = !rx.hist;
    const c10::DeviceGuard guard(dev);
    // maxima of x, of w; steps; codes of x; codes of w
    const int64_t steps_at = 2 * 4 * kAmaxPartials, x_at = steps_at + 256, w_at = x_at + (m * k + 255) / 256 * 256;
    const Tensor scratch = bytes(w_at + (codes ? 0 : n * k), dev);
    Tensor out = output(*x, n, at::kBFloat16);
    auto* const at = static_cast<uint8_t*>(scratch.data_ptr());
    auto* const steps = reinterpret_cast<float*>(at + steps_at);
    auto* const maxima = reinterpret_cast<float*>(at);
    const int rc = unlocked([&] {
        return astrai_w8a8_linear_fp8_bf16(
            x->data_ptr(), at + x_at, sx ? sx->data_ptr<float>() : steps, maxima, rx.at(), rx.len(), (int)rx.idx,
            codes ? nullptr : w->data_ptr(), codes ? codes->data_ptr() : at + w_at, sw ? sw->data_ptr<float>() : steps + 1,
            maxima + kAmaxPartials, rw.at(), rw.len(), (int)rw.idx, ptr(bias), measure, out.data_ptr(), m, n, k, (int)fmt, measure,
            (float)fmax, (float)margin, stream_of(dev));
    });
    return rc ? failed(rc) : THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// linear_fp8_backward(g, x, w, want_bias, g_step, x_step, w_step, hist, idx, fmt, fmax, pow2_margin)
PyObject* linear_fp8_backward(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
    HANDLE_TH_ERRORS
    const Tensor *g, *x, *w, *sg, *sx, *sw;
    Ring ring;
    int64_t fmt;
    double fmax, margin;
    if (n_args != 12 || !(g = tensor_of(a[0])) || !(x = tensor_of(a[1])) || !(w = tensor_of(a[2])) || !PyBool_Check(a[3]) ||
        !optional(a[4], sg) || !optional(a[5], sx) || !optional(a[6], sw) || !fp8_operands(*x, *w, nullptr, 1) ||
        !fp8_operands(*g, *w, nullptr, 0))
        Py_RETURN_NONE;
    const auto dev = x->device();
    const int64_t n = w->size(0), k = w->size(1), m = x->numel() / k;
    if (g->numel() != m * n || g->device() != dev || !ring.read(a[7], a[8], dev) || !whole(a[9], fmt) || !real(a[10], fmax) ||
        !real(a[11], margin) || !step_ok(sg, dev) || !step_ok(sx, dev) || !step_ok(sw, dev))
        Py_RETURN_NONE;
    const bool want_bias = a[3] == Py_True;
    const c10::DeviceGuard guard(dev);
    const Tensor scratch = bytes(astrai_w8a8_linear_fp8_backward_scratch_bytes(m, n, k), dev);
    const auto like = [&](const Tensor& t) { return at::empty(t.sizes(), t.options().requires_grad(false)); };
    Tensor gx = like(*x), gw = like(*w);
    Tensor gb = at::empty({want_bias ? n : 0}, g->options().requires_grad(false));
    auto step = [](const Tensor* t) { return t ? t->data_ptr<float>() : nullptr; };
    const int rc = unlocked([&] {
        return astrai_w8a8_linear_fp8_backward_bf16(g->data_ptr(), x->data_ptr(), w->data_ptr(), step(sg), step(sx), step(sw),
                                                    scratch.data_ptr(), gx.data_ptr(), gw.data_ptr(),
                                                    want_bias ? gb.data_ptr() : nullptr, m, n, k, (int)fmt, ring.at(), ring.len(),
                                                    (int)ring.idx, (float)fmax, (float)margin, stream_of(dev));
    });
    if (rc) return failed(rc);
    return Py_BuildValue("(NNN)", THPVariable_Wrap(std::move(gx)), THPVariable_Wrap(std::move(gw)), THPVariable_Wrap(std::move(gb)));
    END_HANDLE_TH_ERRORS
}

// linear_backward(g, x, w, want_x, want_w, want_bias): the kernels' own products, those that want_* ask for
PyObject* linear_backward(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
    HANDLE_TH_ERRORS
    const Tensor *g, *x, *w;
    if (n_args != 6 || !(g = tensor_of(a[0])) || !(x = tensor_of(a[1])) || !(w = tensor_of(a[2])) || !PyBool_Check(a[3]) ||
        !PyBool_Check(a[4]) || !PyBool_Check(a[5]) || !g->is_cuda() || g->dim() != 2 || x->dim() != 2 || w->dim() != 2)
        Py_RETURN_NONE;
    const auto dev = g->device();
    const int64_t m = g->size(0), n = w->size(0), k = w->size(1);
    const bool want_x = a[3] == Py_True, want_w = a[4] == Py_True, want_bias = a[5] == Py_True;
    if (g->size(1) != n || x->size(0) != m || x->size(1) != k || !plain16(*g, at::kBFloat16, dev) || !plain16(*x, at::kBFloat16, dev) ||
        !plain16(*w, at::kBFloat16, dev) || !(want_x || want_w) || (want_bias && !want_w))
        Py_RETURN_NONE;
    const int64_t need = astrai_w8a8_linear_backward_scratch_bytes(m, n, k);
    if (need < 0) Py_RETURN_NONE;
    const c10::DeviceGuard guard(dev);
    const Tensor scratch = need ? bytes(need, dev) : Tensor();
    const auto bf16 = at::TensorOptions().device(dev).dtype(at::kBFloat16);
    auto matrix = [&](bool want, int64_t rows) { return want ? at::empty({rows, k}, bf16) : at::empty({0}, bf16); };
    Tensor gx = matrix(want_x, m), gw = matrix(want_w, n), gb = at::empty({want_bias ? n : 0}, bf16);
    const int rc = unlocked([&] {
        return astrai_w8a8_linear_backward_bf16(g->data_ptr(), x->data_ptr(), w->data_ptr(), need ? scratch.data_ptr() : nullptr,
                                                want_x ? gx.data_ptr() : nullptr, want_w ? gw.data_ptr() : nullptr,
                                                want_bias ? gb.data_ptr() : nullptr, m, n, k, stream_of(dev));
    });
    if (rc) return failed(rc);
    return Py_BuildValue("(NNN)", THPVariable_Wrap(std::move(gx)), THPVariable_Wrap(std::move(gw)), THPVariable_Wrap(std::move(gb)));
    END_HANDLE_TH_ERRORS
}

// quantize_block128_act(x)
PyObject* quantize_block128_act(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
    HANDLE_TH_ERRORS
    const Tensor* x;
    if (n_args != 1 || !(x = tensor_of(a[0])) || !x->is_cuda() || x->dim() != 2 || x->size(1) % 128 || !x->numel() ||
        !plain(*x, at::kBFloat16, x->device()))
        Py_RETURN_NONE;
    const auto dev = x->device();
    const int64_t m = x->size(0), k = x->size(1);
    const c10::DeviceGuard guard(dev);
    const auto on = at::TensorOptions().device(dev);
    Tensor codes = at::empty({m, k}, on.dtype(at::kFloat8_e4m3fn)), steps = at::empty({m, k / 128}, on.dtype(at::kFloat));
    const int rc = unlocked([&] {
        return astrai_w8a8_quantize_bf16_fp8_block128_act(x->data_ptr(), codes.data_ptr(), steps.data_ptr<float>(), m, k,
                                                          stream_of(dev));
    });
    if (rc) return failed(rc);
    return Py_BuildValue("(NN)", THPVariable_Wrap(std::move(codes)), THPVariable_Wrap(std::move(steps)));
    END_HANDLE_TH_ERRORS
}

// mm_block128(a, b, sa, sb, bias)
PyObject* mm_block128(PyObject*, PyObject* const* args, Py_ssize_t n_args) {
    HANDLE_TH_ERRORS
    const Tensor *a, *b, *sa, *sb, *bias;
    if (n_args != 5 || !(a = tensor_of(args[0])) || !(b = tensor_of(args[1])) || !(sa = tensor_of(args[2])) ||
        !(sb = tensor_of(args[3])) || !optional(args[4], bias) || !a->is_cuda() || a->dim() != 2 || b->dim() != 2)
        Py_RETURN_NONE;
    const auto dev = a->device();
    const int64_t m = a->size(0), k = a->size(1), n = b->size(0), kb = k / 128;
    if (!m || !n || !k || k % 128 || b->size(1) != k || !plain(*a, at::kFloat8_e4m3fn, dev) || !plain(*b, at::kFloat8_e4m3fn, dev) ||
        !plain(*sa, at::kFloat, dev) || sa->numel() != m * kb || !plain(*sb, at::kFloat, dev) ||
        sb->numel() != (n + 127) / 128 * kb || (bias && (!plain(*bias, at::kBFloat16, dev) || bias->numel() != n)))
        Py_RETURN_NONE;
    const c10::DeviceGuard guard(dev);
    Tensor out = at::empty({m, n}, at::TensorOptions().device(dev).dtype(at::kBFloat16));
    const int rc = unlocked([&] {
        return astrai_w8a8_gemm_fp8_block128(a->data_ptr(), b->data_ptr(), sa->data_ptr<float>(), sb->data_ptr<float>(), ptr(bias),
                                             out.data_ptr(), m, n, k, stream_of(dev));
    });
    return rc ? failed(rc) : THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// Whether a dispatcher op on these would do nothing but call its device kernel: plain tensors of one GPU that need no
// gradient and carry no tangent, no dispatch or function mode, transform, trace, functionalization or profiler about.
bool nothing_above(std::initializer_list<const Tensor*> tensors) {
    using K = c10::DispatchKey;
    static const c10::DispatchKeySet above({K::Python, K::PythonTLSSnapshot, K::PythonDispatcher, K::PreDispatch, K::Functionalize,
                                            K::FuncTorchDynamicLayerFrontMode, K::FuncTorchDynamicLayerBackMode, K::FuncTorchBatched,
                                            K::FuncTorchVmapMode, K::FuncTorchGradWrapper, K::FuncTorchBatchedDecomposition,
                                            K::BatchedNestedTensor, K::NestedTensor, K::Tracer, K::Fake, K::Negative, K::Conjugate,
                                            K::DeferredInit});
    const auto on = c10::impl::tls_local_dispatch_key_set();
    if (!(on.included_ & above).empty() || at::impl::torch_function_mode_enabled() || at::hasCallbacks()) return false;
    const bool grads = c10::GradMode::is_enabled();
    for (const Tensor* t : tensors)
        if (t && (!(t->key_set() & above).empty() || (grads && t->requires_grad()) || t->_fw_grad(0).defined())) return false;
    return true;
}

// mm_block128_eager(a, b, sa, sb, bias): the op fp8_gemm_blockscaled where nothing is above its device kernel
PyObject* mm_block128_eager(PyObject* self, PyObject* const* args, Py_ssize_t n_args) {
    HANDLE_TH_ERRORS
    const Tensor* t[5] = {};
    if (n_args != 5 || !optional(args[4], t[4])) Py_RETURN_NONE;
    for (int i = 0; i < 4; ++i)
        if (!(t[i] = tensor_of(args[i]))) Py_RETURN_NONE;
    if (!nothing_above({t[0], t[1], t[2], t[3], t[4]})) Py_RETURN_NONE;
    return mm_block128(self, args, n_args);
    END_HANDLE_TH_ERRORS
}

// queries over pools behind a slot table
struct Paged {
    const Tensor *q, *k, *v, *table, *rows, *kv_indptr;
    int64_t h = 0, d = 0, slots = 0, hkv = 0, b = 0;
    bool read(PyObject* const* a) {
        if (!(q = tensor_of(a[0])) || !(k = tensor_of(a[1])) || !(v = tensor_of(a[2])) || !(table = tensor_of(a[3])) ||
            !(rows = tensor_of(a[4])) || !(kv_indptr = tensor_of(a[5])) || !q->is_cuda() || q->dim() != 3 || k->dim() != 3 ||
            k->sizes() != v->sizes() || table->dim() != 2)
            return false;
        const auto dev = q->device();
        h = q->size(1), d = q->size(2), slots = k->size(0), hkv = k->size(1), b = rows->numel();
        // (the pools' device is the library's business, as it was)
        return k->size(2) == d && hkv && h % hkv == 0 && q->numel() && b && plain(*q, at::kBFloat16, dev) &&
               plain(*k, at::kBFloat16, k->device()) && plain(*v, at::kBFloat16, v->device()) && plain(*table, at::kInt, dev) &&
               plain(*rows, at::kInt, dev) && plain(*kv_indptr, at::kInt, dev) && kv_indptr->numel() == b + 1;
    }
    Tensor out() const { return at::empty(q->sizes(), at::TensorOptions().device(q->device()).dtype(at::kBFloat16)); }
    Tensor floats(int64_t n) const {
        return at::empty({std::max<int64_t>(n, 1)}, at::TensorOptions().device(q->device()).dtype(at::kFloat));
    }
};

// attn_paged_decode(q, k, v, table, rows, kv_indptr, general, nsplit, scale)
PyObject* attn_paged_decode(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
    HANDLE_TH_ERRORS
    Paged p;
    int64_t nsplit;
    double scale;
    if (n_args != 9 || !p.read(a) || !PyBool_Check(a[6]) || !whole(a[7], nsplit) || nsplit < 1 || !real(a[8], scale) ||
        p.q->size(0) != p.b)
        Py_RETURN_NONE;
    const bool general = a[6] == Py_True;
    const int64_t need = general ? astrai_w8a8_attn_paged_rows_workspace_floats(p.b, p.h, p.hkv, p.d, nsplit, 0)
                                 : astrai_w8a8_attn_decode_workspace_floats(p.b, p.hkv, nsplit, p.h / p.hkv);
    if (need < 0) Py_RETURN_NONE;
    const auto dev = p.q->device();
    const c10::DeviceGuard guard(dev);
    Tensor out = p.out();
    const Tensor ws = p.floats(need);
    const int rc = unlocked([&] {
        auto* const q = p.q->data_ptr();
        auto* const k = p.k->data_ptr();
        auto* const v = p.v->data_ptr();
        const int *table = p.table->data_ptr<int>(), *rows = p.rows->data_ptr<int>(), *kv = p.kv_indptr->data_ptr<int>();
        if (general)
            return astrai_w8a8_attn_paged_rows_bf16(q, k, v, table, rows, kv, nullptr, nullptr, nullptr, nullptr, 0, 0, 0, 1, 0,
                                                    ws.data_ptr<float>(), ws.numel(), out.data_ptr(), p.b, p.h, p.hkv, p.d, p.slots,
                                                    p.table->size(0), p.table->size(1), 0, nsplit, (float)scale, stream_of(dev));
        return astrai_w8a8_attn_paged_decode_masked_bf16(q, k, v, table, rows, kv, nullptr, 0, 0, ws.data_ptr<float>(), ws.numel(),
                                                         out.data_ptr(), p.b, p.h, p.hkv, p.d, p.slots, p.table->size(0),
                                                         p.table->size(1), nsplit, (float)scale, stream_of(dev));
    });
    return rc ? failed(rc) : THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// attn_paged_prefill(q, k, v, table, rows, kv_indptr, qo_indptr, tile_batch, tile_index, general, nsplit, causal, scale)
PyObject* attn_paged_prefill(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
    HANDLE_TH_ERRORS
    Paged p;
    const Tensor *qo, *tb, *ti;
    int64_t nsplit;
    double scale;
    if (n_args != 13 || !p.read(a) || !(qo = tensor_of(a[6])) || !(tb = tensor_of(a[7])) || !(ti = tensor_of(a[8])) ||
        !PyBool_Check(a[9]) || !whole(a[10], nsplit) || nsplit < 1 || !PyBool_Check(a[11]) || !real(a[12], scale))
        Py_RETURN_NONE;
    const auto dev = p.q->device();
    if (!plain(*qo, at::kInt, dev) || !plain(*tb, at::kInt, dev) || !plain(*ti, at::kInt, dev) || qo->numel() != p.b + 1 ||
        tb->dim() != 1 || ti->dim() != 1 || !tb->numel() || tb->numel() != ti->numel())
        Py_RETURN_NONE;
    const int64_t tiles = tb->numel();
    const int causal = a[11] == Py_True;
    const bool general = a[9] == Py_True;
    const int64_t need = general ? astrai_w8a8_attn_paged_rows_workspace_floats(tiles, p.h, p.hkv, p.d, nsplit, 1) : 0;
    if (need < 0) Py_RETURN_NONE;
    const c10::DeviceGuard guard(dev);
    Tensor out = p.out(), ws;   // (rows that no tile of the schedule covers are left unwritten, as by the reference)
    if (general) ws = p.floats(need);
    const int rc = unlocked([&] {
        auto* const q = p.q->data_ptr();
        auto* const k = p.k->data_ptr();
        auto* const v = p.v->data_ptr();
        const int *table = p.table->data_ptr<int>(), *rows = p.rows->data_ptr<int>(), *kv = p.kv_indptr->data_ptr<int>();
        if (general)
            return astrai_w8a8_attn_paged_rows_bf16(q, k, v, table, rows, kv, qo->data_ptr<int>(), tb->data_ptr<int>(),
                                                    ti->data_ptr<int>(), nullptr, 0, 0, 0, 0, 0, ws.data_ptr<float>(), ws.numel(),
                                                    out.data_ptr(), tiles, p.h, p.hkv, p.d, p.slots, p.table->size(0),
                                                    p.table->size(1), causal, nsplit, (float)scale, stream_of(dev));
        return astrai_w8a8_attn_paged_prefill_masked_bf16(q, k, v, table, rows, kv, qo->data_ptr<int>(), tb->data_ptr<int>(),
                                                          ti->data_ptr<int>(), nullptr, 0, 0, 0, 0, 0, out.data_ptr(), tiles, p.h,
                                                          p.hkv, p.d, p.slots, p.table->size(0), p.table->size(1), causal,
                                                          (float)scale, stream_of(dev));
    });
    return rc ? failed(rc) : THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// attn_prefill(q, k, v, causal_offset, scale): [batch, rows, heads, size], read where they lie
PyObject* attn_prefill(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
    HANDLE_TH_ERRORS
    const Tensor *t[3];
    int64_t offset;
    double scale;
    if (n_args != 5 || !whole(a[3], offset) || !real(a[4], scale)) Py_RETURN_NONE;
    for (int i = 0; i < 3; ++i)
        if (!(t[i] = tensor_of(a[i])) || !t[i]->is_cuda() || t[i]->dim() != 4 || t[i]->scalar_type() != at::kBFloat16 ||
            t[i]->device() != t[0]->device() || !t[i]->numel() || t[i]->size(0) != t[0]->size(0) || t[i]->size(3) != t[0]->size(3) ||
            t[i]->stride(3) != 1 || t[i]->stride(0) % 8 || t[i]->stride(1) % 8 || t[i]->stride(2) % 8 ||
            reinterpret_cast<uintptr_t>(t[i]->data_ptr()) % 16)
            Py_RETURN_NONE;
    const int64_t b = t[0]->size(0), n = t[0]->size(1), h = t[0]->size(2), d = t[0]->size(3), m = t[1]->size(1), hkv = t[1]->size(2);
    if (t[1]->sizes() != t[2]->sizes() || h % hkv || m * std::max(t[1]->stride(1), t[2]->stride(1)) > ((int64_t)1 << 31) - 128)
        Py_RETURN_NONE;
    int64_t strides[9];
    for (int i = 0; i < 3; ++i) {
        strides[3 * i] = t[i]->stride(0);
        strides[3 * i + 1] = t[i]->stride(2);
        strides[3 * i + 2] = t[i]->stride(1);
    }
    const auto dev = t[0]->device();
    const c10::DeviceGuard guard(dev);
    Tensor out = at::empty({b, n, h, d}, at::TensorOptions().device(dev).dtype(at::kBFloat16));
    const int rc = unlocked([&] {
        return astrai_w8a8_attn_prefill_strided_bf16(t[0]->data_ptr(), t[1]->data_ptr(), t[2]->data_ptr(), strides, nullptr,
                                                     out.data_ptr(), b, n, m, h, hkv, d, std::min(offset, m), (float)scale,
                                                     stream_of(dev));
    });
    return rc ? failed(rc) : THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

PyMethodDef methods[] = {ENTRY(linear_int8), ENTRY(linear_fp8_operands), ENTRY(linear_fp8), ENTRY(linear_fp8_backward), ENTRY(linear_backward),
                         ENTRY(quantize_block128_act), ENTRY(mm_block128), ENTRY(mm_block128_eager), ENTRY(attn_paged_decode), ENTRY(attn_paged_prefill),
                         ENTRY(attn_prefill), {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host", nullptr, -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit__host() { return with_built_for(PyModule_Create(&module), ASTRAI_W8A8_ABI_VERSION); }
