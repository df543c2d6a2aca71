// host.cpp's native calls for libastrai_mix.so: the few-rows products and row operations that a prompt or an eager step of
// the models with sequence mixers is made of. A prompt of 40 tokens through a few layers, some 60 such calls: with their
// checks in Python 526 (latent, lightning) and 1003 us (recurrences, delta rule), here 426 and 720.
#include "host.h"

#include "../../include/astrai_mix.h"

namespace {

PyObject* failed(int rc) {
    PyErr_Format(PyExc_RuntimeError, "astrai_mix error %d: %s", rc, astrai_mix_last_error());
    return nullptr;
}

bool dense(const Tensor* t, c10::Device dev, int64_t rows, int64_t cols) {   // fp32; rows < 0: a vector
    return !t || (plain(*t, at::kFloat, dev) && (rows < 0 ? t->dim() == 1 && t->size(0) == cols
                                                          : t->dim() == 2 && t->size(0) == rows && t->size(1) == cols));
}

bool near16(const Tensor& t, uintptr_t q = 16) { return reinterpret_cast<uintptr_t>(t.data_ptr()) % q == 0; }

struct FewRows {
    const Tensor *x, *w, *bias = nullptr;
    int64_t act, most, m, n, k, ldx;   // act -1: none
    // x, weight, bias, act, most rows
    bool read(PyObject* const* a) {
        return (x = tensor_of(a[0])) && (w = tensor_of(a[1])) && optional(a[2], bias) && whole(a[3], act) && whole(a[4], most) && fits();
    }
    bool fits() {
        if (!x->is_cuda() || x->dim() < 1 || w->dim() != 2) return false;
        const auto dev = x->device();
        n = w->size(0) / (act < 0 ? 1 : 2), k = w->size(1), m = k ? x->numel() / k : 0;
        if (x->size(-1) != k || m <= 0 || m > most || k % 128 || n % 4 || w->numel() * 2 >= (int64_t)1 << 31 ||
            x->scalar_type() != at::kBFloat16 || !plain16(*w, at::kBFloat16, dev) || !near16(*x) ||
            (bias && (act >= 0 || bias->numel() != n || !plain(*bias, at::kBFloat16, dev) || !near16(*bias, 8))))
            return false;
        ldx = k;
        if (x->is_contiguous()) return true;
        ldx = x->dim() == 2 && x->stride(1) == 1 ? x->stride(0) : 0;
        return ldx >= k && ldx % 8 == 0 && ldx < 1 << 23;
    }
};

// few_rows_linear_takes(x, weight, bias, act, most): True, or None for the adapter's own answer
PyObject* few_rows_linear_takes(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
    HANDLE_TH_ERRORS
    FewRows r;
    if (n_args == 5 && r.read(a)) Py_RETURN_TRUE;
    Py_RETURN_NONE;
    END_HANDLE_TH_ERRORS
}

// few_rows_parts(x, weight, most, parts)
PyObject* few_rows_parts(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
    HANDLE_TH_ERRORS
    FewRows r;
    int64_t parts;
    if (n_args != 4 || !whole(a[3], parts) || parts < 1) Py_RETURN_NONE;
    r.act = -1;
    if (!(r.x = tensor_of(a[0])) || !(r.w = tensor_of(a[1])) || !whole(a[2], r.most) || !r.fits()) Py_RETURN_NONE;
    const auto dev = r.x->device();
    const c10::DeviceGuard guard(dev);
    Tensor out = at::empty({parts, r.m, r.n}, at::TensorOptions().device(dev).dtype(at::kFloat));
    const int rc = unlocked([&] {
        return astrai_mix_few_rows_parts(r.x->data_ptr(), r.ldx, r.w->data_ptr(), out.data_ptr<float>(), r.m, r.n, r.k, parts,
                                         stream_of(dev));
    });
    return rc ? failed(rc) : THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// few_rows_linear(x, weight, bias, act, most, out_float)
PyObject* few_rows_linear(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
    HANDLE_TH_ERRORS
    FewRows r;
    if (n_args != 6 || !r.read(a) || !PyBool_Check(a[5])) Py_RETURN_NONE;
    const bool out_float = a[5] == Py_True;
    const auto dev = r.x->device();
    const c10::DeviceGuard guard(dev);
    Tensor out = output(*r.x, r.n, out_float ? at::kFloat : at::kBFloat16);
    const int rc = unlocked([&] {
        return astrai_mix_few_rows_linear(r.x->data_ptr(), r.ldx, r.w->data_ptr(), ptr(r.bias), out.data_ptr(), r.m, r.n, r.k,
                                          (int)r.act, out_float, stream_of(dev));
    });
    return rc ? failed(rc) : THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// sum_norm(y, w, bf16, eps, x, u, vec, tokens, mult, out)
PyObject* sum_norm(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
    HANDLE_TH_ERRORS
    const Tensor *y, *w, *x, *u, *vec, *tokens, *given;
    double eps, mult;
    if (n_args != 10 || !(y = tensor_of(a[0])) || !optional(a[1], w) || !PyBool_Check(a[2]) || !real(a[3], eps) || !optional(a[4], x) ||
        !optional(a[5], u) || !optional(a[6], vec) || !optional(a[7], tokens) || !real(a[8], mult) || !optional(a[9], given) ||
        !y->is_cuda() || (y->dim() != 2 && y->dim() != 3))
        Py_RETURN_NONE;
    const auto dev = y->device();
    const auto type = a[2] == Py_True ? at::kBFloat16 : at::kFloat;
    const bool parts = y->dim() == 3;   // planes to add up
    const int64_t width = y->size(-1), n = tokens ? tokens->numel() : y->size(-2);
    if (parts && (y->scalar_type() != at::kFloat || tokens || y->stride(2) != 1 || y->stride(1) < width)) Py_RETURN_NONE;
    for (const Tensor* t : {parts ? u : y, u})
        if (t && (t->dim() != 2 || t->size(1) != width || t->stride(1) != 1 || t->stride(0) < width || t->device() != dev ||
                  t->scalar_type() != y->scalar_type() || (t->scalar_type() != type && t->scalar_type() != at::kFloat)))
            Py_RETURN_NONE;
    if ((tokens && !plain(*tokens, at::kLong, dev)) || (u && u->size(0) != n) || !dense(x, dev, n, width) ||
        !dense(given, dev, n, width) || !dense(vec, dev, -1, width) || !dense(w, dev, -1, width))
        Py_RETURN_NONE;
    const c10::DeviceGuard guard(dev);
    const auto on = at::TensorOptions().device(dev);
    Tensor out = given ? *given : at::empty({n, width}, on.dtype(at::kFloat)), h = at::empty({n, width}, on.dtype(type));
    const int rc = unlocked([&] {
        auto vector = [](const Tensor* t) { return t ? t->data_ptr<float>() : nullptr; };
        if (parts)
            return astrai_mix_sum_norm_parts(y->data_ptr<float>(), y->stride(1), y->stride(0), y->size(0), (float)mult, vector(x), vector(u),
                                             u ? u->stride(0) : 0, vector(vec), out.data_ptr<float>(), vector(w), h.data_ptr(), n, width,
                                             (float)eps, type == at::kFloat, stream_of(dev));
        return astrai_mix_sum_norm(y->data_ptr(), y->stride(0), tokens ? tokens->data_ptr<int64_t>() : nullptr, y->size(0), (float)mult,
                                   vector(x), ptr(u), u ? u->stride(0) : 0, vector(vec), out.data_ptr<float>(), vector(w),
                                   h.data_ptr(), n, width, (float)eps, y->scalar_type() == at::kFloat, type == at::kFloat,
                                   stream_of(dev));
    });
    if (rc) return failed(rc);
    PyObject* first = given ? Py_NewRef(a[9]) : THPVariable_Wrap(std::move(out));
    return Py_BuildValue("(NN)", first, THPVariable_Wrap(std::move(h)));
    END_HANDLE_TH_ERRORS
}

// residual_norm(y, x, w_post, w_pre, mult, eps)
PyObject* residual_norm(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
    HANDLE_TH_ERRORS
    const Tensor *y, *x, *post, *pre;
    double mult, eps;
    if (n_args != 6 || !(y = tensor_of(a[0])) || !(x = tensor_of(a[1])) || !(post = tensor_of(a[2])) || !(pre = tensor_of(a[3])) ||
        !real(a[4], mult) || !real(a[5], eps) || !y->is_cuda() || (y->dim() != 2 && y->dim() != 3))
        Py_RETURN_NONE;
    const auto dev = y->device();
    const bool parts = y->dim() == 3;   // fp32 planes to add up, h in bf16
    if (parts && y->scalar_type() != at::kFloat) Py_RETURN_NONE;
    const auto type = parts ? at::kBFloat16 : y->scalar_type();
    const int64_t n = y->size(-2), width = y->size(-1);
    if ((type != at::kBFloat16 && type != at::kFloat) || !y->is_contiguous() || !dense(x, dev, n, width) ||
        !dense(post, dev, -1, width) || !dense(pre, dev, -1, width))
        Py_RETURN_NONE;
    const c10::DeviceGuard guard(dev);
    Tensor h = at::empty({n, width}, at::TensorOptions().device(dev).dtype(type));
    const int rc = unlocked([&] {
        if (parts)
            return astrai_mix_residual_norm_parts(y->data_ptr<float>(), n * width, y->size(0), x->data_ptr<float>(), x->data_ptr<float>(),
                                                  post->data_ptr<float>(), pre->data_ptr<float>(), h.data_ptr(), n, width, (float)mult,
                                                  (float)eps, stream_of(dev));
        return astrai_mix_residual_norm(y->data_ptr(), x->data_ptr<float>(), x->data_ptr<float>(), post->data_ptr<float>(),
                                        pre->data_ptr<float>(), h.data_ptr(), n, width, (float)mult, (float)eps, type == at::kFloat,
                                        stream_of(dev));
    });
    return rc ? failed(rc) : THPVariable_Wrap(std::move(h));
    END_HANDLE_TH_ERRORS
}

PyMethodDef methods[] = {ENTRY(few_rows_linear_takes), ENTRY(few_rows_linear), ENTRY(few_rows_parts), ENTRY(sum_norm), ENTRY(residual_norm), {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host_mix", nullptr, -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit__host_mix() { return with_built_for(PyModule_Create(&module), ASTRAI_MIX_ABI_VERSION); }
