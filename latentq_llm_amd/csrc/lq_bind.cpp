// CPython fast paths of the tensor-level wrappers in ops.py: check, allocate, take the current stream, call the C ABI.
//
// A decoding program makes one such call per linear layer and token, and a call's kernel runs for 5 to 15 us; the
// wrappers written in Python (attribute checks, a device guard, a stream object, a ctypes call of a dozen arguments) took
// 15 to 20 us of host time each, so the device waited for the host. The functions here take the same tensors and do the
// same work in about 2 us plus the launch.
//
// Every function returns None when an operand is not in the plain form the kernels take (wrong type, device, layout or
// size, a tensor subclass, a shape without work): the Python wrapper then goes through its own checks, which raise what
// they always raised. An error of the library itself is raised as the binding's LatentQError.
#include <torch/csrc/autograd/python_variable.h>
#include <ATen/ATen.h>
#include <ATen/SavedTensorHooks.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/GradMode.h>
#include <c10/core/InferenceMode.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/forward_grad.h>
#include <torch/csrc/jit/frontend/tracer.h>

#include "../../include/latentq.h"

namespace {

PyObject *g_error = nullptr;  // LatentQError

// A plain tensor (Tensor or Parameter, no other subclass) on a GPU, contiguous, of the given type. The wrappers of function
// transforms (vmap, functional gradients, functionalisation) have the Python type of a plain tensor and no memory of their own.
const at::Tensor *plain(PyObject *o, at::ScalarType type) {
    if (!THPVariable_CheckExact(o)) return nullptr;
    const at::Tensor &t = THPVariable_Unpack(o);
    constexpr c10::DispatchKeySet kWrapped({c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchGradWrapper,
                                            c10::DispatchKey::Batched, c10::DispatchKey::Functionalize, c10::DispatchKey::Python,
                                            c10::DispatchKey::ZeroTensor, c10::DispatchKey::Conjugate, c10::DispatchKey::Negative});
    if (t.key_set().has_any(kWrapped) || !t.has_storage()) return nullptr;
    return t.is_cuda() && t.scalar_type() == type && t.is_contiguous() ? &t : nullptr;
}

const at::Tensor *bf16(PyObject *o) { return plain(o, at::kBFloat16); }

// Packed codes of an [N, K] matrix
const at::Tensor *codes4(PyObject *o, int64_t N, int64_t K) {
    const at::Tensor *t = plain(o, at::kChar);
    if (!t) t = plain(o, at::kByte);
    return t && t->numel() == N * K / 2 ? t : nullptr;
}

const at::Tensor *sized(const at::Tensor *t, int64_t n) { return t && t->numel() == n ? t : nullptr; }

struct W4 {
    const at::Tensor *codes, *scales, *zeros;
    bool load(PyObject *const *o, int64_t N, int64_t K) {
        if (N <= 0 || K <= 0) return false;
        codes = codes4(o[0], N, K);
        scales = sized(bf16(o[1]), N * K / LQ_GROUP);
        zeros = sized(bf16(o[2]), N * K / LQ_GROUP);
        return codes && scales && zeros;
    }
};

int64_t integer(PyObject *o) { return PyLong_AsLongLong(o); }

PyObject *none() { Py_RETURN_NONE; }

PyObject *fail(const char *who, int rc) {
    PyErr_Format(g_error ? g_error : PyExc_RuntimeError, "%s failed (%d): %s", who, rc, lq_last_error());
    return nullptr;
}

// The device of `t` made current, and its current stream
struct On {
    c10::OptionalDeviceGuard guard;
    void *stream;
    explicit On(const at::Tensor &t) {
        guard.reset_device(t.device());
        stream = (void *)c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(t.device().index()).stream();
    }
};

bool same_device(const at::Tensor *a, const at::Tensor *b) { return a->device() == b->device(); }

at::Tensor make(at::IntArrayRef shape, at::ScalarType type, const at::Tensor &like) {
    return at::empty(shape, like.options().dtype(type));
}

// The shape of x with its last dimension replaced
at::Tensor make_rows(const at::Tensor &x, int64_t last, at::ScalarType type) {
    at::DimVector shape(x.sizes().begin(), x.sizes().end());
    shape.back() = last;
    return make(shape, type, x);
}

// Token rows of an operand whose last dimension is `width`: 0 if there are none or the width differs
int64_t rows_of(const at::Tensor *x, int64_t width) {
    return x && x->dim() >= 1 && width > 0 && x->size(-1) == width ? x->numel() / width : 0;
}

bool aligned16(const at::Tensor *t) { return ((uintptr_t)t->data_ptr() & 15) == 0; }

// A workspace argument: None, or bytes on the operand's device
bool workspace(PyObject *o, const at::Tensor *x, void **p, int64_t *bytes) {
    *p = nullptr;
    *bytes = 0;
    if (o == Py_None) return true;
    const at::Tensor *t = plain(o, at::kByte);
    if (!t || !same_device(t, x)) return false;
    *p = t->data_ptr();
    *bytes = t->numel();
    return true;
}

PyObject *wrap(at::Tensor t) { return THPVariable_Wrap(std::move(t)); }

#define LQ_CALL(name, ...)                              \
    do {                                                \
        int rc_;                                        \
        Py_BEGIN_ALLOW_THREADS                          \
        rc_ = name(__VA_ARGS__);                        \
        Py_END_ALLOW_THREADS                            \
        if (rc_ != LQ_OK) return fail(#name, rc_);      \
    } while (0)

// bias argument: None, or bf16 [N]; false if it is neither
bool bias_of(PyObject *o, int64_t N, const void **p) {
    *p = nullptr;
    if (o == Py_None) return true;
    const at::Tensor *t = sized(bf16(o), N);
    if (!t) return false;
    *p = t->data_ptr();
    return true;
}

#define LQ_ARGS(n) \
    if (nargs != (n)) { PyErr_SetString(PyExc_TypeError, "wrong number of arguments"); return nullptr; }

// Whether something looks at calls that autograd itself does not: a trace being recorded, an open forward-mode level, an active
// function transform
bool watched() {
    const c10::DispatchKeySet included = c10::impl::tls_local_dispatch_key_set().included_;
    return torch::jit::tracer::isTracing() || torch::autograd::ForwardADLevel::try_get_by_idx(0) ||
           included.has(c10::DispatchKey::FuncTorchDynamicLayerFrontMode) || included.has(c10::DispatchKey::FuncTorchDynamicLayerBackMode);
}

// x, codes, scales, zeros, N, K, bias, workspace -> y
PyObject *linear4(PyObject *, PyObject *const *a, Py_ssize_t nargs) {
    LQ_ARGS(8)
    const int64_t N = integer(a[4]), K = integer(a[5]);
    const at::Tensor *x = bf16(a[0]);
    const int64_t M = rows_of(x, K);
    W4 w;
    const void *bias;
    void *ws;
    int64_t ws_bytes;
    if (M <= 0 || !w.load(a + 1, N, K) || !same_device(x, w.codes) || !bias_of(a[6], N, &bias) || !workspace(a[7], x, &ws, &ws_bytes))
        return none();
    On on(*x);
    at::Tensor y = make_rows(*x, N, at::kBFloat16);
    LQ_CALL(lq_a16w4_fwd_ws, x->data_ptr(), w.codes->data_ptr(), w.scales->data_ptr(), w.zeros->data_ptr(), bias, y.data_ptr(), M, N,
            K, LQ_GROUP, ws, ws_bytes, on.stream);
    return wrap(std::move(y));
}

// x, codes, scales, zeros, N, K, bias -> y, for a layer in inference: the whole call where nothing watches and the tokens
// are few enough to need no workspace
PyObject *linear4_eval(PyObject *self, PyObject *const *a, Py_ssize_t nargs) {
    LQ_ARGS(7)
    const int64_t K = integer(a[5]);
    const at::Tensor *x = bf16(a[0]);
    if (!x || K <= 0 || x->numel() > 16 * K || watched()) return none();
    PyObject *all[8] = {a[0], a[1], a[2], a[3], a[4], a[5], a[6], Py_None};
    return linear4(self, all, 8);
}

// dy, codes, scales, zeros, N, K, workspace -> dx
PyObject *dx4(PyObject *, PyObject *const *a, Py_ssize_t nargs) {
    LQ_ARGS(7)
    const int64_t N = integer(a[4]), K = integer(a[5]);
    const at::Tensor *dy = bf16(a[0]);
    const int64_t M = rows_of(dy, N);
    W4 w;
    void *ws;
    int64_t ws_bytes;
    if (M <= 0 || !w.load(a + 1, N, K) || !same_device(dy, w.codes) || !workspace(a[6], dy, &ws, &ws_bytes)) return none();
    On on(*dy);
    at::Tensor dx = make_rows(*dy, K, at::kBFloat16);
    LQ_CALL(lq_a16w4_dx_ws, dy->data_ptr(), w.codes->data_ptr(), w.scales->data_ptr(), w.zeros->data_ptr(), dx.data_ptr(), M, N, K,
            LQ_GROUP, ws, ws_bytes, on.stream);
    return wrap(std::move(dx));
}

// x, gate (codes, scales, zeros), up (codes, scales, zeros), N, K, save, workspace -> h, or (h, g, u)
PyObject *gate_up(PyObject *, PyObject *const *a, Py_ssize_t nargs) {
    LQ_ARGS(11)
    const int64_t N = integer(a[7]), K = integer(a[8]);
    const bool save = a[9] == Py_True;
    const at::Tensor *x = bf16(a[0]);
    const int64_t M = rows_of(x, K);
    W4 g, u;
    void *ws;
    int64_t ws_bytes;
    if (M <= 0 || !g.load(a + 1, N, K) || !u.load(a + 4, N, K) || !same_device(x, g.codes) || !same_device(x, u.codes) ||
        !workspace(a[10], x, &ws, &ws_bytes))
        return none();
    On on(*x);
    at::Tensor h = make_rows(*x, N, at::kBFloat16), go, uo;
    if (save) go = make_rows(*x, N, at::kBFloat16), uo = make_rows(*x, N, at::kBFloat16);
    LQ_CALL(lq_a16w4_gate_up_silu_ws, x->data_ptr(), g.codes->data_ptr(), g.scales->data_ptr(), g.zeros->data_ptr(),
            u.codes->data_ptr(), u.scales->data_ptr(), u.zeros->data_ptr(), h.data_ptr(), save ? go.data_ptr() : nullptr,
            save ? uo.data_ptr() : nullptr, M, N, K, LQ_GROUP, ws, ws_bytes, on.stream);
    if (!save) return wrap(std::move(h));
    return Py_BuildValue("NNN", wrap(std::move(h)), wrap(std::move(go)), wrap(std::move(uo)));
}

// dy, codes, scales, zeros, N, K, g, u -> (dg, du)
PyObject *dx_silu(PyObject *, PyObject *const *a, Py_ssize_t nargs) {
    LQ_ARGS(8)
    const int64_t N = integer(a[4]), K = integer(a[5]);
    const at::Tensor *dy = bf16(a[0]), *g = bf16(a[6]), *u = bf16(a[7]);
    const int64_t M = rows_of(dy, N);
    W4 w;
    if (M <= 0 || !w.load(a + 1, N, K) || !same_device(dy, w.codes) || rows_of(g, K) != M || rows_of(u, K) != M ||
        !same_device(dy, g) || !same_device(dy, u))
        return none();
    On on(*dy);
    at::Tensor dg = make_rows(*dy, K, at::kBFloat16), du = make_rows(*dy, K, at::kBFloat16);
    LQ_CALL(lq_a16w4_dx_silu_bwd, dy->data_ptr(), w.codes->data_ptr(), w.scales->data_ptr(), w.zeros->data_ptr(), g->data_ptr(),
            u->data_ptr(), dg.data_ptr(), du.data_ptr(), M, N, K, LQ_GROUP, on.stream);
    return Py_BuildValue("NN", wrap(std::move(dg)), wrap(std::move(du)));
}

// dy1, w1 (3), dy2, w2 (3), N, K, workspace -> dx
PyObject *dx_pair(PyObject *, PyObject *const *a, Py_ssize_t nargs) {
    LQ_ARGS(11)
    const int64_t N = integer(a[8]), K = integer(a[9]);
    const at::Tensor *d1 = bf16(a[0]), *d2 = bf16(a[4]);
    const int64_t M = rows_of(d1, N);
    W4 w1, w2;
    void *ws;
    int64_t ws_bytes;
    if (M <= 0 || rows_of(d2, N) != M || !w1.load(a + 1, N, K) || !w2.load(a + 5, N, K) || !same_device(d1, w1.codes) ||
        !same_device(d1, d2) || !same_device(d1, w2.codes) || !workspace(a[10], d1, &ws, &ws_bytes))
        return none();
    On on(*d1);
    at::Tensor dx = make_rows(*d1, K, at::kBFloat16);
    LQ_CALL(lq_a16w4_dx_pair_ws, d1->data_ptr(), w1.codes->data_ptr(), w1.scales->data_ptr(), w1.zeros->data_ptr(), d2->data_ptr(),
            w2.codes->data_ptr(), w2.scales->data_ptr(), w2.zeros->data_ptr(), dx.data_ptr(), M, N, K, LQ_GROUP, ws,
            ws_bytes, on.stream);
    return wrap(std::move(dx));
}

// x8, w8, sx, sw (fp32 or bf16), bias -> y
PyObject *linear8(PyObject *, PyObject *const *a, Py_ssize_t nargs) {
    LQ_ARGS(5)
    const at::Tensor *x = plain(a[0], at::kChar), *w = plain(a[1], at::kChar), *sx = plain(a[2], at::kFloat), *sw = plain(a[3], at::kFloat);
    const bool fp32 = sw != nullptr;
    if (!sw) sw = bf16(a[3]);
    if (!x || !w || !sx || !sw || w->dim() != 2 || w->numel() == 0) return none();
    const int64_t N = w->size(0), K = w->size(1), M = rows_of(x, K);
    const void *bias;
    if (M <= 0 || sx->numel() != M || sw->numel() != N || !bias_of(a[4], N, &bias) || !same_device(x, w) || !same_device(x, sx) ||
        !same_device(x, sw))
        return none();
    On on(*x);
    at::Tensor y = make_rows(*x, N, at::kBFloat16);
    if (fp32)
        LQ_CALL(lq_a8w8_fwd, x->data_ptr(), w->data_ptr(), (const float *)sx->data_ptr(), (const float *)sw->data_ptr(), bias,
                y.data_ptr(), nullptr, M, N, K, on.stream);
    else
        LQ_CALL(lq_a8w8_fwd_qs, x->data_ptr(), w->data_ptr(), (const float *)sx->data_ptr(), sw->data_ptr(), bias, y.data_ptr(),
                nullptr, M, N, K, on.stream);
    return wrap(std::move(y));
}

// x, w8, qscales, bias, per_token -> y: the forward of an 8-bit layer in inference (quantise the activations, int8 product)
PyObject *infer8(PyObject *, PyObject *const *a, Py_ssize_t nargs) {
    LQ_ARGS(5)
    const at::Tensor *x = bf16(a[0]), *w = plain(a[1], at::kChar), *qs = bf16(a[2]);
    if (!x || !w || !qs || w->dim() != 2 || w->numel() == 0) return none();
    const int64_t N = w->size(0), K = w->size(1), M = rows_of(x, K);
    const void *bias;
    if (M <= 0 || K % 8 || qs->numel() != N || !bias_of(a[3], N, &bias) || !same_device(x, w) || !same_device(x, qs)) return none();
    On on(*x);
    at::Tensor y = make_rows(*x, N, at::kBFloat16);
    if (aligned16(x) && aligned16(w) && lq_a8w8_infer_takes(M, N, K)) {
        LQ_CALL(lq_a8w8_infer, x->data_ptr(), w->data_ptr(), qs->data_ptr(), bias, y.data_ptr(), a[4] == Py_True, M, N, K, on.stream);
        return wrap(std::move(y));
    }
    // what the quantiser leaves for the product, in one allocation: x8 [M, K], sx [M], the quantiser's scratch
    const int64_t at_sx = (M * K + 15) / 16 * 16, at_work = at_sx + (M * 4 + 15) / 16 * 16;
    at::Tensor scratch = make({at_work + LQ_ACT_WORK_FLOATS * 4}, at::kByte, *x);
    uint8_t *p = (uint8_t *)scratch.data_ptr();
    int8_t *x8 = (int8_t *)p;
    float *sx = (float *)(p + at_sx), *work = (float *)(p + at_work);
    if (a[4] == Py_True)
        LQ_CALL(lq_act_quant_i8_per_token, x->data_ptr(), x8, sx, M, K, on.stream);
    else
        LQ_CALL(lq_act_quant_i8_dynamic, x->data_ptr(), x8, sx, work, M, K, 0, on.stream);
    LQ_CALL(lq_a8w8_fwd_qs, x8, w->data_ptr(), sx, qs->data_ptr(), bias, y.data_ptr(), nullptr, M, N, K, on.stream);
    return wrap(std::move(y));
}

// The same for a layer in inference: None where something watches
PyObject *infer8_eval(PyObject *self, PyObject *const *a, Py_ssize_t nargs) {
    return watched() ? none() : infer8(self, a, nargs);
}

// dy, w8, qscales, workspace -> dx
PyObject *dx8(PyObject *, PyObject *const *a, Py_ssize_t nargs) {
    LQ_ARGS(4)
    const at::Tensor *dy = bf16(a[0]), *w = plain(a[1], at::kChar), *qs = bf16(a[2]);
    if (!dy || !w || !qs || w->dim() != 2 || w->numel() == 0) return none();
    const int64_t N = w->size(0), K = w->size(1), M = rows_of(dy, N);
    void *ws;
    int64_t ws_bytes;
    if (M <= 0 || qs->numel() != N || N % 64 || K % 128 || !aligned16(dy) || !aligned16(w) || !same_device(dy, w) || !same_device(dy, qs) ||
        !workspace(a[3], dy, &ws, &ws_bytes))
        return none();
    On on(*dy);
    at::Tensor dx = make_rows(*dy, K, at::kBFloat16);
    LQ_CALL(lq_a8w8_dx_ws, dy->data_ptr(), w->data_ptr(), qs->data_ptr(), dx.data_ptr(), M, N, K, ws, ws_bytes, on.stream);
    return wrap(std::move(dx));
}

// x, alpha_bf16 -> (x8, sx, work)
PyObject *quant8(PyObject *, PyObject *const *a, Py_ssize_t nargs) {
    LQ_ARGS(2)
    const at::Tensor *x = bf16(a[0]);
    if (!x || x->dim() != 2 || x->numel() == 0) return none();
    const int64_t M = x->size(0), K = x->size(1);
    On on(*x);
    at::Tensor x8 = make(x->sizes(), at::kChar, *x), sx = make({M}, at::kFloat, *x), work = make({LQ_ACT_WORK_FLOATS}, at::kFloat, *x);
    LQ_CALL(lq_act_quant_i8_dynamic, x->data_ptr(), (int8_t *)x8.data_ptr(), (float *)sx.data_ptr(), (float *)work.data_ptr(), M, K,
            a[1] == Py_True, on.stream);
    return Py_BuildValue("NNN", wrap(std::move(x8)), wrap(std::move(sx)), wrap(std::move(work)));
}

// x -> (x8, sx)
PyObject *quant8_token(PyObject *, PyObject *const *a, Py_ssize_t nargs) {
    LQ_ARGS(1)
    const at::Tensor *x = bf16(a[0]);
    if (!x || x->dim() != 2 || x->numel() == 0 || x->size(1) % 8) return none();
    const int64_t M = x->size(0), K = x->size(1);
    On on(*x);
    at::Tensor x8 = make(x->sizes(), at::kChar, *x), sx = make({M}, at::kFloat, *x);
    LQ_CALL(lq_act_quant_i8_per_token, x->data_ptr(), (int8_t *)x8.data_ptr(), (float *)sx.data_ptr(), M, K, on.stream);
    return Py_BuildValue("NN", wrap(std::move(x8)), wrap(std::move(sx)));
}

// x8, scale, per_token -> x
PyObject *dequant8(PyObject *, PyObject *const *a, Py_ssize_t nargs) {
    LQ_ARGS(3)
    const at::Tensor *x8 = plain(a[0], at::kChar), *scale = plain(a[1], at::kFloat);
    if (!x8 || !scale || x8->dim() != 2 || x8->numel() == 0 || x8->size(1) % 16 || !aligned16(x8) || !same_device(x8, scale)) return none();
    const bool per_token = a[2] == Py_True;
    const int64_t M = x8->size(0), K = x8->size(1);
    if (scale->numel() != (per_token ? M : 1)) return none();
    On on(*x8);
    at::Tensor x = make(x8->sizes(), at::kBFloat16, *x8);
    LQ_CALL(lq_act_dequant_i8, (const int8_t *)x8->data_ptr(), (const float *)scale->data_ptr(), per_token, x.data_ptr(), M, K, on.stream);
    return wrap(std::move(x));
}

// The operands of a weight gradient: 2-D, the same tokens, sizes the GEMM takes
bool dw_operands(PyObject *const *a, const at::Tensor **dy, const at::Tensor **x, int k_mult) {
    *dy = bf16(a[0]);
    *x = bf16(a[1]);
    return *dy && *x && (*dy)->dim() == 2 && (*x)->dim() == 2 && (*dy)->size(0) == (*x)->size(0) && (*dy)->size(0) > 0 &&
           (*dy)->size(1) > 0 && (*dy)->size(1) % 8 == 0 && (*x)->size(1) > 0 && (*x)->size(1) % k_mult == 0 &&
           aligned16(*dy) && aligned16(*x) && same_device(*dy, *x);
}

// dy, x -> dW
PyObject *weight_grad(PyObject *, PyObject *const *a, Py_ssize_t nargs) {
    LQ_ARGS(2)
    const at::Tensor *dy, *x;
    if (!dw_operands(a, &dy, &x, 8)) return none();
    const int64_t M = dy->size(0), N = dy->size(1), K = x->size(1);
    On on(*dy);
    at::Tensor dw = make({N, K}, at::kBFloat16, *dy);
    LQ_CALL(lq_weight_grad, dy->data_ptr(), x->data_ptr(), dw.data_ptr(), M, N, K, on.stream);
    return wrap(std::move(dw));
}

// dy, x, g -> g, dW added onto it
PyObject *weight_grad_acc(PyObject *, PyObject *const *a, Py_ssize_t nargs) {
    LQ_ARGS(3)
    const at::Tensor *dy, *x, *g = bf16(a[2]);
    if (!dw_operands(a, &dy, &x, 8)) return none();
    const int64_t M = dy->size(0), N = dy->size(1), K = x->size(1);
    if (!g || g->dim() != 2 || g->size(0) != N || g->size(1) != K || !same_device(dy, g) || !aligned16(g)) return none();
    On on(*dy);
    LQ_CALL(lq_weight_grad_acc, dy->data_ptr(), x->data_ptr(), g->data_ptr(), M, N, K, on.stream);
    Py_INCREF(a[2]);
    return a[2];
}

// dy, x, q, scale, seed, offset -> q, dW added to the int8 accumulator
PyObject *weight_grad_acc8(PyObject *, PyObject *const *a, Py_ssize_t nargs) {
    LQ_ARGS(6)
    const at::Tensor *dy, *x, *q = plain(a[2], at::kChar), *scale = bf16(a[3]);
    if (!dw_operands(a, &dy, &x, 16)) return none();
    const int64_t M = dy->size(0), N = dy->size(1), K = x->size(1);
    if (!q || q->dim() != 2 || q->size(0) != N || q->size(1) != K || !sized(scale, N) || !same_device(dy, q) || !same_device(dy, scale))
        return none();
    const uint64_t seed = PyLong_AsUnsignedLongLongMask(a[4]), offset = PyLong_AsUnsignedLongLongMask(a[5]);
    On on(*dy);
    LQ_CALL(lq_weight_grad_acc8, dy->data_ptr(), x->data_ptr(), (int8_t *)q->data_ptr(), scale->data_ptr(), M, N, K, nullptr, seed, offset,
            on.stream);
    Py_INCREF(a[2]);
    return a[2];
}

// dw, q, scale, accumulate, seed, offset -> q
PyObject *gradq8(PyObject *, PyObject *const *a, Py_ssize_t nargs) {
    LQ_ARGS(6)
    const at::Tensor *dw = bf16(a[0]), *q = plain(a[1], at::kChar), *scale = bf16(a[2]);
    if (!dw || dw->dim() != 2 || dw->numel() == 0 || !q || q->sizes() != dw->sizes() || !sized(scale, dw->size(0)) ||
        !same_device(dw, q) || !same_device(dw, scale))
        return none();
    const uint64_t seed = PyLong_AsUnsignedLongLongMask(a[4]), offset = PyLong_AsUnsignedLongLongMask(a[5]);
    On on(*dw);
    LQ_CALL(lq_gradq8_quant, dw->data_ptr(), (int8_t *)q->data_ptr(), scale->data_ptr(), a[3] == Py_True, dw->size(0), dw->size(1),
            nullptr, seed, offset, on.stream);
    Py_INCREF(a[1]);
    return a[1];
}

// The operands every form of the optimizer step shares: grad, state1, state2, scale1, max1, scale2, max2
struct Adam {
    const at::Tensor *grad, *s1, *s2, *blocks[4];
    float *f[4];
    int64_t n, block;
    bool load(PyObject *const *o) {
        grad = bf16(o[0]);
        if (!grad || grad->numel() == 0) return false;
        n = grad->numel();
        s1 = sized(plain(o[1], at::kByte), n);
        s2 = sized(plain(o[2], at::kByte), n);
        if (!s1 || !s2 || !same_device(grad, s1) || !same_device(grad, s2)) return false;
        int64_t nblk = 0;
        for (int i = 0; i < 4; ++i) {
            const at::Tensor *t = plain(o[3 + i], at::kFloat);
            if (!t || !same_device(grad, t) || (i ? t->numel() != nblk : (nblk = t->numel()) == 0)) return false;
            blocks[i] = t;
            f[i] = (float *)t->data_ptr();
        }
        block = n / nblk;
        return n % nblk == 0;
    }
    uint8_t *p1() const { return (uint8_t *)s1->data_ptr(); }
    uint8_t *p2() const { return (uint8_t *)s2->data_ptr(); }
};

bool doubles(PyObject *const *o, double *v, int n) {
    for (int i = 0; i < n; ++i) {
        v[i] = PyFloat_AsDouble(o[i]);
        if (v[i] == -1.0 && PyErr_Occurred()) {
            PyErr_Clear();
            return false;
        }
    }
    return true;
}

// grad, state1, state2, scale1, max1, scale2, max2, beta1, beta2, eps, step_size, param -> param
PyObject *adam8_param(PyObject *, PyObject *const *a, Py_ssize_t nargs) {
    LQ_ARGS(12)
    Adam s;
    double v[4];
    const at::Tensor *p = bf16(a[11]);
    if (!s.load(a) || !doubles(a + 7, v, 4) || !sized(p, s.n) || !same_device(p, s.grad)) return none();
    On on(*s.grad);
    LQ_CALL(lq_adam8_update, s.grad->data_ptr(), p->data_ptr(), nullptr, s.p1(), s.p2(), s.f[0], s.f[1], s.f[2], s.f[3], s.n, (int)s.block,
            v[0], v[1], v[2], v[3], on.stream);
    Py_INCREF(a[11]);
    return a[11];
}

// Steps of several parameters that one launch will run: what is queued, on which stream, and the tensors it works on
#define ADAM_STATE(s) (s).s1, (s).s2, (s).blocks[0], (s).blocks[1], (s).blocks[2], (s).blocks[3]
struct AdamQueue {
    void *items = nullptr;
    void *stream = nullptr;
    c10::Device device{c10::kCPU};
    std::vector<at::Tensor> keep;
    ~AdamQueue() { lq_adam8_queue_free(items); }
    static constexpr const char *kName = "adam8_queue";

    // The queue to append to, or null to run the step now: no queue given, or one of another stream or device. The tensors
    // stay referenced until the queue is run.
    static void *take(PyObject *o, const On &on, const at::Tensor &like, std::initializer_list<const at::Tensor *> used) {
        if (!PyCapsule_IsValid(o, kName)) return nullptr;
        AdamQueue *q = static_cast<AdamQueue *>(PyCapsule_GetPointer(o, kName));
        if (q->keep.empty()) {
            q->stream = on.stream;
            q->device = like.device();
        }
        if (q->stream != on.stream || q->device != like.device()) return nullptr;
        for (const at::Tensor *t : used) q->keep.push_back(*t);
        return q->items;
    }
};

// -> a queue
PyObject *adam8_queue(PyObject *, PyObject *const *, Py_ssize_t nargs) {
    LQ_ARGS(0)
    AdamQueue *q = new AdamQueue;
    if (lq_adam8_queue_new(&q->items) != LQ_OK) {
        delete q;
        return PyErr_NoMemory();
    }
    PyObject *o = PyCapsule_New(q, AdamQueue::kName, [](PyObject *c) { delete static_cast<AdamQueue *>(PyCapsule_GetPointer(c, AdamQueue::kName)); });
    if (!o) delete q;
    return o;
}

// queue ->: runs what is in it
PyObject *adam8_run(PyObject *, PyObject *const *a, Py_ssize_t nargs) {
    LQ_ARGS(1)
    AdamQueue *q = static_cast<AdamQueue *>(PyCapsule_GetPointer(a[0], AdamQueue::kName));
    if (!q) return nullptr;
    if (q->keep.empty()) return none();
    c10::OptionalDeviceGuard guard(q->device);
    std::vector<at::Tensor> keep;  // until the launches are out
    keep.swap(q->keep);
    LQ_CALL(lq_adam8_queue_run, q->items, q->stream);
    return none();
}

// grad ... max2, beta1, beta2, eps, step_size, codes, scales, zeros, N, K, seed, offset, queue -> new codes
PyObject *adam8_sr(PyObject *, PyObject *const *a, Py_ssize_t nargs) {
    LQ_ARGS(19)
    Adam s;
    double v[4];
    const int64_t N = integer(a[14]), K = integer(a[15]);
    W4 w;
    if (!s.load(a) || !doubles(a + 7, v, 4) || !w.load(a + 11, N, K) || s.n != N * K || !same_device(s.grad, w.codes)) return none();
    const uint64_t seed = PyLong_AsUnsignedLongLongMask(a[16]), offset = PyLong_AsUnsignedLongLongMask(a[17]);
    On on(*s.grad);
    at::Tensor out = at::empty_like(*w.codes);
    void *queue = AdamQueue::take(a[18], on, *s.grad, {s.grad, w.codes, &out, w.scales, w.zeros, ADAM_STATE(s)});
    LQ_CALL(lq_adam8_sr_step_queued, s.grad->data_ptr(), w.codes->data_ptr(), out.data_ptr(), w.scales->data_ptr(), w.zeros->data_ptr(), s.p1(),
            s.p2(), s.f[0], s.f[1], s.f[2], s.f[3], N, K, LQ_GROUP, (int)s.block, v[0], v[1], v[2], v[3], seed, offset, on.stream, queue);
    return wrap(std::move(out));
}

// (k1, b1, k2, b2, k3) of a residual curve
struct Curve {
    int k1, k2, k3;
    float b1, b2;
    bool load(PyObject *o) {
        if (!PyTuple_CheckExact(o) || PyTuple_GET_SIZE(o) != 5) return false;
        double v[5];
        for (int i = 0; i < 5; ++i) {
            PyObject *e = PyTuple_GET_ITEM(o, i);
            if (!doubles(&e, v + i, 1)) return false;
        }
        k1 = (int)v[0]; k2 = (int)v[2]; k3 = (int)v[4];
        b1 = (float)v[1]; b2 = (float)v[3];
        return true;
    }
};

// grad ... max2, beta1, beta2, eps, step_size, codes, scales, zeros, N, K, residual, dequant curve, quant curve, queue -> codes
PyObject *adam8_w4(PyObject *, PyObject *const *a, Py_ssize_t nargs) {
    LQ_ARGS(20)
    Adam s;
    double v[4];
    const int64_t N = integer(a[14]), K = integer(a[15]);
    W4 w;
    Curve d, q;
    const at::Tensor *r = plain(a[16], at::kInt);
    if (!s.load(a) || !doubles(a + 7, v, 4) || !w.load(a + 11, N, K) || s.n != N * K || !sized(r, N * K / 8) || !d.load(a[17]) ||
        !q.load(a[18]) || !same_device(s.grad, w.codes) || !same_device(s.grad, r))
        return none();
    On on(*s.grad);
    void *queue = AdamQueue::take(a[19], on, *s.grad, {s.grad, w.codes, r, w.scales, w.zeros, ADAM_STATE(s)});
    LQ_CALL(lq_adam8_latent_w4_step_queued, s.grad->data_ptr(), w.codes->data_ptr(), (int32_t *)r->data_ptr(), w.scales->data_ptr(),
            w.zeros->data_ptr(), s.p1(), s.p2(), s.f[0], s.f[1], s.f[2], s.f[3], N, K, LQ_GROUP, (int)s.block, d.k1, d.b1, d.k2, d.b2,
            d.k3, q.k1, q.b1, q.k2, q.b2, q.k3, v[0], v[1], v[2], v[3], on.stream, queue);
    Py_INCREF(a[11]);
    return a[11];
}

// grad ... max2, beta1, beta2, eps, step_size, codes, qscales, residual, dequant curve, quant curve, queue -> codes
PyObject *adam8_w8(PyObject *, PyObject *const *a, Py_ssize_t nargs) {
    LQ_ARGS(17)
    Adam s;
    double v[4];
    Curve d, q;
    const at::Tensor *c = plain(a[11], at::kChar), *qs = bf16(a[12]), *r = plain(a[13], at::kInt);
    if (!s.load(a) || !doubles(a + 7, v, 4) || !c || c->dim() != 2 || c->numel() != s.n || c->size(1) % 8 || !sized(qs, c->size(0)) ||
        !sized(r, s.n / 8) || !d.load(a[14]) || !q.load(a[15]) || !same_device(s.grad, c) || !same_device(s.grad, qs) || !same_device(s.grad, r))
        return none();
    On on(*s.grad);
    void *queue = AdamQueue::take(a[16], on, *s.grad, {s.grad, c, r, qs, ADAM_STATE(s)});
    LQ_CALL(lq_adam8_latent_w8_step_queued, s.grad->data_ptr(), (int8_t *)c->data_ptr(), (int32_t *)r->data_ptr(), qs->data_ptr(), s.p1(), s.p2(),
            s.f[0], s.f[1], s.f[2], s.f[3], c->size(0), c->size(1), (int)s.block, d.k1, d.b1, d.k2, d.b2, d.k3, q.k1, q.b1, q.k2, q.b2,
            q.k3, v[0], v[1], v[2], v[3], on.stream, queue);
    Py_INCREF(a[11]);
    return a[11];
}

// device index -> the current stream's handle
PyObject *current_stream(PyObject *, PyObject *const *a, Py_ssize_t nargs) {
    LQ_ARGS(1)
    return PyLong_FromVoidPtr((void *)c10::hip::getCurrentHIPStreamMasqueradingAsCUDA((c10::DeviceIndex)integer(a[0])).stream());
}

PyObject *set_error(PyObject *, PyObject *const *a, Py_ssize_t nargs) {
    LQ_ARGS(1)
    Py_INCREF(a[0]);
    Py_XSETREF(g_error, a[0]);
    return none();
}

// x -> whether a layer in training can take its short way: activations in plain form, autograd records, and nothing looks at the call
// that is given the tensors of the Function over rows otherwise (a trace, a transform, hooks on saved tensors, a dispatch mode)
PyObject *records_plainly(PyObject *, PyObject *const *a, Py_ssize_t nargs) {
    LQ_ARGS(1)
    const at::Tensor *x = bf16(a[0]);
    return PyBool_FromLong(x && x->dim() >= 1 && x->numel() > 0 && c10::GradMode::is_enabled() && !c10::InferenceMode::is_enabled() &&
                           !watched() && !c10::impl::dispatch_mode_enabled() && at::SavedTensorDefaultHooks::get_tls_state().stack.empty());
}

#define LQ_METHOD(f) {#f, (PyCFunction)(void (*)(void))guarded<f>, METH_FASTCALL, nullptr}

// Until a thread has touched the thread-local storage of the library loaded last, its every access to that of another library (the tensor
// library's dispatch state and modes are full of them) goes the slow way through the C library's __tls_get_addr (glibc before 2.39, its bug
// 19924). This library is loaded at the first call of a program, behind those others, and a store brings the calling thread up to date:
// torch.empty_like on the GPU 1.15 -> 0.90 us, seven layers on four tokens, 1536 columns, 38 -> 35, six steps of the optimizer 69 -> 62.
thread_local volatile char touched;

// A C++ exception (out of memory, say) leaves as the Python exception the tensor library would raise
template <PyObject *(*F)(PyObject *, PyObject *const *, Py_ssize_t)>
PyObject *guarded(PyObject *self, PyObject *const *a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    touched = 1;
    PyObject *r = F(self, a, n);
    if (r && PyErr_Occurred()) {  // an argument that is no number
        Py_DECREF(r);
        return nullptr;
    }
    return r;
    END_HANDLE_TH_ERRORS
}

PyMethodDef methods[] = {
    LQ_METHOD(linear4), LQ_METHOD(linear4_eval), LQ_METHOD(dx4), LQ_METHOD(gate_up), LQ_METHOD(dx_silu), LQ_METHOD(dx_pair), LQ_METHOD(linear8), LQ_METHOD(infer8),
    LQ_METHOD(infer8_eval), LQ_METHOD(dx8), LQ_METHOD(quant8), LQ_METHOD(quant8_token), LQ_METHOD(dequant8), LQ_METHOD(weight_grad),
    LQ_METHOD(weight_grad_acc), LQ_METHOD(weight_grad_acc8), LQ_METHOD(gradq8), LQ_METHOD(adam8_param), LQ_METHOD(adam8_sr),
    LQ_METHOD(adam8_queue), LQ_METHOD(adam8_run), LQ_METHOD(adam8_w4), LQ_METHOD(adam8_w8), LQ_METHOD(current_stream),
    LQ_METHOD(records_plainly), LQ_METHOD(set_error), {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_lqbind", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__lqbind() { return PyModule_Create(&module); }
