// dabnn_amd._ops_native: the operators a program calls once per layer, from torch tensors to the C ABI without a detour
// through ctypes.  A call is a few microseconds of GPU work, and checking the tensors, finding the stream and
// marshalling a dozen arguments in Python took longer than that (10 us; 3 to 4 here, most of it the allocation of the
// result and the launch).
//
// Each function takes the arguments of its Python counterpart in dabnn_amd/ops.py, in order, and returns the result, or
// None when an argument is not the plain case (another type, a tensor on the host, not contiguous, an empty output, a
// size that does not match): the Python function then does what it does without this module, errors included.  An error
// code of the C ABI comes back as an int for capi.check.
#include <ATen/ATen.h>
#include <ATen/hip/EmptyTensor.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include <climits>

#include "../../include/dabnn_hip.h"

namespace {

constexpr int64_t kMostElements = int64_t(1) << 40;

struct Args {
    PyObject *const *v;
    bool ok = true;
    bool is_none(int i) const { return v[i] == Py_None; }
    const at::Tensor &tensor(int i, at::ScalarType type) {
        static const at::Tensor none;
        if (!THPVariable_Check(v[i])) return ok = false, none;
        const at::Tensor &t = THPVariable_Unpack(v[i]);
        if (!t.is_cuda() || t.scalar_type() != type || !t.is_contiguous() || t.requires_grad()) return ok = false, none;
        return t;
    }
    int integer(int i) {
        if (!PyLong_CheckExact(v[i])) return ok = false, 0;
        const long long x = PyLong_AsLongLong(v[i]);
        if (x < -(1ll << 30) || x > (1ll << 30)) {
            PyErr_Clear();
            ok = false;
        }
        return (int)x;
    }
};

PyObject *none() { Py_RETURN_NONE; }

dab_stream_t stream_of(const at::Tensor &t) {
    return reinterpret_cast<dab_stream_t>(c10::hip::getCurrentHIPStream(t.device().index()).stream());
}

// The tensors of a call live on one device and it is the current one: the launch goes there.
bool on_current_device(const at::Tensor &t) { return t.device().index() == c10::hip::current_device(); }

template <class... T>
bool same_device(const at::Tensor &t, const T &...rest) {
    return on_current_device(t) && (... && (!rest.defined() || rest.device() == t.device()));
}

// every extent fits the C ABI's ints
bool small_extents(const at::Tensor &t) {
    for (const int64_t d : t.sizes())
        if (d > INT_MAX) return false;
    return true;
}

at::Tensor fresh(at::IntArrayRef shape, at::ScalarType type, const at::Tensor &like) {
    return at::detail::empty_cuda(shape, type, like.device(), std::nullopt);
}

int out_dim(int64_t size, int pad, int k, int stride) { return (int)((size + 2ll * pad - k) / stride + 1); }

PyObject *result(int rc, const at::Tensor &out) { return rc == DAB_OK ? THPVariable_Wrap(out) : PyLong_FromLong(rc); }

template <class T>
T *ptr(const at::Tensor &t) {
    return reinterpret_cast<T *>(t.data_ptr());
}

// pack_mat(x)
PyObject *pack_mat(PyObject *, PyObject *const *v, Py_ssize_t n) {
    Args a{v};
    if (n != 1) return none();
    const at::Tensor &x = a.tensor(0, at::kFloat);
    if (!a.ok || x.dim() < 1 || x.numel() == 0 || !same_device(x)) return none();
    const int64_t c = x.size(-1);
    if (c % 64 != 0 || c > (1 << 30)) return none();
    at::DimVector shape(x.sizes());
    shape.back() = c / 64;
    const at::Tensor out = fresh(shape, at::kLong, x);
    return result(dab_bitpack_nhwc(ptr<float>(x), ptr<uint64_t>(out), x.numel() / c, (int)c, stream_of(x)), out);
}

// A 3x3 convolution's operands and output shape
struct Conv3x3 {
    const at::Tensor &x, &w;
    int n, h, wd, cw, cout, stride, pad, oh, ow;
    bool ok;
    Conv3x3(Args &a, int stride_at, int pad_at) : x(a.tensor(0, at::kLong)), w(a.tensor(1, at::kLong)), stride(a.integer(stride_at)), pad(a.integer(pad_at)) {
        ok = a.ok && x.dim() == 4 && w.dim() >= 1 && x.numel() > 0 && x.numel() < kMostElements && stride > 0 && pad >= 0 && same_device(x, w) && small_extents(x) &&
             small_extents(w);
        if (!ok) return;
        n = (int)x.size(0), h = (int)x.size(1), wd = (int)x.size(2), cw = (int)x.size(3), cout = (int)w.size(0);
        ok = w.numel() == (int64_t)cout * 9 * cw && h + 2ll * pad >= 3 && wd + 2ll * pad >= 3;
        if (!ok) return;
        oh = out_dim(h, pad, 3, stride), ow = out_dim(wd, pad, 3, stride);
        ok = cout > 0 && (int64_t)n * oh * ow * cout < kMostElements;
    }
};

// bconv_3x3(x, weight, stride, pad)
PyObject *bconv_3x3(PyObject *, PyObject *const *v, Py_ssize_t n) {
    Args a{v};
    if (n != 4) return none();
    const Conv3x3 c(a, 2, 3);
    if (!c.ok) return none();
    const at::Tensor out = fresh({c.n, c.oh, c.ow, c.cout}, at::kFloat, c.x);
    return result(dab_bconv3x3(ptr<uint64_t>(c.x), c.n, c.h, c.wd, c.cw * 64, ptr<uint64_t>(c.w), c.cout, c.stride, c.pad, ptr<float>(out), stream_of(c.x)), out);
}

// bconv_3x3_affine_add(x, weight, a, b, shortcut, stride, pad), and with the sign-packed copy of the result
PyObject *fused_3x3(PyObject *const *v, Py_ssize_t n, bool sign) {
    Args a{v};
    if (n != 7) return none();
    const Conv3x3 c(a, 5, 6);
    if (!c.ok) return none();
    const at::Tensor &ca = a.tensor(2, at::kFloat), &cb = a.tensor(3, at::kFloat);
    at::Tensor shortcut;
    if (!a.is_none(4)) shortcut = a.tensor(4, at::kFloat);
    if (!a.ok || ca.numel() != c.cout || cb.numel() != c.cout || !same_device(c.x, ca, cb, shortcut)) return none();
    const std::array<int64_t, 4> shape{c.n, c.oh, c.ow, c.cout};
    if (shortcut.defined() && shortcut.sizes() != at::IntArrayRef(shape)) return none();
    if (sign && c.cout % 64 != 0) return none();
    const at::Tensor out = fresh(shape, at::kFloat, c.x);
    const float *sc = shortcut.defined() ? ptr<float>(shortcut) : nullptr;
    if (!sign)
        return result(dab_bconv3x3_affine_add(ptr<uint64_t>(c.x), c.n, c.h, c.wd, c.cw * 64, ptr<uint64_t>(c.w), c.cout, c.stride, c.pad, ptr<float>(ca),
                                              ptr<float>(cb), sc, ptr<float>(out), stream_of(c.x)),
                      out);
    const at::Tensor packed = fresh({c.n, c.oh, c.ow, c.cout / 64}, at::kLong, c.x);
    const int rc = dab_bconv3x3_affine_add_sign(ptr<uint64_t>(c.x), c.n, c.h, c.wd, c.cw * 64, ptr<uint64_t>(c.w), c.cout, c.stride, c.pad, ptr<float>(ca),
                                                ptr<float>(cb), sc, ptr<float>(out), ptr<uint64_t>(packed), stream_of(c.x));
    if (rc != DAB_OK) return PyLong_FromLong(rc);
    return Py_BuildValue("(NN)", THPVariable_Wrap(out), THPVariable_Wrap(packed));
}
PyObject *bconv_3x3_affine_add(PyObject *, PyObject *const *v, Py_ssize_t n) { return fused_3x3(v, n, false); }
PyObject *bconv_3x3_affine_add_sign(PyObject *, PyObject *const *v, Py_ssize_t n) { return fused_3x3(v, n, true); }

// bgemm(m, n, k, a, lda, b, ldb, c, ldc): the return value is c itself
PyObject *gemm(PyObject *const *v, Py_ssize_t nargs, bool overwrite) {
    Args a{v};
    if (nargs != 9) return none();
    const int m = a.integer(0), n = a.integer(1), k = a.integer(2), lda = a.integer(4), ldb = a.integer(6), ldc = a.integer(8);
    const at::Tensor &ta = a.tensor(3, at::kLong), &tb = a.tensor(5, at::kLong), &tc = a.tensor(7, at::kFloat);
    if (!a.ok || m <= 0 || n <= 0 || k <= 0 || lda <= 0 || ldb <= 0 || ldc <= 0 || !same_device(tc, ta, tb)) return none();
    if (ta.numel() < (k - 1ll) * lda + m || tb.numel() < (n - 1ll) * ldb + k || tc.numel() < (n - 1ll) * ldc + m) return none();
    const int rc = (overwrite ? dab_bgemm_overwrite : dab_bgemm)(m, n, k, ptr<uint64_t>(ta), lda, ptr<uint64_t>(tb), ldb, ptr<float>(tc), ldc, stream_of(tc));
    if (rc != DAB_OK) return PyLong_FromLong(rc);
    Py_INCREF(v[7]);
    return v[7];
}
PyObject *bgemm(PyObject *, PyObject *const *v, Py_ssize_t n) { return gemm(v, n, false); }
PyObject *bgemm_overwrite(PyObject *, PyObject *const *v, Py_ssize_t n) { return gemm(v, n, true); }

// binconv(x, weight, transposed_weight, workspace or None, kh, kw, pad_h, pad_w, stride_h, stride_w)
//   -> (out, method, workspace)
PyObject *binconv(PyObject *, PyObject *const *v, Py_ssize_t n) {
    Args a{v};
    if (n != 10) return none();
    const at::Tensor &x = a.tensor(0, at::kFloat), &w = a.tensor(1, at::kLong), &wt = a.tensor(2, at::kLong);
    at::Tensor ws;
    if (!a.is_none(3)) ws = a.tensor(3, at::kByte);
    int g[6];
    for (int i = 0; i < 6; ++i) g[i] = a.integer(4 + i);
    if (!a.ok || x.dim() != 4 || w.dim() != 2 || x.numel() == 0 || x.numel() >= kMostElements || !same_device(x, w, wt) || !small_extents(x) ||
        !small_extents(w))
        return none();
    for (int i = 0; i < 6; ++i)
        if (g[i] < (i == 2 || i == 3 ? 0 : 1)) return none();
    const int nn = (int)x.size(0), h = (int)x.size(1), wd = (int)x.size(2), c = (int)x.size(3), cout = (int)w.size(0);
    if (h + 2ll * g[2] < g[0] || wd + 2ll * g[3] < g[1] || cout <= 0) return none();
    const int oh = out_dim(h, g[2], g[0], g[4]), ow = out_dim(wd, g[3], g[1], g[5]);
    if ((int64_t)nn * oh * ow * cout >= kMostElements) return none();
    const size_t need = dab_binconv_workspace_bytes(nn, h, wd, c, g[0], g[1], g[2], g[3], g[4], g[5]);
    if (!ws.defined() || (size_t)ws.numel() < need || ws.device() != x.device()) ws = fresh({(int64_t)(need < 16 ? 16 : need)}, at::kByte, x);
    const at::Tensor out = fresh({nn, oh, ow, cout}, at::kFloat, x);
    int method = -1;
    const int rc = dab_binconv_forward(ptr<float>(x), nn, h, wd, c, ptr<uint64_t>(w), ptr<uint64_t>(wt), (int)w.size(1), g[0], g[1], g[2], g[3], g[4], g[5],
                                       cout, ptr<float>(out), ws.data_ptr(), (size_t)ws.numel(), &method, stream_of(x));
    if (rc != DAB_OK) return PyLong_FromLong(rc);
    return Py_BuildValue("(NiN)", THPVariable_Wrap(out), method, THPVariable_Wrap(ws));
}

// C++ exceptions of torch (an allocation that fails) become Python's
template <PyObject *(*F)(PyObject *, PyObject *const *, Py_ssize_t)>
PyObject *guarded(PyObject *self, PyObject *const *v, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    return F(self, v, n);
    END_HANDLE_TH_ERRORS
}

#define DAB_METHOD(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(guarded<name>)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {DAB_METHOD(pack_mat), DAB_METHOD(bconv_3x3),       DAB_METHOD(bconv_3x3_affine_add), DAB_METHOD(bconv_3x3_affine_add_sign),
                         DAB_METHOD(bgemm),    DAB_METHOD(bgemm_overwrite), DAB_METHOD(binconv),              {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_ops_native", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__ops_native() { return PyModule_Create(&module); }
