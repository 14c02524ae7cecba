// Native side of any_precision_ext, AnyPrecisionLinear and its sets: the checks, the allocation of the result and the launch of one
// call, as Python functions over torch tensors.
//
// A linear's kernel takes 4 to 15 us at the batch sizes of decoding; the same steps written in Python over ctypes take
// 11 to 15 us of host time per call, and a stream of such calls runs at the host's pace (28 linears of four decoder layers
// at one row and 3 bits: 400 us of which the GPU works 167).  Here a call takes about 5 us, most of it HIP's launch.
//
// A function returns None for anything it does not serve -- wrong types, shapes, devices, layouts -- and the Python side
// then takes the way that says what is wrong (or serves the case, where it can).  Errors of the library raise here.
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/autocast_mode.h>
#include <ATen/hip/EmptyTensor.h>
#include <ATen/hip/impl/HIPGuardImplMasqueradingAsCUDA.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <c10/core/GradMode.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include "anyprec_hip.h"

namespace {

using at::Tensor;

PyObject *none() { Py_RETURN_NONE; }

// A C++ exception becomes the Python exception that torch's own bindings make of it: a Python exception raised below (a hook's, a
// mode's) comes out as itself, exhausted memory as torch.OutOfMemoryError.  Warnings become Python warnings.
template <typename F>
PyObject *guarded(F &&f) {
    HANDLE_TH_ERRORS
    return f();
    END_HANDLE_TH_ERRORS
}

PyObject *library_error(int rc, const char *op) {
    if (rc < 0) PyErr_Format(PyExc_ValueError, "%s: %s (code %d)", op, ap_strerror(rc), rc);
    else PyErr_Format(PyExc_RuntimeError, "%s: HIP error %d: %s", op, rc, ap_strerror(rc));
    return nullptr;
}

bool is_tensor(PyObject *o) { return o != nullptr && THPVariable_Check(o); }
bool exact_tensor(PyObject *o) { return THPVariable_CheckTypeExact(Py_TYPE(o)); }  // or a parameter, but no other subclass

// A bit-width given as an int in 3..8, else 0.
int bits_of(PyObject *o) {
    if (!PyLong_Check(o) || PyBool_Check(o)) return 0;
    const long b = PyLong_AsLong(o);
    if (b == -1 && PyErr_Occurred()) PyErr_Clear();
    return b >= 3 && b <= 8 ? (int)b : 0;
}

struct Weight {
    const uint32_t *planes;
    const uint16_t *lut;
    int N, K;
    c10::DeviceIndex device;
};

bool weight_of(const Tensor &q, const Tensor &t, int bits, Weight *w) {
    if (!q.is_cuda() || q.scalar_type() != at::kInt || q.dim() != 3 || !q.is_contiguous()) return false;
    if (!t.is_cuda() || t.scalar_type() != at::kHalf || t.dim() != 2 || !t.is_contiguous() || t.device() != q.device()) return false;
    const int64_t planes = q.size(0), N = q.size(1), W = q.size(2);
    if (planes < bits || N < 1 || W < 1 || N > INT32_MAX || W > INT32_MAX / 32) return false;
    if (t.size(0) != N || t.size(1) != (int64_t)1 << bits) return false;
    w->planes = reinterpret_cast<const uint32_t *>(q.data_ptr());
    w->lut = reinterpret_cast<const uint16_t *>(t.data_ptr());
    w->N = (int)N;
    w->K = (int)(W * 32);
    w->device = q.device().index();
    return true;
}

// Activation rows of x for a linear of K inputs, or 0.
int64_t rows_of(const Tensor &x, const Weight &w) {
    if (!x.is_cuda() || x.scalar_type() != at::kHalf || x.dim() < 1 || x.device().index() != w.device) return 0;
    if (x.size(-1) != w.K) return 0;
    const int64_t rows = x.numel() / w.K;
    return rows <= INT32_MAX ? rows : 0;
}

const uint16_t *half_ptr(const Tensor &t) { return reinterpret_cast<const uint16_t *>(t.data_ptr()); }
uint16_t *half_out(const Tensor &t) { return reinterpret_cast<uint16_t *>(t.data_ptr()); }

Tensor empty_half(at::IntArrayRef shape, const at::Device &device) {
    return Tensor(at::detail::empty_cuda(shape, at::kHalf, device, std::nullopt));
}

// A result of x's leading dimensions and N columns.
Tensor result_for(const Tensor &x, int64_t N) {
    c10::SmallVector<int64_t, 6> shape(x.sizes().begin(), x.sizes().end());
    shape.back() = N;
    return empty_half(shape, x.device());
}

// Makes the tensors' device the current one for a call (a no-op where it is) and gives its current stream.
struct OnDevice {
    explicit OnDevice(c10::DeviceIndex d) {
        if (c10::hip::current_device() != d) guard.set_index(d);
        stream = static_cast<void *>(c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(d).stream());
    }
    c10::hip::OptionalHIPGuardMasqueradingAsCUDA guard;
    void *stream;
};

// Other Python threads run meanwhile: a launch may wait for its queue, an allocation for the device.  Nothing in the scope
// touches Python, and tensors that come from a module's dicts are held by copies: a thread may replace them meanwhile.
struct WithoutGil {
    WithoutGil() : state(PyEval_SaveThread()) {}
    ~WithoutGil() { PyEval_RestoreThread(state); }
    WithoutGil(const WithoutGil &) = delete;
    WithoutGil &operator=(const WithoutGil &) = delete;
    PyThreadState *state;
};

PyObject *wrap(Tensor t) { return THPVariable_Wrap(std::move(t)); }

// matmul_kbit(x, qweight, lut, w_bits) and gemm_kbit(x, qweight, lut, w_bits)
PyObject *product(PyObject *const *args, Py_ssize_t n, bool gemm) {
    if (n != 4 || !is_tensor(args[0]) || !is_tensor(args[1]) || !is_tensor(args[2])) return none();
    const int bits = bits_of(args[3]);
    if (bits == 0) return none();
    return guarded([&]() -> PyObject * {
        const Tensor &x = THPVariable_Unpack(args[0]);
        Weight w;
        if (!weight_of(THPVariable_Unpack(args[1]), THPVariable_Unpack(args[2]), bits, &w)) return none();
        const int64_t rows = rows_of(x, w);
        if (rows < 1 || (!gemm && rows > 8) || !x.is_contiguous()) return none();
        Tensor out;
        int rc;
        {
            const WithoutGil free;
            const OnDevice on(w.device);
            out = result_for(x, w.N);
            rc = gemm ? ap_gemm_kbit(half_ptr(x), w.planes, w.lut, half_out(out), (int)rows, w.N, w.K, bits, on.stream)
                      : ap_matmul_kbit(half_ptr(x), w.planes, w.lut, half_out(out), (int)rows, w.N, w.K, bits, on.stream);
        }
        if (rc != AP_OK) return library_error(rc, gemm ? "gemm_kbit" : "matmul_kbit");
        return wrap(std::move(out));
    });
}

PyObject *matmul_kbit(PyObject *, PyObject *const *args, Py_ssize_t n) { return product(args, n, false); }
PyObject *gemm_kbit(PyObject *, PyObject *const *args, Py_ssize_t n) { return product(args, n, true); }

PyObject *dequant_kbit(PyObject *, PyObject *const *args, Py_ssize_t n) {
    if (n != 3 || !is_tensor(args[0]) || !is_tensor(args[1])) return none();
    const int bits = bits_of(args[2]);
    if (bits == 0) return none();
    return guarded([&]() -> PyObject * {
        const Tensor &q = THPVariable_Unpack(args[0]);
        Weight w;
        if (!weight_of(q, THPVariable_Unpack(args[1]), bits, &w)) return none();
        Tensor out;
        int rc;
        {
            const WithoutGil free;
            const OnDevice on(w.device);
            out = empty_half({w.N, w.K}, q.device());
            rc = ap_dequant_kbit(w.planes, w.lut, half_out(out), w.N, w.K, bits, on.stream);
        }
        if (rc != AP_OK) return library_error(rc, "dequant_kbit");
        return wrap(std::move(out));
    });
}

// Some functions of this module replace torch ops, which take part in everything torch does with an op: a call that anything but plain execution follows -- gradients, tangents, subclasses, modes, functorch --
// gets None and runs as torch ops.
bool plain_half(PyObject *o, const at::Device *device) {
    if (!is_tensor(o) || !exact_tensor(o)) return false;
    const Tensor &t = THPVariable_Unpack(o);
    if (!t.is_cuda() || t.scalar_type() != at::kHalf || t.layout() != at::kStrided || !t.is_contiguous() || t.numel() == 0) return false;
    if (device != nullptr && t.device() != *device) return false;
    if (c10::GradMode::is_enabled() && t.requires_grad()) return false;
    const auto keys = t.key_set();
    if (keys.has(c10::DispatchKey::FuncTorchBatched) || keys.has(c10::DispatchKey::FuncTorchGradWrapper) ||
        keys.has(c10::DispatchKey::Functionalize) || keys.has(c10::DispatchKey::Negative) || keys.has(c10::DispatchKey::ZeroTensor) ||
        t._fw_grad(0).defined())
        return false;
    return (reinterpret_cast<uintptr_t>(t.data_ptr()) & 15u) == 0;
}

bool plain_execution() {
    return !c10::impl::TorchDispatchModeTLS::any_modes_set() && !at::impl::torch_function_mode_enabled() &&
           !c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode) &&
           !c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::Tracer);
}

// Whether torch's product of fp16 operands gives fp16 results: under autocast it gives autocast's type.
bool product_is_half() { return !at::autocast::is_autocast_enabled(at::kCUDA) || at::autocast::get_autocast_dtype(at::kCUDA) == at::kHalf; }

// Names in a module's dicts, made once.
PyObject *key_buffers, *key_qweight, *key_bias, *key_lut[9];

// The tensors of one AnyPrecisionLinear, read from its __dict__ in the order of nn.Module's attribute lookup.
struct ModuleTensors {
    PyObject *qweight, *table, *bias;  // bias: null where the module has none
};

// False where a tensor is not a buffer: a bias may also be a parameter (assigned, loaded with assign=True) or the result of a
// parametrisation, and then shows in neither dict.
bool tensors_of(PyObject *module_dict, int bits, ModuleTensors *m) {
    if (!PyDict_Check(module_dict)) return false;
    PyObject *buffers = PyDict_GetItem(module_dict, key_buffers);
    if (buffers == nullptr || !PyDict_Check(buffers)) return false;
    m->qweight = PyDict_GetItem(buffers, key_qweight);
    m->table = PyDict_GetItem(buffers, key_lut[bits]);
    m->bias = PyDict_GetItem(module_dict, key_bias);
    if (m->bias == nullptr) m->bias = PyDict_GetItem(buffers, key_bias);
    if (m->bias == nullptr) return false;
    if (m->bias == Py_None) m->bias = nullptr;
    return is_tensor(m->qweight) && is_tensor(m->table) && (m->bias == nullptr || is_tensor(m->bias));
}

// linear(module.__dict__, x, w_bits): AnyPrecisionLinear.forward.  ap_linear up to 8 rows, and beyond
// where ap_gemm_kbit_pays, or ap_gemm_kbit_quick and nothing but plain execution follows the call; else the weight in fp16 and
// torch's own product (which takes part in autograd and autocast).
PyObject *linear(PyObject *, PyObject *const *args, Py_ssize_t n) {
    if (n != 3 || !is_tensor(args[1])) return none();
    const int bits = bits_of(args[2]);
    ModuleTensors m;
    if (bits == 0 || !tensors_of(args[0], bits, &m)) return none();
    return guarded([&]() -> PyObject * {
        const Tensor &x = THPVariable_Unpack(args[1]);
        const Tensor q = THPVariable_Unpack(m.qweight), t = THPVariable_Unpack(m.table);
        const Tensor bias = m.bias == nullptr ? Tensor() : THPVariable_Unpack(m.bias);
        Weight w;
        if (!weight_of(q, t, bits, &w)) return none();
        const int64_t rows = rows_of(x, w);
        if (rows < 1) return none();
        const bool pays = rows <= 8 || ap_gemm_kbit_pays((int)rows, w.N, w.K, bits) == 1 ||
                          (ap_gemm_kbit_quick((int)rows, w.N, w.K, bits) == 1 && plain_execution() && product_is_half() && plain_half(args[1], nullptr));
        // torch's product and sum as Python calls them, where a subclass or a mode wants to see them
        const bool torch_op = !pays || bias.defined();
        if (torch_op && (at::impl::torch_function_mode_enabled() || !exact_tensor(args[1]) || (m.bias != nullptr && !exact_tensor(m.bias))))
            return none();
        const char *op = rows <= 8 ? "matmul_kbit" : "gemm_kbit";
        // a bias that is N plain numbers, with nothing that follows the sum as an operation of its own, goes along in the launch
        const at::Device device = x.device();
        const bool fused_bias = pays && bias.defined() && bias.dim() == 1 && bias.size(0) == w.N && plain_execution() && plain_half(m.bias, &device);
        Tensor out;
        int rc, added = 0;
        {
            const WithoutGil free;
            const OnDevice on(w.device);
            if (pays) {
                const Tensor dense = x.is_contiguous() ? x : x.contiguous();  // the kernels take dense rows
                out = result_for(x, w.N);
                rc = ap_linear(half_ptr(dense), w.planes, w.lut, fused_bias ? half_ptr(bias) : nullptr, half_out(out), (int)rows, w.N, w.K, bits,
                               on.stream, &added);
            } else {
                op = "dequant_kbit";
                const Tensor dense = empty_half({w.N, w.K}, x.device());
                // The product finds a weight of up to 192 MB (and its activations) in the last-level cache of 256: us past the caches / through
                // them 4096 x 11008 at 512 rows 102 / 88, at 2048 196 / 181, 4096 x 4096 at 1024 rows 56 / 53, 14336 x 4096 127 / 123 (8 bits);
                // a larger one is written out before it is read: 28672 x 8192 at 512 rows 301 / 317, 32000 x 4096 159 / 170.
                const auto dequant = (int64_t)w.N * w.K <= 96 << 20 ? ap_dequant_kbit_near : ap_dequant_kbit;
                rc = dequant(w.planes, w.lut, half_out(dense), w.N, w.K, bits, on.stream);
                if (rc == AP_OK) out = at::matmul(x, dense.t());
            }
            if (rc == AP_OK && bias.defined() && !added) out.add_(bias);
        }
        if (rc != AP_OK) return library_error(rc, op);
        return wrap(std::move(out));
    });
}

// linear_group(__dict__ of 2..4 modules, x, w_bits, concat as a bool): forward_group for bias-free linears of one input length.  A list of
// results, or with concat one tensor of them side by side (a list yet where a torch-function mode is to see torch.cat).  ap_linear_group where ap_linear_staged or, beyond 8 rows, where
// ap_gemm_kbit_group_pays or _taken; up to 8 rows ap_matmul_kbit_group else; None where the modules are better called one by one.
PyObject *linear_group(PyObject *, PyObject *const *args, Py_ssize_t n) {
    constexpr int MOST = 4;
    if (n != 4 || !PyTuple_Check(args[0]) || !is_tensor(args[1])) return none();
    const int bits = bits_of(args[2]), count = (int)PyTuple_GET_SIZE(args[0]);
    const bool concat = args[3] == Py_True;
    if (bits == 0 || count < 2 || count > MOST) return none();
    ModuleTensors m[MOST];
    for (int g = 0; g < count; g++)
        if (!tensors_of(PyTuple_GET_ITEM(args[0], g), bits, &m[g]) || m[g].bias != nullptr) return none();
    return guarded([&]() -> PyObject * {
        const Tensor &given = THPVariable_Unpack(args[1]);
        Tensor q[MOST], t[MOST];
        Weight w[MOST];
        int N[MOST];
        int64_t total = 0;
        const uint32_t *planes[MOST];
        const uint16_t *luts[MOST];
        for (int g = 0; g < count; g++) {
            q[g] = THPVariable_Unpack(m[g].qweight);
            t[g] = THPVariable_Unpack(m[g].table);
            if (!weight_of(q[g], t[g], bits, &w[g])) return none();
            if (w[g].K != w[0].K || w[g].device != w[0].device) return none();
            N[g] = w[g].N;
            total += N[g];
            planes[g] = w[g].planes;
            luts[g] = w[g].lut;
        }
        const int64_t rows = rows_of(given, w[0]);
        const int K = w[0].K;
        if (rows < 1) return none();
        const bool staged = ap_linear_staged(count, N, (int)rows, K, bits) == 1, gemm = rows > 8 || staged;
        if (rows > 8 && ap_gemm_kbit_group_pays(count, N, (int)rows, K, bits) != 1 &&
            !((staged || ap_gemm_kbit_group_taken(count, N, (int)rows, K, bits) == 1) && plain_execution() && product_is_half() && plain_half(args[1], nullptr)))
            return none();
        // side by side in one allocation: one row's results always are dense, and the tiled, block-tile and staged kernels write rows that are
        // not.  At 2..8 rows torch joins them wherever something else than plain execution may look at that; for a torch-function mode the
        // caller does.
        const bool joint = concat && (rows > 8 ? K % 128 == 0 : rows == 1 || (staged && plain_execution()));
        const bool join = concat && !joint && !at::impl::torch_function_mode_enabled();
        Tensor all, outs[MOST];
        int rc;
        {
            const WithoutGil free;
            const OnDevice on(w[0].device);
            const Tensor x = given.is_contiguous() ? given : given.contiguous();
            uint16_t *to[MOST];
            long long ldo[MOST];
            if (joint) {
                all = result_for(x, total);
                int64_t at = 0;
                for (int g = 0; g < count; at += N[g], g++) {
                    to[g] = half_out(all) + at;
                    ldo[g] = total;
                }
            } else {
                for (int g = 0; g < count; g++) {
                    outs[g] = result_for(x, N[g]);
                    to[g] = half_out(outs[g]);
                }
            }
            rc = gemm ? ap_linear_group(half_ptr(x), count, planes, luts, to, N, joint ? ldo : nullptr, (int)rows, K, bits, on.stream)
                      : ap_matmul_kbit_group(half_ptr(x), count, planes, luts, to, N, (int)rows, K, bits, on.stream);
            if (rc == AP_OK && join) all = at::cat(std::vector<Tensor>(outs, outs + count), -1);
        }
        if (rc == AP_ELIMIT) return none();  // beyond the tiled kernel's offsets
        if (rc != AP_OK) return library_error(rc, gemm ? "gemm_kbit_group" : "matmul_kbit_group");
        if (joint || join) return wrap(std::move(all));
        PyObject *list = PyList_New(count);
        if (list == nullptr) return nullptr;
        for (int g = 0; g < count; g++) {
            PyObject *o = wrap(std::move(outs[g]));
            if (o == nullptr) {
                Py_DECREF(list);
                return nullptr;
            }
            PyList_SET_ITEM(list, g, o);
        }
        return list;
    });
}

// plain(tensors): whether the functions below take each of them, all on one device.
PyObject *plain(PyObject *, PyObject *const *args, Py_ssize_t n) {
    return guarded([&]() -> PyObject * {
        bool all = n > 0 && plain_execution() && plain_half(args[0], nullptr);
        for (Py_ssize_t i = 1; all && i < n; i++) {
            const at::Device device = THPVariable_Unpack(args[0]).device();
            all = plain_half(args[i], &device);
        }
        return PyBool_FromLong(all);
    });
}

// rmsnorm(x, weight, eps): x * rsqrt(mean(x^2) + eps) * weight over the last dimension.
PyObject *rmsnorm(PyObject *, PyObject *const *args, Py_ssize_t n) {
    if (n != 3 || !PyFloat_Check(args[2]) || !plain_execution()) return none();
    return guarded([&]() -> PyObject * {
        if (!plain_half(args[0], nullptr)) return none();
        const Tensor &x = THPVariable_Unpack(args[0]);
        const at::Device device = x.device();
        if (!plain_half(args[1], &device)) return none();
        const Tensor &weight = THPVariable_Unpack(args[1]);
        const float eps = (float)PyFloat_AS_DOUBLE(args[2]);
        const int64_t H = x.dim() < 1 ? 0 : x.size(-1);
        if (weight.dim() != 1 || weight.size(0) != H || H < 8 || H % 8 || H > INT32_MAX || x.numel() / H > INT32_MAX) return none();
        Tensor out;
        int rc;
        {
            const WithoutGil free;
            const OnDevice on(device.index());
            out = empty_half(x.sizes(), device);
            // nothing is added, so h_out = h is not written
            rc = ap_add_rmsnorm(half_ptr(x), nullptr, half_ptr(weight), half_out(x), half_out(out), (int)(x.numel() / H), (int)H, eps,
                                on.stream);
        }
        if (rc != AP_OK) return library_error(rc, "rmsnorm");
        return wrap(std::move(out));
    });
}

// silu_mul(gate, up): silu(gate) * up.
PyObject *silu_mul(PyObject *, PyObject *const *args, Py_ssize_t n) {
    if (n != 2 || !plain_execution()) return none();
    return guarded([&]() -> PyObject * {
        if (!plain_half(args[0], nullptr)) return none();
        const Tensor &gate = THPVariable_Unpack(args[0]);
        const at::Device device = gate.device();
        if (!plain_half(args[1], &device)) return none();
        const Tensor &up = THPVariable_Unpack(args[1]);
        if (gate.sizes() != up.sizes() || gate.numel() % 8) return none();
        Tensor out;
        int rc;
        {
            const WithoutGil free;
            const OnDevice on(device.index());
            out = empty_half(gate.sizes(), device);
            rc = ap_silu_mul(half_ptr(gate), half_ptr(up), half_out(out), gate.numel(), on.stream);
        }
        if (rc != AP_OK) return library_error(rc, "silu_mul");
        return wrap(std::move(out));
    });
}

// rope(x [B, T, heads * hd], cos, sin [B or 1, T, hd]): [B, T, heads, hd].
PyObject *rope(PyObject *, PyObject *const *args, Py_ssize_t n) {
    if (n != 3 || !plain_execution()) return none();
    return guarded([&]() -> PyObject * {
        if (!plain_half(args[0], nullptr)) return none();
        const Tensor &x = THPVariable_Unpack(args[0]);
        const at::Device device = x.device();
        if (!plain_half(args[1], &device) || !plain_half(args[2], &device)) return none();
        const Tensor &c = THPVariable_Unpack(args[1]), &s = THPVariable_Unpack(args[2]);
        if (x.dim() != 3 || c.dim() != 3 || c.sizes() != s.sizes()) return none();
        const int64_t B = x.size(0), T = x.size(1), hd = c.size(2);
        if (c.size(1) != T || (c.size(0) != B && c.size(0) != 1) || hd % 16 || x.size(2) % hd || x.numel() / 16 > INT32_MAX) return none();
        Tensor out;
        int rc;
        {
            const WithoutGil free;
            const OnDevice on(device.index());
            out = empty_half({B, T, x.size(2) / hd, hd}, device);
            rc = ap_rope_heads(half_ptr(x), half_ptr(c), half_ptr(s), half_out(out), (int)(B * T), (int)(c.size(0) * T),
                               (int)(x.size(2) / hd), (int)hd, on.stream);
        }
        if (rc != AP_OK) return library_error(rc, "rope");
        return wrap(std::move(out));
    });
}

PyMethodDef methods[] = {
    {"matmul_kbit", reinterpret_cast<PyCFunction>(reinterpret_cast<void *>(matmul_kbit)), METH_FASTCALL, nullptr},
    {"gemm_kbit", reinterpret_cast<PyCFunction>(reinterpret_cast<void *>(gemm_kbit)), METH_FASTCALL, nullptr},
    {"dequant_kbit", reinterpret_cast<PyCFunction>(reinterpret_cast<void *>(dequant_kbit)), METH_FASTCALL, nullptr},
    {"linear", reinterpret_cast<PyCFunction>(reinterpret_cast<void *>(linear)), METH_FASTCALL, nullptr},
    {"linear_group", reinterpret_cast<PyCFunction>(reinterpret_cast<void *>(linear_group)), METH_FASTCALL, nullptr},
    {"plain", reinterpret_cast<PyCFunction>(reinterpret_cast<void *>(plain)), METH_FASTCALL, nullptr},
    {"rmsnorm", reinterpret_cast<PyCFunction>(reinterpret_cast<void *>(rmsnorm)), METH_FASTCALL, nullptr},
    {"silu_mul", reinterpret_cast<PyCFunction>(reinterpret_cast<void *>(silu_mul)), METH_FASTCALL, nullptr},
    {"rope", reinterpret_cast<PyCFunction>(reinterpret_cast<void *>(rope)), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_anyprec_torch", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__anyprec_torch(void) {
    key_buffers = PyUnicode_InternFromString("_buffers");
    key_qweight = PyUnicode_InternFromString("qweight");
    key_bias = PyUnicode_InternFromString("bias");
    for (int b = 3; b <= 8; b++) key_lut[b] = PyUnicode_InternFromString(("lut" + std::to_string(b)).c_str());
    PyObject *m = PyModule_Create(&module);
    if (m != nullptr && (PyModule_AddIntConstant(m, "abi_version", AP_ABI_VERSION) != 0 ||
                         PyModule_AddStringConstant(m, "torch_version", AP_TORCH_VERSION) != 0)) {
        Py_DECREF(m);
        return nullptr;
    }
    return m;
}
