// Python entry points of the library on torch tensors, as a native module (host code only, no kernels).
//
// A call of a small GEMM is a few microseconds of GPU time. The same checks and the same C call written in Python over
// ctypes took 9 to 14 us of host time (operand checks 5 us, stream and device objects 3 us, argument conversion 3 us),
// which is what a loop of such calls then ran at: a single-token GEMM (M = 1, N = 7168, K = 2048) took 13.4 us a call
// however fast its kernels were. Here the tensors are read through torch's C++ API.
//
// The functions check the operands exactly as gemm.py documents them (ValueError), launch on the current stream of the
// operands' device through the C ABI of libgemm.so, and raise RuntimeError with the library's message if that fails.
#include <torch/csrc/autograd/python_variable.h>
#include <ATen/ATen.h>
#include <ATen/hip/EmptyTensor.h>
#include <ATen/record_function.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>

#include <string>
#include <vector>

#include "../../include/rf_gemm.h"

namespace {

struct PyError {};                       // a Python exception has been set

[[noreturn]] void raise(PyObject *type, const std::string &msg) {
    PyErr_SetString(type, msg.c_str());
    throw PyError();
}

const at::Tensor &tensor(PyObject *o) {
    if (!THPVariable_Check(o)) raise(PyExc_TypeError, std::string("expected a torch.Tensor, got ") + Py_TYPE(o)->tp_name);
    return THPVariable_Unpack(o);
}

// Makes a tensor's device current for the call, and gives its current stream. Nearly every call finds it current
// already: then nothing is set and nothing restored.
struct OnDeviceOf {
    int before, dev;
    hipStream_t stream;
    explicit OnDeviceOf(const at::Tensor &t) : before(c10::hip::current_device()), dev(t.device().index()) {
        if (dev != before) c10::hip::set_device(dev);
        stream = c10::hip::getCurrentHIPStream(dev).stream();
    }
    ~OnDeviceOf() {
        if (dev != before) (void)hipSetDevice(before);
    }
};

template <typename F>
void call(const char *name, const F &f) {
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = f();
    Py_END_ALLOW_THREADS
    if (rc != RF_OK)
        raise(PyExc_RuntimeError, std::string(name) + " failed (" + std::to_string(rc) + "): " + rf_gemm_last_error());
}

// Every function: COUNT arguments by position, C++ exceptions turned into Python ones.
template <PyObject *(*F)(PyObject *const *), int COUNT>
PyObject *entry(PyObject *, PyObject *const *args, Py_ssize_t count) {
    if (count != COUNT) {
        PyErr_Format(PyExc_TypeError, "expected %d arguments, got %zd", COUNT, count);
        return nullptr;
    }
    try {
        return F(args);
    } catch (const PyError &) {
    } catch (const std::exception &e) {
        PyErr_SetString(PyExc_RuntimeError, e.what());
    }
    return nullptr;
}

bool shape_is(const at::Tensor &t, int64_t x, int64_t y) { return t.dim() == 2 && t.size(0) == x && t.size(1) == y; }
// storage [cols][rows]: the tensor is the transposed view the launcher's layout is
bool column_major(const at::Tensor &t) {
    const int64_t r = t.size(0), c = t.size(1);
    return (t.stride(0) == 1 || r == 1) && (t.stride(1) == r || c == 1);
}

struct Shape {
    int m, n, k;
};
Shape check_operands(const at::Tensor &a, const at::Tensor &b, const at::Tensor &as, const at::Tensor &bs, const at::Tensor &c) {
    if (!(a.is_cuda() && b.is_cuda() && as.is_cuda() && bs.is_cuda() && c.is_cuda()))
        raise(PyExc_ValueError, "fp8_mm needs GPU tensors");
    if (a.dim() != 2 || b.dim() < 2) raise(PyExc_ValueError, "a and b must be matrices");
    const int64_t m = a.size(0), k = a.size(1), n = b.size(0), qk = k / 128, qn = (n + 127) / 128;
    if (a.element_size() != 1 || b.element_size() != 1)
        raise(PyExc_ValueError, "a and b must be 1-byte fp8 (e4m3fn) tensors");
    if (!shape_is(b, n, k) || !shape_is(as, m, qk) || !shape_is(bs, qn, qk) || !shape_is(c, m, n))
        raise(PyExc_ValueError, "inconsistent shapes");
    if (as.scalar_type() != at::kFloat || bs.scalar_type() != at::kFloat || c.scalar_type() != at::kBFloat16)
        raise(PyExc_ValueError, "scales must be fp32 and c bf16");
    if (!(column_major(a) && column_major(b) && column_major(as) && column_major(bs) && c.is_contiguous()))
        raise(PyExc_ValueError, "a, b, a_scale, b_scale must be column-major (transposed views), c row-major contiguous");
    return {(int)m, (int)n, (int)k};
}

// check_operands(a, b, a_scale, b_scale, c) -> (m, n, k)
PyObject *py_check_operands(PyObject *const *v) {
    const Shape s = check_operands(tensor(v[0]), tensor(v[1]), tensor(v[2]), tensor(v[3]), tensor(v[4]));
    return Py_BuildValue("iii", s.m, s.n, s.k);
}

// fp8_mm(a, b, a_scale, b_scale, c, address of a rf_gemm_config or 0)
PyObject *py_fp8_mm(PyObject *const *v) {
    const at::Tensor &a = tensor(v[0]), &b = tensor(v[1]), &as = tensor(v[2]), &bs = tensor(v[3]), &c = tensor(v[4]);
    const Shape s = check_operands(a, b, as, bs, c);
    const rf_gemm_config *cfg = (const rf_gemm_config *)PyLong_AsVoidPtr(v[5]);
    if (PyErr_Occurred()) throw PyError();
    OnDeviceOf dev(a);
    const void *pa = a.const_data_ptr(), *pb = b.const_data_ptr();
    const float *pas = (const float *)as.const_data_ptr(), *pbs = (const float *)bs.const_data_ptr();
    void *pc = c.mutable_data_ptr();
    call("rf_fp8_gemm", [&] { return rf_fp8_gemm_ex(pa, pb, pas, pbs, pc, s.m, s.n, s.k, cfg, dev.stream); });
    Py_RETURN_NONE;
}

// fp8_mm_static(a, b, a_scale, b_scale, c)
PyObject *py_fp8_mm_static(PyObject *const *v) {
    const at::Tensor &a = tensor(v[0]), &b = tensor(v[1]), &as = tensor(v[2]), &bs = tensor(v[3]), &c = tensor(v[4]);
    const Shape s = check_operands(a, b, as, bs, c);
    OnDeviceOf dev(a);
    const void *pa = a.const_data_ptr(), *pb = b.const_data_ptr();
    const float *pas = (const float *)as.const_data_ptr(), *pbs = (const float *)bs.const_data_ptr();
    void *pc = c.mutable_data_ptr();
    call("rf_fp8_gemm_static", [&] { return rf_fp8_gemm_static(pa, pb, pas, pbs, pc, s.m, s.n, s.k, dev.stream); });
    Py_RETURN_NONE;
}

// A sequence of ints (or of things int() takes) as the C ABI's row offsets; ValueError for one that 32 bits do not hold.
std::vector<int> offsets_of(PyObject *o) {
    PyObject *seq = PySequence_Fast(o, "row_offsets must be a sequence");
    if (!seq) throw PyError();
    const Py_ssize_t n = PySequence_Fast_GET_SIZE(seq);
    std::vector<int> out((size_t)n);
    for (Py_ssize_t i = 0; i < n; i++) {
        PyObject *x = PySequence_Fast_GET_ITEM(seq, i);
        PyObject *num = PyLong_Check(x) ? (Py_INCREF(x), x) : PyNumber_Long(x);
        if (num) {
            int overflow = 0;
            const long long value = PyLong_AsLongLongAndOverflow(num, &overflow);
            Py_DECREF(num);
            out[(size_t)i] = (int)value;
            if (!PyErr_Occurred() && (overflow || value != out[(size_t)i]))
                PyErr_SetString(PyExc_ValueError, "row_offsets must fit 32 bits");
        }
        if (PyErr_Occurred()) {
            Py_DECREF(seq);
            throw PyError();
        }
    }
    Py_DECREF(seq);
    return out;
}

// b [G, N, K] stride (K*N, 1, N) and b_scale [G, QN, QK] stride (QK*QN, 1, QN)
bool grouped_weights_ok(const at::Tensor &b, const at::Tensor &bs, int64_t k) {
    const int64_t groups = b.size(0), n = b.size(1), qk = k / 128, qn = (n + 127) / 128;
    return b.scalar_type() == at::kFloat8_e4m3fn && bs.scalar_type() == at::kFloat && b.size(2) == k &&
           (b.stride(0) == k * n || groups == 1) && b.stride(1) == 1 && b.stride(2) == n && bs.dim() == 3 &&
           bs.size(0) == groups && bs.size(1) == qn && bs.size(2) == qk &&
           (((bs.stride(0) == qk * qn || groups == 1) && bs.stride(1) == 1 && bs.stride(2) == qn) || qn == 1 || qk == 1);
}

// fp8_mm_grouped(a, b, a_scale, b_scale, c, row_offsets, variant)
PyObject *py_fp8_mm_grouped(PyObject *const *v) {
    const at::Tensor &a = tensor(v[0]), &b = tensor(v[1]), &as = tensor(v[2]), &bs = tensor(v[3]), &c = tensor(v[4]);
    const std::vector<int> offs = offsets_of(v[5]);
    const int variant = (int)PyLong_AsLong(v[6]);
    if (PyErr_Occurred()) throw PyError();
    if (a.dim() != 2 || b.dim() != 3) raise(PyExc_ValueError, "a must be a matrix and b a batch of matrices");
    const int64_t m = a.size(0), k = a.size(1), groups = b.size(0), n = b.size(1), qk = k / 128;
    const bool ok = a.scalar_type() == at::kFloat8_e4m3fn && c.scalar_type() == at::kBFloat16 && as.scalar_type() == at::kFloat &&
                    grouped_weights_ok(b, bs, k) && shape_is(c, m, n) && c.is_contiguous() &&
                    (m <= 1 || k == 1 || (a.stride(0) == 1 && a.stride(1) == m)) && shape_is(as, m, qk) &&
                    (m <= 1 || qk == 1 || (as.stride(0) == 1 && as.stride(1) == m)) && (int64_t)offs.size() == groups + 1;
    if (!ok) raise(PyExc_ValueError, "fp8_mm_grouped: operands do not have the documented dtypes / shapes / strides");
    if (!a.is_cuda()) raise(PyExc_ValueError, "fp8_mm_grouped needs GPU tensors");
    OnDeviceOf dev(a);
    const void *pa = a.const_data_ptr(), *pb = b.const_data_ptr();
    const float *pas = (const float *)as.const_data_ptr(), *pbs = (const float *)bs.const_data_ptr();
    void *pc = c.mutable_data_ptr();
    call("rf_fp8_gemm_grouped", [&] {
        return rf_fp8_gemm_grouped(pa, pb, pas, pbs, pc, offs.data(), (int)groups, (int)n, (int)k, variant, dev.stream);
    });
    Py_RETURN_NONE;
}

// Row count of the padded layout; RuntimeError if the offsets are refused.
int padded_rows(const std::vector<int> &offs) {
    std::vector<int> padded(offs.size() + 1);
    call("rf_grouped_padded_offsets", [&] { return rf_grouped_padded_offsets(offs.data(), (int)offs.size() - 1, padded.data()); });
    return padded[offs.size() - 1];
}

// fp8_mm_grouped_padded(a, b, a_scale, b_scale, c, row_offsets, variant)
PyObject *py_fp8_mm_grouped_padded(PyObject *const *v) {
    const at::Tensor &a = tensor(v[0]), &b = tensor(v[1]), &as = tensor(v[2]), &bs = tensor(v[3]), &c = tensor(v[4]);
    const std::vector<int> offs = offsets_of(v[5]);
    const int variant = (int)PyLong_AsLong(v[6]);
    if (PyErr_Occurred()) throw PyError();
    if (a.dim() != 2 || b.dim() != 3 || offs.empty()) raise(PyExc_ValueError, "a must be a matrix and b a batch of matrices");
    const int64_t m_pad = a.size(0), k = a.size(1), groups = b.size(0), n = b.size(1), qk = k / 128;
    const bool ok = a.scalar_type() == at::kFloat8_e4m3fn && c.scalar_type() == at::kBFloat16 && as.scalar_type() == at::kFloat &&
                    (int64_t)offs.size() == groups + 1 && m_pad == padded_rows(offs) && a.stride(0) == 1 && a.stride(1) == m_pad &&
                    shape_is(as, m_pad, qk) && (qk == 1 || (as.stride(0) == 1 && as.stride(1) == m_pad)) &&
                    grouped_weights_ok(b, bs, k) && shape_is(c, offs.back(), n) && c.is_contiguous();
    if (!ok) raise(PyExc_ValueError, "fp8_mm_grouped_padded: operands do not have the documented dtypes / shapes / strides");
    if (!a.is_cuda()) raise(PyExc_ValueError, "fp8_mm_grouped_padded needs GPU tensors");
    OnDeviceOf dev(a);
    const void *pa = a.const_data_ptr(), *pb = b.const_data_ptr();
    const float *pas = (const float *)as.const_data_ptr(), *pbs = (const float *)bs.const_data_ptr();
    void *pc = c.mutable_data_ptr();
    call("rf_fp8_gemm_grouped_padded", [&] {
        return rf_fp8_gemm_grouped_padded(pa, pb, pas, pbs, pc, offs.data(), (int)groups, (int)n, (int)k, variant, dev.stream);
    });
    Py_RETURN_NONE;
}

void check_source(const at::Tensor &x) {
    if (x.dim() != 2 || !x.is_contiguous() || (x.scalar_type() != at::kFloat && x.scalar_type() != at::kBFloat16))
        raise(PyExc_ValueError, "source must be a contiguous 2-D fp32 or bf16 tensor [rows, K]");
}

// A [rows, cols] tensor over [cols][rows] storage: the transposed view that fp8_mm takes.
at::Tensor empty_column_major(const at::Tensor &like, int64_t rows, int64_t cols, at::ScalarType type) {
    const int64_t size[2] = {rows, cols}, stride[2] = {1, rows};
    // Straight to the allocation where nothing listens on the way: no dispatch mode, functorch level, autocast, inference mode
    // or profiler of this thread. Through the dispatcher a tensor costs 0.28 us more (quantize_a on 7 x 1536: 4.4 -> 4.95 us).
    const c10::impl::LocalDispatchKeySet keys = c10::impl::tls_local_dispatch_key_set();
    if (keys.included_ == c10::default_included_set && keys.excluded_ == c10::default_excluded_set && !at::hasCallbacks())
        return at::detail::empty_strided_cuda(size, stride, type, like.device());
    return at::empty_strided(size, stride, at::TensorOptions().dtype(type).device(like.device()));
}

PyObject *pair_of(const at::Tensor &x, const at::Tensor &y) {
    PyObject *px = THPVariable_Wrap(x), *py = px ? THPVariable_Wrap(y) : nullptr;
    PyObject *out = py ? PyTuple_New(2) : nullptr;
    if (!out) {
        Py_XDECREF(px);
        Py_XDECREF(py);
        throw PyError();
    }
    PyTuple_SET_ITEM(out, 0, px);
    PyTuple_SET_ITEM(out, 1, py);
    return out;
}

// quantize(x, per_row) -> (q [rows, K], scales [rows or ceil(rows/128), K/128])
PyObject *py_quantize(PyObject *const *v) {
    const at::Tensor &x = tensor(v[0]);
    const bool per_row = v[1] == Py_True, f32 = x.scalar_type() == at::kFloat;
    check_source(x);
    const int64_t rows = x.size(0), k = x.size(1);
    if (k < 128 || k % 128) raise(PyExc_ValueError, "K must be a positive multiple of 128");
    if (!x.is_cuda()) raise(PyExc_ValueError, "source must be on the GPU");
    OnDeviceOf dev(x);
    const at::Tensor q = empty_column_major(x, rows, k, at::kFloat8_e4m3fn);
    const at::Tensor s = empty_column_major(x, per_row ? rows : (rows + 127) / 128, k / 128, at::kFloat);
    const void *px = x.const_data_ptr();
    void *pq = q.mutable_data_ptr();
    float *ps = (float *)s.mutable_data_ptr();
    call(per_row ? f32 ? "rf_quantize_a_f32" : "rf_quantize_a_bf16" : f32 ? "rf_quantize_b_f32" : "rf_quantize_b_bf16", [&] {
        return per_row ? f32 ? rf_quantize_a_f32((const float *)px, (int)rows, (int)k, pq, ps, dev.stream)
                             : rf_quantize_a_bf16(px, (int)rows, (int)k, pq, ps, dev.stream)
               : f32   ? rf_quantize_b_f32((const float *)px, (int)rows, (int)k, pq, ps, dev.stream)
                       : rf_quantize_b_bf16(px, (int)rows, (int)k, pq, ps, dev.stream);
    });
    return pair_of(q, s);
}

// quantize_a_grouped(x, row_offsets) -> (a [M_pad, K], a_scale [M_pad, K/128]) in the padded layout
PyObject *py_quantize_a_grouped(PyObject *const *v) {
    const at::Tensor &x = tensor(v[0]);
    check_source(x);
    const std::vector<int> offs = offsets_of(v[1]);
    const int64_t rows = x.size(0), k = x.size(1);
    if (k < 128 || k % 128 || offs.empty() || offs.back() != rows)
        raise(PyExc_ValueError, "K must be a positive multiple of 128 and row_offsets must end at the number of rows");
    if (!x.is_cuda()) raise(PyExc_ValueError, "source must be on the GPU");
    const int m_pad = padded_rows(offs), groups = (int)offs.size() - 1;
    const bool f32 = x.scalar_type() == at::kFloat;
    OnDeviceOf dev(x);
    const at::Tensor a = empty_column_major(x, m_pad, k, at::kFloat8_e4m3fn);
    const at::Tensor s = empty_column_major(x, m_pad, k / 128, at::kFloat);
    const void *px = x.const_data_ptr();
    void *pa = a.mutable_data_ptr();
    float *ps = (float *)s.mutable_data_ptr();
    call(f32 ? "rf_quantize_a_grouped_f32" : "rf_quantize_a_grouped_bf16", [&] {
        return f32 ? rf_quantize_a_grouped_f32((const float *)px, offs.data(), groups, (int)k, pa, ps, dev.stream)
                   : rf_quantize_a_grouped_bf16(px, offs.data(), groups, (int)k, pa, ps, dev.stream);
    });
    return pair_of(a, s);
}

#define RF_ENTRY(name, f, count) {name, (PyCFunction)(void (*)(void))entry<f, count>, METH_FASTCALL, nullptr}
PyMethodDef methods[] = {RF_ENTRY("check_operands", py_check_operands, 5),
                         RF_ENTRY("fp8_mm", py_fp8_mm, 6),
                         RF_ENTRY("fp8_mm_static", py_fp8_mm_static, 5),
                         RF_ENTRY("fp8_mm_grouped", py_fp8_mm_grouped, 7),
                         RF_ENTRY("fp8_mm_grouped_padded", py_fp8_mm_grouped_padded, 7),
                         RF_ENTRY("quantize", py_quantize, 2),
                         RF_ENTRY("quantize_a_grouped", py_quantize_a_grouped, 2),
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_torch_binding", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__torch_binding(void) { return PyModule_Create(&module); }
