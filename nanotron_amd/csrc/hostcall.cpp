// Host side of the hot calls: output allocation, descriptors and the C-ABI call in one step.
//
// A small layer's training step is bound by the host, not by the GPU (128 x 128 x 128: 39 us of kernels in a step of
// 340 us), and most of that is Python: every attribute of an FP8Tensor passes through __torch_function__ (1.1 us, the
// shape 2.4 us), every allocation and every view is a Python call, a descriptor is filled field by field.  The
// functions below take tensors as they are (subclasses unwrapped without dispatch), allocate below autograd, and call
// libntfp8.so's C entry points.  They are thin: no arithmetic and no kernel lives here.
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/core/LegacyTypeDispatch.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <optional>
#include <unordered_map>

#include "../../include/ntfp8.h"

namespace {

PyObject* g_check = nullptr;   // nanotron_amd._native.check: raises RuntimeError, has the workspaces dropped after a failed launch

PyObject* g_observer = nullptr;   // of the GEMM calls, see set_gemm_observer

struct Stop {};   // a Python error is set

[[noreturn]] void stop(PyObject* type, const char* msg) {
    PyErr_SetString(type, msg);
    throw Stop{};
}
void require(bool ok, const char* msg) {
    if (!ok) stop(PyExc_AssertionError, msg);
}

// Reduction workspaces, zero between launches: one for calls of one tensor and a pool for batched calls, per (device,
// stream).  The package's other callers take theirs from here too (workspace() below).  Guarded by the GIL; the table is
// never destroyed (its tensors must not outlive the runtime's teardown).
using Key = std::pair<int, void*>;
struct KeyHash {
    size_t operator()(const Key& k) const { return reinterpret_cast<size_t>(k.second) * 31u + (size_t)k.first; }
};
struct Space {
    at::Tensor one, many;
};
using Spaces = std::unordered_map<Key, Space, KeyHash>;
Spaces& workspaces() {
    static auto* m = new Spaces();
    return *m;
}
// Those of a stream that records a graph: made in the capture that uses them (the fill is a node of its graph, the memory
// comes from its pool) and never seen by another capture or by eager calls, of which the graph's replays know nothing.
// Only the table lets go of them afterwards, at the next eager call.
struct CapturedSpace {
    unsigned long long capture;
    Space space;
};
std::unordered_map<Key, CapturedSpace, KeyHash>& captured_workspaces() {
    static auto* m = new std::unordered_map<Key, CapturedSpace, KeyHash>();
    return *m;
}

void call(int rc, const char* what) {
    if (rc == NTFP8_OK) return;
    PyObject* r = PyObject_CallFunction(g_check, "is", rc, what);
    Py_XDECREF(r);
    if (r != nullptr) stop(PyExc_RuntimeError, what);
    throw Stop{};
}

const at::Tensor& tensor(PyObject* o) {
    if (!THPVariable_Check(o)) stop(PyExc_TypeError, "a tensor is expected");
    return THPVariable_Unpack(o);
}
bool none(PyObject* o) { return o == Py_None || o == nullptr; }
long number(PyObject* o) {
    const long v = PyLong_AsLong(o);
    if (v == -1 && PyErr_Occurred()) throw Stop{};
    return v;
}
bool truth(PyObject* o) {
    if (o == Py_True) return true;
    if (o == Py_False || o == Py_None) return false;
    const int v = PyObject_IsTrue(o);
    if (v < 0) throw Stop{};
    return v != 0;
}
PyObject* wrap(at::Tensor t) {
    PyObject* o = THPVariable_Wrap(std::move(t));
    if (o == nullptr) throw Stop{};
    return o;
}
PyObject* wrap_or_none(at::Tensor t) {
    if (t.defined()) return wrap(std::move(t));
    Py_RETURN_NONE;
}

void* stream_of(const at::Tensor& t) {
    return static_cast<void*>(c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(t.get_device()).stream());
}
Space& space_of(int device, void* stream) {
    const Key key{device, stream};
    if (stream != nullptr) {   // (the legacy stream cannot be captured, and must not be asked while another one is)
        hipStreamCaptureStatus status;
        unsigned long long id = 0;
        if (hipStreamGetCaptureInfo(static_cast<hipStream_t>(stream), &status, &id) != hipSuccess) stop(PyExc_RuntimeError, "hipStreamGetCaptureInfo failed");
        if (status == hipStreamCaptureStatusActive) {
            CapturedSpace& c = captured_workspaces()[key];
            if (c.capture != id) c = CapturedSpace{id, Space{}};
            return c.space;
        }
    }
    if (!captured_workspaces().empty()) captured_workspaces().clear();
    return workspaces()[key];
}
at::Tensor zeroed(int device, int64_t count) {
    return at::zeros({count, NTFP8_WORKSPACE_BYTES / 4}, at::TensorOptions().dtype(at::kInt).device(at::kCUDA, (c10::DeviceIndex)device));
}
const at::Tensor& workspace_at(int device, void* stream) {
    at::Tensor& w = space_of(device, stream).one;
    if (!w.defined()) w = zeroed(device, 1).squeeze(0);
    return w;
}
// [>= count] workspaces for the tensors of a batched call
const at::Tensor& pool_at(int device, void* stream, int64_t count) {
    at::Tensor& w = space_of(device, stream).many;
    if (!w.defined() || w.size(0) < count) w = zeroed(device, count < 16 ? 16 : count);
    return w;
}
void* workspace_of(const at::Tensor& t, void* stream) { return workspace_at((int)t.get_device(), stream).data_ptr(); }

int code_of(at::ScalarType t) {   // NTFP8_F32 / F16 / BF16, or -1
    return t == at::kFloat ? NTFP8_F32 : t == at::kHalf ? NTFP8_F16 : t == at::kBFloat16 ? NTFP8_BF16 : -1;
}
at::ScalarType type_of(long code) {
    return code == NTFP8_F32 ? at::kFloat : code == NTFP8_F16 ? at::kHalf : code == NTFP8_BF16 ? at::kBFloat16 : at::kByte;
}
at::Tensor bytes_like(const at::Tensor& x, at::IntArrayRef sizes) {
    return at::empty(sizes, at::TensorOptions().dtype(at::kByte).device(x.device()));
}
at::Tensor dense(const at::Tensor& t) { return t.is_contiguous() ? t : t.contiguous(); }
// the same of an operand that a kernel is about to read: an address of host memory would fault the GPU
at::Tensor operand(PyObject* o) {
    const at::Tensor& t = tensor(o);
    require(t.is_cuda(), "a tensor on a CUDA device is expected");
    return dense(t);
}

// fp32 values in device memory that a kernel will read or write: a scale, a flag, a delayed-scaling state.  An address of host
// memory would fault the GPU here as well, and another type would be read as something else.
float* values(PyObject* o, c10::Device device, int64_t count = 1) {
    const at::Tensor& t = tensor(o);
    require(t.is_cuda() && t.device() == device, "scales and delayed-scaling states must be on the device of the operand");
    require(t.scalar_type() == at::kFloat && t.numel() >= count && (count == 1 || t.is_contiguous()),
            "scales and delayed-scaling states are fp32 tensors of one value, or of a scale and its history");
    return static_cast<float*>(t.data_ptr());
}
// fp8 codes: one byte each
const at::Tensor& codes(const at::Tensor& t) {
    require(t.element_size() == 1, "fp8 codes take one byte each");
    return t;
}

// [amax, scale used] of a quantisation: one allocation, and its two elements as 0-dim tensors
struct Scalars {
    at::Tensor both;
    float* p;
    explicit Scalars(const at::Tensor& like)
        : both(at::empty({2}, at::TensorOptions().dtype(at::kFloat).device(like.device()))), p(static_cast<float*>(both.data_ptr())) {}
    Scalars(at::Tensor inside, float* at) : both(std::move(inside)), p(at) {}   // two values inside an allocation of something else
    at::Tensor element(int64_t i) const {
        at::Tensor v = at::detail::make_tensor<c10::TensorImpl>(c10::TensorImpl::VIEW, c10::Storage(both.storage()), both.key_set(), both.dtype());
        v.unsafeGetTensorImpl()->set_sizes_and_strides(c10::IntArrayRef{}, c10::IntArrayRef{}, i);
        return v;
    }
};

// Every GEMM call of this file, on the calling thread's stream, between the two calls of an observer if there is one
void tell(const ntfp8_gemm_desc* d, int n, bool issued) {
    PyObject* shapes = PyTuple_New(n);
    if (shapes == nullptr) throw Stop{};
    for (int i = 0; i < n; ++i) PyTuple_SET_ITEM(shapes, i, Py_BuildValue("(LLL)", (long long)d[i].M, (long long)d[i].N, (long long)d[i].K));
    PyObject* const observer = Py_NewRef(g_observer);
    PyObject* r = PyObject_CallFunction(observer, "ON", issued ? Py_True : Py_False, shapes);
    Py_DECREF(observer);
    if (r == nullptr) throw Stop{};
    Py_DECREF(r);
}
void multiply(const ntfp8_gemm_desc* d, int n, void* stream) {
    const bool observed = g_observer != nullptr;
    if (observed) tell(d, n, false);
    call(ntfp8_gemm_batch(d, n, stream), "ntfp8_gemm_batch");
    if (observed && g_observer != nullptr) tell(d, n, true);
}
void multiply_fp8(ntfp8_gemm_desc& d, int margin, float* state, int hist, const Scalars& s, void* stream) {
    const bool observed = g_observer != nullptr;
    if (observed) tell(&d, 1, false);
    d.amax_workspace = workspace_of(s.both, stream);   // (not before the observer: while it runs, others may drop workspaces)
    call(ntfp8_gemm_fp8(&d, margin, state, state + 1, hist, s.p, s.p + 1, stream), "ntfp8_gemm_fp8");
    if (observed && g_observer != nullptr) tell(&d, 1, true);
}

void rows_cols(const at::Tensor& x, int64_t* rows, int64_t* cols) {
    *cols = x.dim() >= 2 ? x.size(-1) : x.numel();
    *rows = *cols ? x.numel() / *cols : 0;
}

PyObject* quantised(at::Tensor out, at::Tensor out_t, const Scalars& s) {
    return Py_BuildValue("(NNNN)", wrap(std::move(out)), wrap_or_none(std::move(out_t)), wrap(s.element(0)), wrap(s.element(1)));
}

struct Quantised {
    at::Tensor out, out_t;
    Scalars s;
};
PyObject* quantised(Quantised&& q) { return quantised(std::move(q.out), std::move(q.out_t), q.s); }

// Room for the bytes and the scalars of a quantisation.  `together`: one allocation, which nobody outside the call will see
Quantised room_for(const at::Tensor& x, bool together) {
    if (!together) return Quantised{bytes_like(x, x.sizes()), at::Tensor(), Scalars(x)};
    const int64_t n = (x.numel() + 15) / 16 * 16;
    at::Tensor buf = bytes_like(x, {n + 2 * (int64_t)sizeof(float)});
    float* const p = reinterpret_cast<float*>(static_cast<char*>(buf.data_ptr()) + n);
    return Quantised{buf, at::Tensor(), Scalars(buf, p)};
}

// A dense tensor on a CUDA device.  buf [scale, hist[0..H-1]] null: current scaling; flag given: the role may not hold a scale
// yet; otherwise the fused delayed-scaling step
Quantised quantise(const at::Tensor& x, int fmt, int margin, float* buf, float* flag, int hist, bool with_t, bool together = false) {
    int64_t rows, cols;
    rows_cols(x, &rows, &cols);
    require(!with_t || x.dim() == 2, "with_transpose needs a 2-D tensor");
    Quantised q = room_for(x, together);
    if (with_t) q.out_t = bytes_like(x, {cols, rows});
    void* st = stream_of(x);
    void* ws = workspace_of(x, st);
    void* out = q.out.data_ptr();
    void* tp = with_t ? q.out_t.data_ptr() : nullptr;
    const int xd = code_of(x.scalar_type());
    float* const p = q.s.p;
    if (buf == nullptr)
        call(ntfp8_quantize_current(x.data_ptr(), xd, rows, cols, fmt, margin, p, p + 1, out, tp, nullptr, 0, nullptr, ws, st), "ntfp8_quantize_current");
    else if (flag != nullptr)
        call(ntfp8_quantize_first_use(x.data_ptr(), xd, rows, cols, fmt, margin, buf, buf + 1, hist, flag, p, p + 1, out, tp, ws, st), "ntfp8_quantize_first_use");
    else
        call(ntfp8_quantize_delayed(x.data_ptr(), xd, rows, cols, fmt, margin, buf, buf + 1, hist, p, p + 1, out, tp, ws, st), "ntfp8_quantize_delayed");
    return q;
}
Quantised cast_held(const at::Tensor& x, const float* scale, int fmt, bool with_t, bool together = false) {
    int64_t rows, cols;
    rows_cols(x, &rows, &cols);
    require(!with_t || x.dim() == 2, "with_transpose needs a 2-D tensor");
    Quantised q = room_for(x, together);
    if (with_t) q.out_t = bytes_like(x, {cols, rows});
    call(ntfp8_cast_with_scale(x.data_ptr(), code_of(x.scalar_type()), rows, cols, scale, fmt, q.s.p, q.s.p + 1, q.out.data_ptr(),
                               with_t ? q.out_t.data_ptr() : nullptr, stream_of(x)),
         "ntfp8_cast_with_scale");
    return q;
}

// quantize(x, fmt, margin, state | None, flag | None, history_len, with_transpose) -> (bytes, bytes^T | None, amax, scale)
PyObject* quantize(PyObject* const* a) {
    const at::Tensor x = operand(a[0]);
    const int hist = (int)number(a[5]);
    float* const buf = none(a[3]) ? nullptr : values(a[3], x.device(), 1 + hist);
    float* const flag = none(a[4]) ? nullptr : values(a[4], x.device());
    return quantised(quantise(x, (int)number(a[1]), (int)number(a[2]), buf, flag, hist, truth(a[6])));
}

// quantize_batch([(x, state, history_len, margin, with_transpose), ...], fmt) -> [(bytes, bytes^T | None, amax, scale), ...]:
// the fused delayed-scaling step of several tensors, one library call
PyObject* quantize_batch(PyObject* const* args) {
    PyObject* const list = args[0];
    const int fmt = (int)number(args[1]);
    if (!PyList_Check(list)) stop(PyExc_TypeError, "a list of tensors is expected");
    const Py_ssize_t n = PyList_GET_SIZE(list);
    require(n >= 1 && n <= NTFP8_MAX_BATCH, "between 1 and 64 tensors");
    std::vector<ntfp8_quant_desc> d(n);
    std::vector<at::Tensor> x(n), out(n), out_t(n);
    std::vector<Scalars> s;
    s.reserve(n);
    void* st = nullptr;
    at::Tensor pool;
    for (Py_ssize_t i = 0; i < n; ++i) {
        PyObject* t = PyList_GET_ITEM(list, i);
        if (!PyTuple_Check(t) || PyTuple_GET_SIZE(t) != 5) stop(PyExc_TypeError, "a tensor comes as a tuple of 5");
        PyObject* const* f = &PyTuple_GET_ITEM(t, 0);
        x[i] = dense(tensor(f[0]));
        require(x[i].is_cuda() && x[i].device() == x[0].device(), "all tensors of a batch are on one device");
        require(x[i].numel() > 0, "cannot quantise an empty tensor");
        const bool with_t = truth(f[4]);
        require(!with_t || x[i].dim() == 2, "with_transpose needs a 2-D tensor");
        ntfp8_quant_desc& q = d[i];
        q = {};
        q.history_len = (int)number(f[2]);
        q.scale_state = values(f[1], x[0].device(), 1 + q.history_len);
        if (i == 0) {
            st = stream_of(x[0]);
            pool = pool_at((int)x[0].get_device(), st, n);
        }
        rows_cols(x[i], &q.rows, &q.cols);
        out[i] = bytes_like(x[i], x[i].sizes());
        if (with_t) out_t[i] = bytes_like(x[i], {q.cols, q.rows});
        s.emplace_back(x[i]);
        q.x = x[i].data_ptr();
        q.x_dtype = code_of(x[i].scalar_type());
        q.fmt = fmt;
        q.margin = (int)number(f[3]);
        q.amax_history = q.scale_state + 1;
        q.amax_out = s[i].p;
        q.scale_used_out = s[i].p + 1;
        q.out = out[i].data_ptr();
        q.out_t = with_t ? out_t[i].data_ptr() : nullptr;
        q.workspace = static_cast<char*>(pool.data_ptr()) + i * NTFP8_WORKSPACE_BYTES;
    }
    call(ntfp8_quantize_delayed_batch(d.data(), (int)n, st), "ntfp8_quantize_delayed_batch");
    PyObject* res = PyList_New(n);
    if (res == nullptr) throw Stop{};
    for (Py_ssize_t i = 0; i < n; ++i) PyList_SET_ITEM(res, i, quantised(std::move(out[i]), std::move(out_t[i]), s[i]));
    return res;
}

// One GEMM problem: (a, fmt_a, scale_a, b, fmt_b, scale_b, out_code, accumulate_into | None, b_transposed, bias | None,
// a_transposed); fills the descriptor, keeps what it points to alive, returns the output
constexpr int kProblem = 11;
struct Problem {
    at::Tensor a, b, bias, out;
};
void fill(PyObject* const* p, ntfp8_gemm_desc* d, Problem* k, bool fp8_out = false) {
    k->a = dense(tensor(p[0]));
    k->b = dense(tensor(p[3]));
    const bool bt = truth(p[8]), at_ = truth(p[10]);
    require(k->a.dim() == 2 && k->b.dim() == 2 && k->a.size(at_ ? 0 : 1) == k->b.size(bt ? 0 : 1), "GEMM operands do not fit together");
    require(k->a.is_cuda() && k->a.device() == k->b.device(), "GEMM operands must be on one CUDA device");
    codes(k->a), codes(k->b);
    d->scale_a = values(p[2], k->a.device());
    d->scale_b = values(p[5], k->a.device());
    const int64_t M = k->a.size(at_ ? 1 : 0), K = k->a.size(at_ ? 0 : 1), N = k->b.size(bt ? 1 : 0);
    const long code = number(p[6]);
    d->accumulate = 0;
    if (!none(p[7])) {
        k->out = tensor(p[7]);
        require(k->out.scalar_type() == at::kFloat && k->out.dim() == 2 && k->out.size(0) == M && k->out.size(1) == N &&
                    k->out.is_contiguous() && k->out.device() == k->a.device(),
                "accumulate_into must be a contiguous fp32 tensor of the result's shape");
        d->accumulate = 1;
    } else {
        k->out = at::empty({M, N}, at::TensorOptions().dtype(type_of(code)).device(k->a.device()));
    }
    if (!none(p[9])) {
        k->bias = dense(tensor(p[9]));
        require(k->bias.dim() == 1 && k->bias.size(0) == N && k->bias.device() == k->a.device(), "bias must hold one value per output column");
        const int bc = code_of(k->bias.scalar_type());
        require(bc >= 0, "unsupported bias dtype");
        require(!fp8_out || !bt, "no bias together with a transposed B operand");
        d->bias = k->bias.data_ptr();
        d->bias_dtype = bc;
    }
    d->A = k->a.data_ptr();
    d->B = k->b.data_ptr();
    d->D = k->out.data_ptr();
    d->fmt_a = (int)number(p[1]);
    d->fmt_b = (int)number(p[4]);
    d->d_dtype = d->accumulate ? NTFP8_F32 : (int)code;
    d->M = M;
    d->N = N;
    d->K = K;
    d->b_transposed = bt;
    d->a_transposed = at_;
}

// gemm(problem fields...) -> output
PyObject* gemm(PyObject* const* p) {
    ntfp8_gemm_desc d = {};
    Problem k;
    fill(p, &d, &k);
    multiply(&d, 1, stream_of(k.a));
    return wrap(std::move(k.out));
}

// gemm_batch([problem, ...]) -> [output, ...], one library call
PyObject* gemm_batch(PyObject* const* args) {
    PyObject* const list = args[0];
    if (!PyList_Check(list)) stop(PyExc_TypeError, "a list of problems is expected");
    const Py_ssize_t n = PyList_GET_SIZE(list);
    require(n >= 1 && n <= NTFP8_MAX_BATCH, "between 1 and 64 problems");
    std::vector<ntfp8_gemm_desc> d(n);
    std::vector<Problem> k(n);
    for (Py_ssize_t i = 0; i < n; ++i) {
        PyObject* t = PyList_GET_ITEM(list, i);
        if (!PyTuple_Check(t) || PyTuple_GET_SIZE(t) != kProblem) stop(PyExc_TypeError, "a problem is a tuple of 11");
        d[i] = {};
        fill(&PyTuple_GET_ITEM(t, 0), &d[i], &k[i]);
        require(k[i].a.device() == k[0].a.device(), "all problems of a batch are on one device");
    }
    multiply(d.data(), (int)n, stream_of(k[0].a));
    PyObject* out = PyList_New(n);
    if (out == nullptr) throw Stop{};
    for (Py_ssize_t i = 0; i < n; ++i) PyList_SET_ITEM(out, i, wrap(std::move(k[i].out)));
    return out;
}

// gemm_fp8(problem fields..., state, history_len, margin, with_transpose) -> (bytes, bytes^T | None, amax, scale):
// the epilogue casts with the held scale, the workgroup that finishes last does the bookkeeping
PyObject* gemm_fp8(PyObject* const* p) {
    ntfp8_gemm_desc d = {};
    Problem k;
    const int hist = (int)number(p[kProblem + 1]), margin = (int)number(p[kProblem + 2]);
    float* const buf = values(p[kProblem], tensor(p[0]).device(), 1 + hist);
    fill(p, &d, &k, true);
    at::Tensor out_t;
    if (truth(p[kProblem + 3])) out_t = bytes_like(k.a, {d.N, d.M});
    const Scalars s(k.a);
    void* st = stream_of(k.a);
    d.scale_d = buf;
    d.D_t = out_t.defined() ? out_t.data_ptr() : nullptr;
    multiply_fp8(d, margin, buf, hist, s, st);
    return quantised(std::move(k.out), std::move(out_t), s);
}

// cast_with_scale(x, scale, fmt, with_transpose) -> (bytes, bytes^T | None, amax = 0, scale)
PyObject* cast_with_scale(PyObject* const* a) {
    const at::Tensor x = operand(a[0]);
    return quantised(cast_held(x, values(a[1], x.device()), (int)number(a[2]), truth(a[3])));
}

at::Tensor sum_columns(const at::Tensor& x, int out_code) {
    const auto opt = at::TensorOptions().device(x.device());
    at::Tensor out = at::empty({x.size(1)}, opt.dtype(type_of(out_code))), scratch;
    const int64_t need = ntfp8_column_sum_scratch(x.size(0), x.size(1));
    if (need > 0) scratch = at::empty({need / 4}, opt.dtype(at::kFloat));
    void* st = stream_of(x);
    call(ntfp8_column_sum(x.data_ptr(), code_of(x.scalar_type()), x.size(0), x.size(1), out.data_ptr(), out_code,
                          need > 0 ? scratch.data_ptr() : nullptr, workspace_of(x, st), st),
         "ntfp8_column_sum");
    return out;
}
// column_sum([rows, cols], out_code) -> [cols]
PyObject* column_sum(PyObject* const* a) {
    const at::Tensor x = operand(a[0]);
    require(x.dim() == 2, "a 2-D tensor is expected");
    return wrap(sum_columns(x, (int)number(a[1])));
}

// cast(x, scale, fmt, with_transpose) -> (bytes, bytes^T | None)
PyObject* cast(PyObject* const* a) {
    const at::Tensor x = operand(a[0]);
    const int fmt = (int)number(a[2]);
    const float* scale = values(a[1], x.device());
    int64_t rows, cols;
    rows_cols(x, &rows, &cols);
    at::Tensor out = bytes_like(x, x.sizes()), out_t;
    const bool with_t = truth(a[3]);
    require(!with_t || x.dim() == 2, "with_transpose needs a 2-D tensor");
    if (with_t) out_t = bytes_like(x, {cols, rows});
    call(ntfp8_cast_to_fp8(x.data_ptr(), code_of(x.scalar_type()), rows, cols, scale, fmt, out.data_ptr(), with_t ? out_t.data_ptr() : nullptr, stream_of(x)),
         "ntfp8_cast_to_fp8");
    return Py_BuildValue("(NN)", wrap(std::move(out)), wrap_or_none(std::move(out_t)));
}

at::Tensor widened(const at::Tensor& q, int fmt, const float* scale, long code, bool inverse) {   // contiguous bytes
    at::Tensor out = at::empty(q.sizes(), at::TensorOptions().dtype(type_of(code)).device(q.device()));
    if (q.numel()) {
        if (inverse) call(ntfp8_cast_from_fp8_scale_inv(q.data_ptr(), fmt, scale, q.numel(), out.data_ptr(), (int)code, stream_of(q)), "cast_from_fp8");
        else call(ntfp8_cast_from_fp8(q.data_ptr(), fmt, scale, q.numel(), out.data_ptr(), (int)code, stream_of(q)), "ntfp8_cast_from_fp8");
    }
    return out;
}
// dequantize(bytes, fmt, scale, out_code, inverse) -> tensor
PyObject* dequantize(PyObject* const* a) {
    const at::Tensor q = codes(operand(a[0]));
    return wrap(widened(q, (int)number(a[1]), values(a[2], q.device()), number(a[3]), truth(a[4])));
}

at::Tensor turned(const at::Tensor& q) {   // contiguous bytes [rows, cols] -> [cols, rows]
    at::Tensor out = bytes_like(q, {q.size(1), q.size(0)});
    if (q.numel()) call(ntfp8_transpose(q.data_ptr(), q.size(0), q.size(1), out.data_ptr(), stream_of(q)), "ntfp8_transpose");
    return out;
}
// transpose([rows, cols] bytes) -> contiguous [cols, rows] bytes
PyObject* transpose(PyObject* const* a) {
    const at::Tensor q = codes(operand(a[0]));
    require(q.dim() == 2, "a 2-D tensor is expected");
    return wrap(turned(q));
}

// Whether the library reads B [K, N] (and, in the second form, A [K, M] as well) from its transpose: include/ntfp8.h
bool reads_b(int64_t M, int64_t N, int64_t K) {
    return N % 16 == 0 && K % 16 == 0 && M > 128 && N > 128 && K >= 256 && (M + 256) * K < (1LL << 31) && (N + 256) * K < (1LL << 31);
}
PyObject* b_transposed_supported(PyObject* const* a) { return PyBool_FromLong(reads_b(number(a[0]), number(a[1]), number(a[2]))); }

bool aligned16(const at::Tensor& t) { return (reinterpret_cast<uintptr_t>(t.data_ptr()) & 15) == 0; }   // 16-byte loads / stores
// What the library's A and B of D = op(mat_b) . mat_a are: 1 A is mat_b's transposed copy, 2 B is mat_a's transposed copy, 4 B
// read as its transpose, 8 A read as its transpose.  `a_plain`: mat_a may be read as it is.
bool readable(const at::Tensor& a, bool has_copy, bool read_b) { return read_b && !has_copy && a.dim() == 2 && a.is_contiguous() && aligned16(a); }
int form_wgrad(bool a_plain, int64_t K, int64_t N, int64_t M, bool b_plain, bool read_a, bool b_copy_aligned) {
    // D[cols of mat_b, cols of mat_a], reduction over the rows of both
    if (a_plain && read_a && b_plain && M % 16 == 0 && reads_b(M, N, K)) return 4 | 8;
    if (a_plain && b_copy_aligned && reads_b(M, N, K)) return 1 | 4;
    return 1 | 2;
}
int form_dgrad(bool a_plain, int64_t K, int64_t N, int64_t M) { return a_plain && reads_b(M, N, K) ? 4 : 2; }

// operand_form(mat_a, its transposed copy | None, transpose_a, mat_b, its transposed copy | None, transpose_b, accumulate_into |
// None, allow_bt, read_b, read_a) -> bits as above
PyObject* operand_form(PyObject* const* p) {
    const at::Tensor &a = tensor(p[0]), &b = tensor(p[3]);
    require(a.is_cuda() && b.is_cuda(), "The tensors must be on a CUDA device in order to use the FP8 kernel!!");
    const bool ta = truth(p[2]), tb = truth(p[5]);
    if (ta) return PyLong_FromLong(tb ? 1 : 0);
    const bool plain_a = readable(a, !none(p[1]), truth(p[7]) && truth(p[8])) && aligned16(b) && (none(p[6]) || aligned16(tensor(p[6])));
    if (a.dim() != 2 || b.dim() != 2) return PyLong_FromLong(tb ? 1 | 2 : 2);
    // (a copy that has yet to be made is a fresh allocation: aligned)
    if (tb) return PyLong_FromLong(form_wgrad(plain_a, a.size(0), a.size(1), b.size(1), none(p[4]) && b.is_contiguous(), truth(p[9]), none(p[4]) || aligned16(tensor(p[4]))));
    return PyLong_FromLong(form_dgrad(plain_a, a.size(0), a.size(1), b.size(0)));
}

// ---- a layer's passes, one call each.  Between the pieces above a pass of a small layer spends more time in Python than the
// pieces take.  What is not served here (None is returned, nothing launched) takes the way through the pieces.
void gemm_desc(ntfp8_gemm_desc* d, const at::Tensor& a, int fa, const float* sa, const at::Tensor& b, int fb, const float* sb, const at::Tensor& out, int64_t M,
              int64_t N, int64_t K, bool bt, bool at_, bool accumulate) {
    *d = {};
    d->A = a.data_ptr(), d->scale_a = sa, d->fmt_a = fa;
    d->B = b.data_ptr(), d->scale_b = sb, d->fmt_b = fb;
    d->D = out.data_ptr(), d->d_dtype = code_of(out.scalar_type()), d->accumulate = accumulate;
    d->M = M, d->N = N, d->K = K;
    d->b_transposed = bt, d->a_transposed = at_;
}
// an fp8 operand [rows, cols] beside a tensor of that device
bool bytes_of(const at::Tensor& t, c10::Device device) {
    return t.is_cuda() && t.device() == device && t.dim() == 2 && t.element_size() == 1 && t.is_contiguous();
}

// linear_forward(x, fmt, margin, state | None, history_len, held, wants a transposed copy unless dW's GEMM reads the input as it
// is, read_b, weight bytes, fmt, scale, bias | None, out_code, only_y) -> (y, bytes, bytes^T | None, amax, scale) | None: quantisation of the input (current scaling, the fused
// delayed-scaling step, or, with `held`, a cast with the state's scale that leaves the state alone) and Y = X . W^T.  `only_y`: (y,),
// for a pass that nobody will look at the operands of
PyObject* linear_forward(PyObject* const* p) {
    const at::Tensor &input = tensor(p[0]), &w = tensor(p[8]);
    if (!input.is_cuda() || input.dim() < 1 || input.numel() == 0 || code_of(input.scalar_type()) < 0 || !bytes_of(w, input.device()) ||
        input.size(-1) != w.size(1))
        Py_RETURN_NONE;
    const int64_t K = w.size(1), N = w.size(0);
    at::Tensor x = input.dim() == 2 ? input : input.reshape({-1, K});
    x = dense(x);
    const int64_t M = x.size(0);
    const int hist = (int)number(p[4]), fmt = (int)number(p[1]);
    const long out_code = number(p[12]);
    if (out_code < 0 || out_code > NTFP8_BF16) Py_RETURN_NONE;
    const bool held = truth(p[5]);
    if (held && tensor(p[3]).device() != x.device()) Py_RETURN_NONE;   // the pieces bring a held scale over
    float* const buf = none(p[3]) ? nullptr : values(p[3], x.device(), 1 + hist);
    const bool with_t = truth(p[6]) && !(truth(p[7]) && reads_b(N, K, M));
    const float* sw = values(p[10], x.device());
    at::Tensor bias;
    if (!none(p[11])) {
        bias = dense(tensor(p[11]));
        require(bias.dim() == 1 && bias.size(0) == N && bias.device() == x.device(), "bias must hold one value per output column");
        require(code_of(bias.scalar_type()) >= 0, "unsupported bias dtype");
    }
    const bool only_y = truth(p[13]);
    Quantised q = held ? cast_held(x, buf, fmt, with_t, only_y) : quantise(x, fmt, (int)number(p[2]), buf, nullptr, hist, with_t, only_y);
    std::vector<int64_t> shape(input.sizes().begin(), input.sizes().end());
    shape.back() = N;
    at::Tensor y = at::empty(shape, at::TensorOptions().dtype(type_of(out_code)).device(x.device()));
    ntfp8_gemm_desc d;
    gemm_desc(&d, q.out, fmt, q.s.p + 1, w, (int)number(p[9]), sw, y, M, N, K, false, false, false);
    if (bias.defined()) d.bias = bias.data_ptr(), d.bias_dtype = code_of(bias.scalar_type());
    multiply(&d, 1, stream_of(x));
    if (only_y) return Py_BuildValue("(N)", wrap(std::move(y)));
    return Py_BuildValue("(NNNNN)", wrap(std::move(y)), wrap(std::move(q.out)), wrap_or_none(std::move(q.out_t)), wrap(q.s.element(0)), wrap(q.s.element(1)));
}

// linear_forward_fp8(x, its scale where it is fp8 bytes | None, fmt, margin, state | None, history_len, wants a transposed copy unless dW's GEMM
// reads the input as it is, read_b, weight bytes, fmt, scale, bias | None, out_code, (state, history_len, margin, wants a transposed
// copy) of an fp8 output | None) -> ((y, y^T | None, amax, scale) of an fp8 output or y, (bytes, bytes^T | None, amax, scale) of an
// input quantised here | None) | None: the forward pass of a layer that takes or hands on fp8 activations
PyObject* linear_forward_fp8(PyObject* const* p) {
    const at::Tensor &x = tensor(p[0]), &w = tensor(p[8]);
    const bool quantised_already = !none(p[1]), fp8_out = !none(p[13]);
    if (!x.is_cuda() || x.numel() == 0 || !bytes_of(w, x.device()) || x.dim() < 1 || x.size(-1) != w.size(1)) Py_RETURN_NONE;
    if (quantised_already ? !bytes_of(x, x.device()) : code_of(x.scalar_type()) < 0) Py_RETURN_NONE;
    const long out_code = number(p[12]);
    if (out_code < 0 || (out_code > NTFP8_BF16) != fp8_out) Py_RETURN_NONE;
    const int64_t K = w.size(1), N = w.size(0), M = x.numel() / K;
    const int fmt = (int)number(p[2]), hist = (int)number(p[5]);
    const bool with_t = truth(p[6]) && !(truth(p[7]) && reads_b(N, K, M));
    const float *sw = values(p[10], x.device()), *sx = quantised_already ? values(p[1], x.device()) : nullptr;
    float* const buf = quantised_already || none(p[4]) ? nullptr : values(p[4], x.device(), 1 + hist);
    at::Tensor bias;
    if (!none(p[11])) {
        bias = dense(tensor(p[11]));
        require(bias.dim() == 1 && bias.size(0) == N && bias.device() == x.device(), "bias must hold one value per output column");
        require(code_of(bias.scalar_type()) >= 0, "unsupported bias dtype");
    }
    int out_hist = 0, out_margin = 0;
    float* out_state = nullptr;
    bool out_with_t = false;
    if (fp8_out) {
        PyObject* const role = p[13];
        if (!PyTuple_Check(role) || PyTuple_GET_SIZE(role) != 4) stop(PyExc_TypeError, "the role of an fp8 output is a tuple of 4");
        out_hist = (int)number(PyTuple_GET_ITEM(role, 1)), out_margin = (int)number(PyTuple_GET_ITEM(role, 2));
        out_with_t = truth(PyTuple_GET_ITEM(role, 3));
        out_state = values(PyTuple_GET_ITEM(role, 0), x.device(), 1 + out_hist);
    }
    std::optional<Quantised> q;
    if (!quantised_already) {
        at::Tensor h = dense(x);
        if (h.dim() != 2) h = h.view({M, K});
        q = quantise(h, fmt, (int)number(p[3]), buf, nullptr, hist, with_t);
        sx = q->s.p + 1;
    }
    // (an fp8 output is [tokens, features] whatever the input's shape: what the next layer multiplies)
    std::vector<int64_t> shape(x.sizes().begin(), x.sizes().end());
    shape.back() = N;
    if (fp8_out) shape = {M, N};
    at::Tensor y = at::empty(shape, at::TensorOptions().dtype(type_of(out_code)).device(x.device())), y_t;
    ntfp8_gemm_desc d;
    gemm_desc(&d, q ? q->out : x, fmt, sx, w, (int)number(p[9]), sw, y, M, N, K, false, false, false);
    if (bias.defined()) d.bias = bias.data_ptr(), d.bias_dtype = code_of(bias.scalar_type());
    PyObject* res;
    if (fp8_out) {
        if (out_with_t) y_t = bytes_like(x, {N, M});
        const Scalars s(x);
        d.d_dtype = (int)out_code;
        d.scale_d = out_state;
        d.D_t = out_with_t ? y_t.data_ptr() : nullptr;
        multiply_fp8(d, out_margin, out_state, out_hist, s, stream_of(x));
        res = quantised(std::move(y), std::move(y_t), s);
    } else {
        multiply(&d, 1, stream_of(x));
        res = wrap(std::move(y));
    }
    return Py_BuildValue("(NN)", res, q ? quantised(std::move(*q)) : Py_NewRef(Py_None));
}

// linear_backward(dY, its scale where it is fp8 bytes | None, input bytes, their transposed copy | None, fmt, scale, weight bytes, their
// transposed copy | None, fmt, scale, gradient fmt, margin, state | None, history_len, bias code | -1, dX code | -1, (state,
// history_len, margin) of an fp8 dX | None, wants dW, dW to accumulate into | None, read_b, read_a, wants the fp8 dY) -> (bias
// gradient | None, dX | None, dW | None, input bytes^T | None, weight bytes^T | None, (amax, scale) of an fp8 dX | None, (bytes,
// bytes^T | None, amax, scale) of dY, of which a dY that came as bytes has only the second, | None) | None: bias gradient,
// quantisation of dY (current scaling or the fused delayed-scaling step), dX = dY . W and dW = dY^T . X.  Transposed copies that
// a GEMM needs and nobody has made (a weight that more tokens would read as it is) are made here, and the caller is
// given those of the input and the weight, to keep beside them.
PyObject* linear_backward(PyObject* const* p) {
    const at::Tensor &grad = tensor(p[0]), &x = tensor(p[2]), &w = tensor(p[6]);
    const bool quantised_already = !none(p[1]);
    if (!grad.is_cuda() || grad.dim() < 1 || grad.numel() == 0) Py_RETURN_NONE;
    const c10::Device dev = grad.device();
    if (!bytes_of(x, dev) || !bytes_of(w, dev)) Py_RETURN_NONE;
    const int64_t N = w.size(0), K = w.size(1), T = x.size(0);
    if (grad.size(-1) != N || grad.numel() != T * N || x.size(1) != K) Py_RETURN_NONE;
    if (quantised_already ? !bytes_of(grad, dev) || !aligned16(grad) : code_of(grad.scalar_type()) < 0) Py_RETURN_NONE;
    const bool has_xt = !none(p[3]), has_wt = !none(p[7]);
    if ((has_xt && !bytes_of(tensor(p[3]), dev)) || (has_wt && !bytes_of(tensor(p[7]), dev))) Py_RETURN_NONE;
    const bool wants_dw = truth(p[17]), read_b = truth(p[19]), read_a = truth(p[20]);
    const long bias_code = number(p[14]), dx_code = number(p[15]);
    const bool fp8_dx = !none(p[16]);
    if (bias_code > NTFP8_BF16 || (dx_code > NTFP8_BF16) != fp8_dx) Py_RETURN_NONE;
    at::Tensor dw;
    const bool accumulate = !none(p[18]);
    if (accumulate) {
        dw = tensor(p[18]);
        if (dw.scalar_type() != at::kFloat || dw.dim() != 2 || dw.size(0) != N || dw.size(1) != K || !dw.is_contiguous() || dw.device() != dev) Py_RETURN_NONE;
    }
    // the forms of the two GEMMs (bytes that are yet to be made are fresh allocations: aligned), before anything is launched
    const bool with_t = !quantised_already && wants_dw && !(!has_xt && read_a && read_b && N % 16 == 0 && reads_b(N, K, T));
    const int dform = dx_code < 0 ? 0 : form_dgrad(readable(w, has_wt, read_b && !(fp8_dx && T % 4)), N, K, T);
    const int wform = !wants_dw ? 0 : form_wgrad(readable(x, has_xt, read_b) && (!accumulate || aligned16(dw)), T, K, N, !with_t, read_a, true);
    const int hist = (int)number(p[13]), fx = (int)number(p[4]), fw = (int)number(p[8]), fg = (int)number(p[10]);
    const float *sx = values(p[5], dev), *sw = values(p[9], dev);
    float* const buf = none(p[12]) ? nullptr : values(p[12], dev, 1 + hist);
    int dx_hist = 0, dx_margin = 0;
    float* state = nullptr;   // of the role of an fp8 dX
    if (fp8_dx) {
        PyObject* const role = p[16];
        if (!PyTuple_Check(role) || PyTuple_GET_SIZE(role) != 3) stop(PyExc_TypeError, "the role of an fp8 gradient is a tuple of 3");
        dx_hist = (int)number(PyTuple_GET_ITEM(role, 1)), dx_margin = (int)number(PyTuple_GET_ITEM(role, 2));
        state = values(PyTuple_GET_ITEM(role, 0), dev, 1 + dx_hist);
    }

    at::Tensor db, dx, gq, gq_t;
    const float* sg;
    std::optional<Scalars> made, own;   // [amax, scale] of an fp8 dX, of a dY quantised here
    if (quantised_already) {
        gq = grad;
        sg = values(p[1], dev);
        if (bias_code >= 0) db = sum_columns(widened(gq, fg, sg, bias_code, false), (int)bias_code);   // the values of the bytes
    } else {
        at::Tensor g = dense(grad);
        if (g.dim() != 2) g = g.view({T, N});
        if (bias_code >= 0) db = sum_columns(g, (int)bias_code);
        Quantised q = quantise(g, fg, (int)number(p[11]), buf, nullptr, hist, with_t);
        gq = std::move(q.out), gq_t = std::move(q.out_t), own = std::move(q.s);
        sg = own->p + 1;
    }
    at::Tensor xt, wt;    // copies made here
    if ((dform & 2) && !has_wt) wt = turned(w);
    if ((wform & 2) && !has_xt) xt = turned(x);
    if ((wform & 1) && !with_t) gq_t = turned(gq);
    ntfp8_gemm_desc d[2];
    int n = 0;
    const auto opt = at::TensorOptions().device(dev);
    void* const st = stream_of(gq);
    if (dx_code >= 0) {   // dX[T, K] = dY[T, N] . W[N, K]
        dx = at::empty({T, K}, opt.dtype(type_of(dx_code)));
        gemm_desc(&d[0], gq, fg, sg, dform & 4 ? w : has_wt ? tensor(p[7]) : wt, fw, sw, dx, T, K, N, dform & 4, false, false);
        if (fp8_dx) {
            made.emplace(gq);
            d[0].d_dtype = (int)dx_code;
            d[0].scale_d = state;
            multiply_fp8(d[0], dx_margin, state, dx_hist, *made, st);
        } else {
            ++n;
        }
    }
    if (wants_dw) {       // dW[N, K] = dY[T, N]^T . X[T, K]
        if (!accumulate) dw = at::empty({N, K}, opt.dtype(at::kFloat));
        gemm_desc(&d[n++], wform & 8 ? gq : gq_t, fg, sg, wform & 4 ? x : has_xt ? tensor(p[3]) : xt, fx, sx, dw, N, K, T, wform & 4, wform & 8, accumulate);
    }
    if (n) multiply(d, n, st);
    auto pair = [](const std::optional<Scalars>& v) { return v ? Py_BuildValue("(NN)", wrap(v->element(0)), wrap(v->element(1))) : Py_NewRef(Py_None); };
    PyObject* kept = Py_NewRef(Py_None);
    if (truth(p[21])) {
        Py_DECREF(kept);
        kept = own ? quantised(std::move(gq), std::move(gq_t), *own) : Py_BuildValue("(ONOO)", Py_None, wrap_or_none(std::move(gq_t)), Py_None, Py_None);
    }
    return Py_BuildValue("(NNNNNNN)", wrap_or_none(std::move(db)), wrap_or_none(std::move(dx)), wrap_or_none(std::move(dw)), wrap_or_none(std::move(xt)),
                         wrap_or_none(std::move(wt)), pair(made), kept);
}

// workspace(device index) -> (workspace, stream); workspace_pool(device index, count) -> ([>= count] workspaces, stream): what
// the calls above use on torch's current stream of that device
PyObject* with_stream(const at::Tensor& w, void* stream) { return Py_BuildValue("(NN)", wrap(w), PyLong_FromVoidPtr(stream)); }
void* current_stream(int device) {
    return static_cast<void*>(c10::hip::getCurrentHIPStreamMasqueradingAsCUDA((c10::DeviceIndex)device).stream());
}
PyObject* workspace(PyObject* const* a) {
    const int device = (int)number(a[0]);
    void* st = current_stream(device);
    return with_stream(workspace_at(device, st), st);
}
PyObject* workspace_pool(PyObject* const* a) {
    const int device = (int)number(a[0]);
    void* st = current_stream(device);
    return with_stream(pool_at(device, st, number(a[1])), st);
}
PyObject* drop_workspaces(PyObject* const*) {
    workspaces().clear();
    captured_workspaces().clear();
    Py_RETURN_NONE;
}

// set_gemm_observer(callable | None) -> the one before: called as f(issued, ((M, N, K), ...)) right before (issued False) and right
// behind (True) every GEMM call of the library that these functions make, on the thread and the stream that makes it, so that
// whoever times a step can put events there.  It changes nothing about the calls; what it raises, the call raises.
PyObject* set_gemm_observer(PyObject* const* a) {
    if (!none(a[0]) && !PyCallable_Check(a[0])) stop(PyExc_TypeError, "a callable or None is expected");
    PyObject* const before = g_observer == nullptr ? Py_NewRef(Py_None) : g_observer;
    g_observer = none(a[0]) ? nullptr : Py_NewRef(a[0]);
    return before;
}

PyObject* set_check(PyObject* const* a) {
    Py_INCREF(a[0]);
    Py_XSETREF(g_check, a[0]);
    Py_RETURN_NONE;
}

// The common frame: argument count, autograd left out, C++ errors turned into Python ones
template <PyObject* (*F)(PyObject* const*), int N>
PyObject* entry(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != N) {
        PyErr_Format(PyExc_TypeError, "%d arguments are expected, got %zd", N, n);
        return nullptr;
    }
    at::AutoDispatchBelowADInplaceOrView guard;
    try {
        return F(args);
    } catch (const Stop&) {
        return nullptr;
    }
    END_HANDLE_TH_ERRORS
}

#define NT_METHOD(name, count) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&entry<name, count>)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {NT_METHOD(quantize, 7), NT_METHOD(quantize_batch, 2), NT_METHOD(gemm, kProblem), NT_METHOD(gemm_batch, 1), NT_METHOD(gemm_fp8, kProblem + 4),
                         NT_METHOD(cast, 4), NT_METHOD(cast_with_scale, 4), NT_METHOD(column_sum, 2), NT_METHOD(dequantize, 5), NT_METHOD(transpose, 1), NT_METHOD(b_transposed_supported, 3),
                         NT_METHOD(operand_form, 10), NT_METHOD(linear_forward, 14), NT_METHOD(linear_forward_fp8, 14), NT_METHOD(linear_backward, 22),
                         NT_METHOD(workspace, 1), NT_METHOD(workspace_pool, 2), NT_METHOD(drop_workspaces, 0), NT_METHOD(set_check, 1), NT_METHOD(set_gemm_observer, 1), {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_hostcall", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__hostcall(void) { return PyModule_Create(&module); }
