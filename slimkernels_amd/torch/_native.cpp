// The host side of a layer call in native code: from the tensors of a call to its kernel launches through the C ABI
// (include/slimk_w2a8.h), without the interpreter in between.
//
// A decode call's kernels run for 5 to 10 us; the same steps in Python (attribute reads, allocations, a ctypes call of
// twenty arguments per launch) took 8 to 12 us for each launch, so the host was what a small call waited for.  A call among
// others, us: 1 x 4096 x 4096 10.4 -> 6.3, the seven linears of a decoder block at 4 rows 90 -> 50, 1 x 14336 x 4096
// weight-only 10.3 -> 7.6, 77 x 11008 x 4096 28.8 -> 20.5 with its bias in a launch behind (17.5 with it in the kernel).
//
// Every function here handles the plain form of its call (tensors of this device, of the types and layouts the kernels read
// directly, no modes or transforms active) and returns None for anything else, which the Python functions of ops.py and
// w4.py then treat as they always have, refusals included.  Nothing is kept between calls but the library's answers for a shape
// (sizes and routes, pure functions of their arguments).
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/core/GradMode.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPCachingAllocator.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <optional>
#include <unordered_map>
#include <vector>

#include "../../include/slimk_w2a8.h"

namespace {

// ---- the C ABI, bound by address from the library that slimkernels_amd._lib loaded
#define SLIMK_FUNCTIONS(X)                                                                                              \
    X(slimk_w2a8_act_quant_rep) X(slimk_w2a8_gemm_bias) X(slimk_w2a8_gemm_workspace_bytes) X(slimk_w2a8_gemm_auto_route)     \
    X(slimk_w2a8_gemm_fused_bias) X(slimk_w2a8_gemm_fused_workspace_bytes) X(slimk_w2a8_linear_bias) X(slimk_w2a8_linear_route)   \
    X(slimk_w2a8_linear_activation_bytes) X(slimk_w2a8_linear_workspace_bytes) X(slimk_w2a8_gemm_grouped)               \
    X(slimk_w2a16_gemm_bias) X(slimk_w2a16_gemm_workspace_bytes) X(slimk_w4a8_gemm_bias) X(slimk_w4a8_gemm_workspace_bytes)
#define X(name) decltype(&name) p_##name = nullptr;
SLIMK_FUNCTIONS(X)
#undef X
PyObject* g_check = nullptr;   // slimkernels_amd._lib.check: raises for a code other than 0

// interned attribute names
#define SLIMK_NAMES(X) \
    X(w_r) X(s_r) X(zp_r) X(zp_const) X(N) X(K) X(group_size) X(workspaces) X(q) X(s_a) X(rowsum) X(planes) X(uniform_zp8)
#define X(name) PyObject* n_##name = nullptr;
SLIMK_NAMES(X)
#undef X

// a reference that is given back
struct Ref {
    PyObject* p = nullptr;
    Ref() = default;
    explicit Ref(PyObject* o) : p(o) {}
    Ref(const Ref&) = delete;
    Ref& operator=(const Ref&) = delete;
    ~Ref() { Py_XDECREF(p); }
    void take(PyObject* o) { Py_XDECREF(p); p = o; }
};

// Attribute reads that fail (or give something that is no whole number) send the call to the Python path.
bool get(PyObject* o, PyObject* name, Ref& to) {
    to.take(PyObject_GetAttr(o, name));
    if (!to.p) PyErr_Clear();
    return to.p != nullptr;
}
bool to_int(PyObject* o, int& v) {
    if (!PyLong_CheckExact(o)) return false;
    int overflow = 0;
    const long l = PyLong_AsLongAndOverflow(o, &overflow);
    if (overflow || l < INT32_MIN || l > INT32_MAX) return false;
    v = (int)l;
    return true;
}
bool get_int(PyObject* o, PyObject* name, int& v) {
    Ref r;
    return get(o, name, r) && to_int(r.p, v);
}

// A tensor whose memory is what it says: no subclass, no transform around it, strided, on the GPU.
bool plain(PyObject* o) {
    if (!THPVariable_CheckExact(o)) return false;
    const at::Tensor& t = THPVariable_Unpack(o);
    static constexpr c10::DispatchKeySet odd({c10::DispatchKey::Python, c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchGradWrapper,
                                              c10::DispatchKey::Functionalize, c10::DispatchKey::Conjugate, c10::DispatchKey::Negative,
                                              c10::DispatchKey::ZeroTensor});
    return t.defined() && t.is_cuda() && t.layout() == at::kStrided && !t.key_set().has_any(odd) && t.has_storage();
}
bool modes() { return c10::impl::TorchDispatchModeTLS::any_modes_set() || at::impl::torch_function_mode_enabled(); }
bool get_tensor(PyObject* o, PyObject* name, Ref& to) { return get(o, name, to) && plain(to.p); }
const at::Tensor& tensor(const Ref& r) { return THPVariable_Unpack(r.p); }

// 0: float16, 1: bfloat16 (the C ABI's numbers), -1: something else
int dtype_code(at::ScalarType t) { return t == at::kHalf ? SLIMK_F16 : t == at::kBFloat16 ? SLIMK_BF16 : -1; }
int dtype_code(PyObject* o) { return THPDtype_Check(o) ? dtype_code(reinterpret_cast<THPDtype*>(o)->scalar_type) : -1; }
at::ScalarType dtype_of(int code) { return code == SLIMK_BF16 ? at::kBFloat16 : at::kHalf; }

// Token rows [M, K] that the kernels read where they are.
struct Rows {
    const void* p;
    int M, K, ld, dtype;
    at::Device device{at::kCUDA, 0};
    bool of(PyObject* o) {
        if (!plain(o)) return false;
        const at::Tensor& x = THPVariable_Unpack(o);
        dtype = dtype_code(x.scalar_type());
        const int64_t dim = x.dim();
        if (dtype < 0 || dim < 1 || x.numel() <= 0 || x.numel() > INT32_MAX * (int64_t)16) return false;
        const int64_t k = x.size(dim - 1), m = x.numel() / k;
        int64_t pitch = k;
        if (dim == 2) {
            if (x.stride(1) != 1) return false;
            pitch = x.stride(0);
        } else if (!x.is_contiguous()) {
            return false;
        }
        p = x.data_ptr();
        if (pitch % 8 != 0 || pitch < k || (reinterpret_cast<uintptr_t>(p) & 15) != 0) return false;
        if (k > INT32_MAX || m > INT32_MAX || pitch > INT32_MAX) return false;
        M = (int)m, K = (int)k, ld = (int)pitch;
        device = x.device();
        return device.index() == c10::hip::current_device();
    }
};

// The weight of a layer (ops.W2A8Weight); its tensors are held for the call.
struct Weight {
    Ref w_r, s_r, zp_r;
    int zp_const, N, K, group;
    bool of(PyObject* o) {
        return get_tensor(o, n_w_r, w_r) && get_tensor(o, n_s_r, s_r) && get(o, n_zp_r, zp_r) && (zp_r.p == Py_None || plain(zp_r.p)) &&
               get_int(o, n_zp_const, zp_const) && get_int(o, n_N, N) && get_int(o, n_K, K) && get_int(o, n_group_size, group) && N > 0 && K > 0 &&
               group > 0;
    }
    bool per_group() const { return zp_r.p != Py_None; }
    const uint32_t* w() const { return static_cast<const uint32_t*>(tensor(w_r).data_ptr()); }
    const uint16_t* s() const { return static_cast<const uint16_t*>(tensor(s_r).data_ptr()); }
    const uint8_t* z() const { return per_group() ? static_cast<const uint8_t*>(tensor(zp_r).data_ptr()) : nullptr; }
};

// A weight's split-K workspace of the current stream (ops._workspace makes it on a shape's first call there): true with
// ws = nullptr where none is needed, false where there is none yet that is large enough.
bool workspace(PyObject* w, hipStream_t stream, size_t need, Ref& keep, void*& ws, size_t& bytes) {
    ws = nullptr, bytes = 0;
    if (need == 0) return true;
    Ref all, key;
    if (!get(w, n_workspaces, all) || !PyDict_CheckExact(all.p)) return false;
    key.take(PyLong_FromVoidPtr(stream));
    PyObject* t = key.p ? PyDict_GetItem(all.p, key.p) : nullptr;
    if (!t || !plain(t)) return false;
    Py_INCREF(t);
    keep.take(t);
    ws = tensor(keep).data_ptr(), bytes = (size_t)tensor(keep).numel();
    return bytes >= need;
}

// A call's own scratch, given back behind the launches: the next call on the stream gets it again, behind them.
struct Scratch {
    char* p = nullptr;
    Scratch(size_t bytes, hipStream_t stream) {
        if (bytes) p = static_cast<char*>(c10::hip::HIPCachingAllocator::raw_alloc_with_stream(bytes, stream));
    }
    Scratch(const Scratch&) = delete;
    Scratch& operator=(const Scratch&) = delete;
    ~Scratch() {
        if (p) c10::hip::HIPCachingAllocator::raw_delete(p);
    }
};
size_t rounded(size_t bytes) { return (bytes + 255) / 256 * 256; }

// A layer's bias.  The kernels add one that is laid out for them and that no derivative is asked of; any other vector is added
// behind the call, as `y + bias` does; the rest goes the general way.
struct Bias {
    Ref keep;
    const void* p = nullptr;
    bool behind = false;
    bool of(PyObject* o, int N, int dtype, at::Device device) {
        if (o == Py_None) return true;
        if (!plain(o)) return false;
        Py_INCREF(o);
        keep.take(o);
        const at::Tensor& t = tensor(keep);
        // (another width: an error, or on a one-channel layer a wider result that the general code can only give for two dimensions)
        if (t.dim() > 1 || (t.dim() == 1 && t.size(0) != N && t.size(0) != 1)) return false;
        p = t.data_ptr();
        behind = dtype_code(t.scalar_type()) != dtype || t.dim() != 1 || t.size(0) != N || (N > 1 && t.stride(0) != 1) || t.device() != device ||
                 (reinterpret_cast<uintptr_t>(p) & 15) != 0 || (t.requires_grad() && c10::GradMode::is_enabled()) || t._fw_grad(0).defined();
        if (behind) p = nullptr;
        return true;
    }
    at::Tensor add(at::Tensor&& y) const { return behind ? at::add(y, tensor(keep)) : std::move(y); }
};

at::Tensor output(at::IntArrayRef sizes, int dtype, at::Device device) {
    return at::empty(sizes, at::TensorOptions().dtype(dtype_of(dtype)).device(device));
}
// the shape of x with its last extent replaced (x has one or two dimensions, or is contiguous)
at::Tensor output_like(PyObject* x, int N, int dtype, at::Device device) {
    at::DimVector sizes(THPVariable_Unpack(x).sizes());
    sizes.back() = N;
    return output(sizes, dtype, device);
}

PyObject* none() { Py_RETURN_NONE; }
// a call's result, or the exception that slimkernels_amd._lib.check raises for the library's code
PyObject* finish(int rc, at::Tensor&& out, const Bias* bias = nullptr) {
    if (rc == SLIMK_OK) return THPVariable_Wrap(bias ? bias->add(std::move(out)) : std::move(out));
    Py_XDECREF(PyObject_CallFunction(g_check, "i", rc));
    if (!PyErr_Occurred()) PyErr_SetString(PyExc_RuntimeError, "slimk_w2a8 call failed");
    return nullptr;
}

// ---- what the library answers for a shape, asked once (under the interpreter's lock; bounded)
enum Question { kLinear, kGemm, kW2A16, kW4 };
struct Answer {
    size_t ws = 0, act = 0;      // split-K workspace, activation scratch of the digit form
    bool digits = false, sums = true;
};
struct ShapeKey {
    int question, M, N, K, group, zp;
    bool operator==(const ShapeKey& o) const {
        return question == o.question && M == o.M && N == o.N && K == o.K && group == o.group && zp == o.zp;
    }
};
struct ShapeHash {
    size_t operator()(const ShapeKey& k) const {
        uint64_t h = 0x9e3779b97f4a7c15ull;
        for (const int v : {k.question, k.M, k.N, k.K, k.group, k.zp}) h = (h ^ (uint32_t)v) * 0xff51afd7ed558ccdull, h ^= h >> 29;
        return (size_t)h;
    }
};
// zp: 0 the symmetric levels (uniform zero-point 2), 1 another uniform one, 2 one per group
Answer ask(Question q, int M, int N, int K, int group, int zp) {
    static std::unordered_map<ShapeKey, Answer, ShapeHash> known;
    const ShapeKey key{q, M, N, K, group, zp};
    const auto hit = known.find(key);
    if (hit != known.end()) return hit->second;
    Answer a;
    if (q == kLinear && M == 1) {
        a.ws = p_slimk_w2a8_gemm_fused_workspace_bytes(M, N, K, group, 0);
    } else if (q == kLinear && p_slimk_w2a8_linear_route(M, N, K, group, zp == 2)) {
        a.digits = true;
        a.act = p_slimk_w2a8_linear_activation_bytes(M, N, K, group);
        a.ws = p_slimk_w2a8_linear_workspace_bytes(M, N, K, group);
    } else if (q == kLinear || q == kGemm) {
        const int route = p_slimk_w2a8_gemm_auto_route(M, N, K, group);
        a.sums = zp != 0 || group > 256 || (route != 2 && route != 4);
        a.ws = p_slimk_w2a8_gemm_workspace_bytes(M, N, K, group, SLIMK_KERNEL_AUTO, 0);
    } else if (q == kW2A16) {
        a.ws = p_slimk_w2a16_gemm_workspace_bytes(M, N, K, group, 0);
    } else {
        a.ws = p_slimk_w4a8_gemm_workspace_bytes(M, N, K, group, 0);
    }
    if (known.size() >= 4096) known.clear();
    known.emplace(key, a);
    return a;
}
int zp_kind(const Weight& w) { return w.per_group() ? 2 : w.zp_const != 2; }
bool one_pass_w4(int M, int K, int group) { return M >= 33 && K % 128 == 0 && (group == 64 || group == 128); }   // (w4.one_pass_applies)

// quantisation into scratch and the GEMM behind it
int quantise_and_gemm(const Rows& x, const Weight& w, int copies, const Answer& a, bool one_pass_w4, const uint8_t* zp, at::Tensor& out,
                      int odt, const void* bias, void* ws, size_t ws_bytes, hipStream_t stream) {
    const int K = x.K * copies, ldr = (x.M + 3) / 4 * 4;
    const size_t q_bytes = rounded((size_t)x.M * K), s_bytes = rounded((size_t)x.M * 4);
    const size_t sum_bytes = a.sums ? rounded((size_t)copies * (x.K / w.group) * ldr * 4) : 0;
    Scratch scratch(q_bytes + s_bytes + sum_bytes, stream);
    int8_t* const q = reinterpret_cast<int8_t*>(scratch.p);
    float* const s_a = reinterpret_cast<float*>(scratch.p + q_bytes);
    int32_t* const sums = a.sums ? reinterpret_cast<int32_t*>(scratch.p + q_bytes + s_bytes) : nullptr;
    const uint32_t* const w_r = w.w();
    const uint16_t* const s_r = w.s();
    void* const y = out.data_ptr();
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = p_slimk_w2a8_act_quant_rep(x.p, x.ld, x.dtype, x.M, x.K, w.group, copies, q, K, s_a, sums, ldr, stream);
    if (rc == SLIMK_OK)
        rc = one_pass_w4 ? p_slimk_w4a8_gemm_bias(q, K, s_a, zp ? sums : nullptr, ldr, w_r, s_r, zp, x.M, w.N, x.K, w.group, y, w.N, odt, ws,
                                                  ws_bytes, 0, bias, stream)
                         : p_slimk_w2a8_gemm_bias(q, K, s_a, sums, ldr, w_r, s_r, zp, w.zp_const, x.M, w.N, K, w.group, y, w.N, odt, ws,
                                                  ws_bytes, SLIMK_KERNEL_AUTO, 0, bias, stream);
    Py_END_ALLOW_THREADS
    return rc;
}

// linear(x, weight, out_dtype, bias): W2A8Linear
PyObject* linear(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    Rows x;
    Weight w;
    Bias bias;
    const int odt = n == 4 ? dtype_code(args[2]) : -1;
    if (odt < 0 || modes() || !x.of(args[0]) || !w.of(args[1]) || x.K != w.K || !bias.of(args[3], w.N, odt, x.device)) return none();
    const hipStream_t stream = c10::hip::getCurrentHIPStream(x.device.index()).stream();
    const Answer a = ask(kLinear, x.M, w.N, w.K, w.group, zp_kind(w));
    Ref keep;
    void* ws;
    size_t ws_bytes;
    if (!workspace(args[1], stream, a.digits ? 0 : a.ws, keep, ws, ws_bytes)) return none();
    at::Tensor out = output_like(args[0], w.N, odt, x.device);
    int rc;
    if (x.M == 1) {
        const uint32_t* const w_r = w.w();
        const uint16_t* const s_r = w.s();
        const uint8_t* const zp = w.z();
        void* const y = out.data_ptr();
        Py_BEGIN_ALLOW_THREADS
        rc = p_slimk_w2a8_gemm_fused_bias(x.p, x.ld, x.dtype, w_r, s_r, zp, w.zp_const, 1, w.N, w.K, w.group, y, w.N, odt, ws, ws_bytes, 0,
                                          bias.p, stream);
        Py_END_ALLOW_THREADS
    } else if (a.digits) {
        Scratch scratch(a.act + a.ws, stream);
        const uint32_t* const w_r = w.w();
        const uint16_t* const s_r = w.s();
        const uint8_t* const zp = w.z();
        void* const y = out.data_ptr();
        Py_BEGIN_ALLOW_THREADS
        rc = p_slimk_w2a8_linear_bias(x.p, x.ld, x.dtype, w_r, s_r, zp, w.zp_const, x.M, w.N, w.K, w.group, y, w.N, odt, scratch.p, a.act,
                                 a.ws ? scratch.p + a.act : nullptr, a.ws, bias.p, stream);
        Py_END_ALLOW_THREADS
    } else {
        rc = quantise_and_gemm(x, w, 1, a, false, w.z(), out, odt, bias.p, ws, ws_bytes, stream);
    }
    return finish(rc, std::move(out), &bias);
    END_HANDLE_TH_ERRORS
}

// linear16(x, weight, out_dtype, bias): W2A16Linear (ops.w2a16_gemm with its own choice of a split)
PyObject* linear16(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    Rows x;
    Weight w;
    Bias bias;
    const int odt = n == 4 ? dtype_code(args[2]) : -1;
    if (odt < 0 || modes() || !x.of(args[0]) || !w.of(args[1]) || x.K != w.K || !bias.of(args[3], w.N, odt, x.device)) return none();
    const hipStream_t stream = c10::hip::getCurrentHIPStream(x.device.index()).stream();
    const Answer a = ask(kW2A16, x.M, w.N, w.K, w.group, 0);
    at::Tensor out = output_like(args[0], w.N, odt, x.device);
    Scratch scratch(a.ws, stream);
    const uint32_t* const w_r = w.w();
    const uint16_t* const s_r = w.s();
    const uint8_t* const zp = w.z();
    void* const y = out.data_ptr();
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = p_slimk_w2a16_gemm_bias(x.p, x.ld, x.dtype, w_r, s_r, zp, w.zp_const, x.M, w.N, w.K, w.group, y, w.N, odt, scratch.p, a.ws, 0,
                                 bias.p, stream);
    Py_END_ALLOW_THREADS
    return finish(rc, std::move(out), &bias);
    END_HANDLE_TH_ERRORS
}

// linear4(x, weight, out_dtype, bias): W4A8Linear (w4.w4a8_linear) on more than one token row
PyObject* linear4(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    Rows x;
    Weight w;
    Ref planes, uniform;
    int N, K, group;
    Bias bias;
    const int odt = n == 4 ? dtype_code(args[2]) : -1;
    if (odt < 0 || modes() || !x.of(args[0]) || x.M == 1 || !get(args[1], n_planes, planes) || !w.of(planes.p) || !get_int(args[1], n_N, N) ||
        !get_int(args[1], n_K, K) || !get_int(args[1], n_group_size, group) || !get(args[1], n_uniform_zp8, uniform) || !PyBool_Check(uniform.p))
        return none();
    if (x.K != K || w.N != N || w.K != 2 * K || w.group != group || K % group != 0 || !w.per_group() || !bias.of(args[3], N, odt, x.device))
        return none();
    const hipStream_t stream = c10::hip::getCurrentHIPStream(x.device.index()).stream();
    const bool one_pass = one_pass_w4(x.M, K, group);
    Answer a = one_pass ? ask(kW4, x.M, N, K, group, 0) : ask(kGemm, x.M, N, 2 * K, group, zp_kind(w));
    const uint8_t* const zp = one_pass && uniform.p == Py_True ? nullptr : w.z();
    a.sums = !one_pass || zp != nullptr;
    Ref keep;
    void* ws;
    size_t ws_bytes;
    if (!workspace(planes.p, stream, a.ws, keep, ws, ws_bytes)) return none();
    at::Tensor out = output_like(args[0], N, odt, x.device);
    const int rc = quantise_and_gemm(x, w, one_pass ? 1 : 2, a, one_pass, zp, out, odt, bias.p, ws, ws_bytes, stream);
    return finish(rc, std::move(out), &bias);
    END_HANDLE_TH_ERRORS
}

// quantize(x, group_size, copies, rowsum) -> (q, s_a, rowsum or None)
PyObject* quantize(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    Rows x;
    int group, copies;
    if (n != 4 || modes() || !x.of(args[0]) || THPVariable_Unpack(args[0]).dim() != 2 || !to_int(args[1], group) || !to_int(args[2], copies) ||
        group <= 0 || copies < 1 || copies > 64 || !PyBool_Check(args[3]))
        return none();
    const bool sums = args[3] == Py_True;
    const int64_t width = (int64_t)copies * x.K;
    if (width > INT32_MAX || x.M > INT32_MAX - 3) return none();
    const int ldr = (x.M + 3) / 4 * 4;
    const auto opts = at::TensorOptions().device(x.device);
    at::Tensor q = at::empty({x.M, width}, opts.dtype(at::kChar)), s_a = at::empty({x.M}, opts.dtype(at::kFloat)), rs;
    if (sums) rs = at::empty({(int64_t)copies * std::max(x.K / group, 1), ldr}, opts.dtype(at::kInt));
    const hipStream_t stream = c10::hip::getCurrentHIPStream(x.device.index()).stream();
    int8_t* const qp = static_cast<int8_t*>(q.data_ptr());
    float* const sp = static_cast<float*>(s_a.data_ptr());
    int32_t* const rp = sums ? static_cast<int32_t*>(rs.data_ptr()) : nullptr;
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = p_slimk_w2a8_act_quant_rep(x.p, x.ld, x.dtype, x.M, x.K, group, copies, qp, (int)width, sp, rp, ldr, stream);
    Py_END_ALLOW_THREADS
    if (rc != SLIMK_OK) return finish(rc, at::Tensor());
    Ref r0(THPVariable_Wrap(std::move(q))), r1(THPVariable_Wrap(std::move(s_a))), r2(sums ? THPVariable_Wrap(std::move(rs)) : none());
    return PyTuple_Pack(3, r0.p, r1.p, r2.p);
    END_HANDLE_TH_ERRORS
}

// A quantised activation (ops.QuantizedActivation), as quantize() lays it down.
struct Quantised {
    Ref q, s_a, rowsum;
    int M, K, group, ldq, ldr;
    at::Device device{at::kCUDA, 0};
    bool of(PyObject* o) {
        if (!get_tensor(o, n_q, q) || !get_tensor(o, n_s_a, s_a) || !get(o, n_rowsum, rowsum) || !get_int(o, n_group_size, group)) return false;
        const at::Tensor& t = tensor(q);
        if (t.scalar_type() != at::kChar || t.dim() != 2 || t.size(0) > INT32_MAX - 3 || t.size(1) > INT32_MAX || t.stride(0) > INT32_MAX) return false;
        M = (int)t.size(0), K = (int)t.size(1), ldq = (int)t.stride(0), ldr = (M + 3) / 4 * 4;
        if (rowsum.p != Py_None) {
            if (!plain(rowsum.p) || tensor(rowsum).dim() != 2 || tensor(rowsum).stride(0) > INT32_MAX) return false;
            ldr = (int)tensor(rowsum).stride(0);
        }
        device = t.device();
        return M > 0 && K > 0 && device.index() == c10::hip::current_device();
    }
    const int8_t* qp() const { return static_cast<const int8_t*>(tensor(q).data_ptr()); }
    const float* sp() const { return static_cast<const float*>(tensor(s_a).data_ptr()); }
    const int32_t* rp() const { return rowsum.p == Py_None ? nullptr : static_cast<const int32_t*>(tensor(rowsum).data_ptr()); }
};

// gemm(qa, weight, out_dtype): ops.w2a8_gemm with its own choices
PyObject* gemm(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    Quantised x;
    Weight w;
    const int odt = n == 3 ? dtype_code(args[2]) : -1;
    if (odt < 0 || modes() || !x.of(args[0]) || !w.of(args[1]) || x.K != w.K || x.group != w.group) return none();
    const hipStream_t stream = c10::hip::getCurrentHIPStream(x.device.index()).stream();
    const Answer a = ask(kGemm, x.M, w.N, w.K, w.group, zp_kind(w));
    Ref keep;
    void* ws;
    size_t ws_bytes;
    if (!workspace(args[1], stream, a.ws, keep, ws, ws_bytes)) return none();
    at::Tensor out = output({x.M, w.N}, odt, x.device);
    const int8_t* const q = x.qp();
    const float* const s_a = x.sp();
    const int32_t* const sums = x.rp();
    const uint32_t* const w_r = w.w();
    const uint16_t* const s_r = w.s();
    const uint8_t* const zp = w.z();
    void* const y = out.data_ptr();
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = p_slimk_w2a8_gemm_bias(q, x.ldq, s_a, sums, x.ldr, w_r, s_r, zp, w.zp_const, x.M, w.N, w.K, w.group, y, w.N, odt, ws, ws_bytes,
                                SLIMK_KERNEL_AUTO, 0, nullptr, stream);
    Py_END_ALLOW_THREADS
    return finish(rc, std::move(out));
    END_HANDLE_TH_ERRORS
}

// grouped(problems, out_dtype): ops.w2a8_gemm_grouped of one launch without a dump
PyObject* grouped(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    const int odt = n == 2 ? dtype_code(args[1]) : -1;
    const bool list = PyList_CheckExact(args[0]);
    if (odt < 0 || modes() || (!list && !PyTuple_CheckExact(args[0]))) return none();
    // (a tuple of its own: another thread may change a list while the lock is given up)
    Ref problems(list ? PyList_AsTuple(args[0]) : (Py_INCREF(args[0]), args[0]));
    const Py_ssize_t count = problems.p ? PyTuple_GET_SIZE(problems.p) : 0;
    if (count < 1 || count > SLIMK_W2A8_MAX_GROUP) return none();
    Quantised x[SLIMK_W2A8_MAX_GROUP];
    Weight w[SLIMK_W2A8_MAX_GROUP];
    slimk_w2a8_problem table[SLIMK_W2A8_MAX_GROUP];
    // everything is looked at before anything is allocated
    for (Py_ssize_t i = 0; i < count; ++i) {
        PyObject* const pr = PyTuple_GET_ITEM(problems.p, i);
        if (!PyTuple_CheckExact(pr)) return none();
        const Py_ssize_t parts = PyTuple_GET_SIZE(pr);
        if (parts < 2 || !x[i].of(PyTuple_GET_ITEM(pr, 0)) || !w[i].of(PyTuple_GET_ITEM(pr, 1))) return none();
        if (x[i].K != w[i].K || x[i].group != w[i].group || w[i].group != w[0].group || x[i].rowsum.p == Py_None ||
            x[i].device != x[0].device)
            return none();
        PyObject* const out = parts > 2 ? PyTuple_GET_ITEM(pr, 2) : Py_None;
        if (out != Py_None) {
            if (!plain(out)) return none();
            const at::Tensor& o = THPVariable_Unpack(out);
            if (dtype_code(o.scalar_type()) != odt || o.dim() < 1 || o.stride(0) > INT32_MAX) return none();
        }
    }
    Ref outs(PyList_New(count));
    if (!outs.p) return nullptr;
    for (Py_ssize_t i = 0; i < count; ++i) {
        PyObject* const pr = PyTuple_GET_ITEM(problems.p, i);
        PyObject* out = PyTuple_GET_SIZE(pr) > 2 ? PyTuple_GET_ITEM(pr, 2) : Py_None;
        if (out == Py_None) out = THPVariable_Wrap(output({x[i].M, w[i].N}, odt, x[0].device));
        else Py_INCREF(out);
        if (!out) return nullptr;
        PyList_SET_ITEM(outs.p, i, out);
        const at::Tensor& o = THPVariable_Unpack(out);
        slimk_w2a8_problem& t = table[i];
        t.q = x[i].qp(), t.s_a = x[i].sp(), t.rowsum = x[i].rp();
        t.w_r = w[i].w(), t.s_r = w[i].s(), t.zp_r = w[i].z();
        t.out = o.data_ptr();
        t.ldq = x[i].ldq, t.ldr = x[i].ldr, t.ldo = (int)o.stride(0);
        t.M = x[i].M, t.N = w[i].N, t.K = w[i].K, t.zp_const = w[i].zp_const;
    }
    const hipStream_t stream = c10::hip::getCurrentHIPStream(x[0].device.index()).stream();
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = p_slimk_w2a8_gemm_grouped(table, (int)count, w[0].group, odt, stream);
    Py_END_ALLOW_THREADS
    if (rc != SLIMK_OK) return finish(rc, at::Tensor());
    PyObject* const r = outs.p;
    outs.p = nullptr;
    return r;
    END_HANDLE_TH_ERRORS
}

// rules(M, N, K, group_size, zp) -> (digits, sums, workspace, scratch, one_pass_w4): what the functions above decide by a call's
// shape, to be held against ops.linear_digits_applies, ops.needs_rowsum, w4.one_pass_applies and the library's sizes
PyObject* rules(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    int v[5];
    for (int i = 0; i < 5; ++i)
        if (n != 5 || !to_int(args[i], v[i])) return none();
    if (!g_check) return none();
    const Answer a = ask(kLinear, v[0], v[1], v[2], v[3], v[4]), b = ask(kGemm, v[0], v[1], v[2], v[3], v[4]);
    return Py_BuildValue("(OOnnO)", a.digits ? Py_True : Py_False, b.sums ? Py_True : Py_False, (Py_ssize_t)a.ws, (Py_ssize_t)a.act,
                         one_pass_w4(v[0], v[2], v[3]) ? Py_True : Py_False);
    END_HANDLE_TH_ERRORS
}

// bind(addresses, check): the C ABI's functions by name, and what raises for their codes
PyObject* bind(PyObject*, PyObject* const* args, Py_ssize_t n) {
    if (n != 2 || !PyDict_Check(args[0]) || !PyCallable_Check(args[1])) {
        PyErr_SetString(PyExc_TypeError, "bind(addresses, check)");
        return nullptr;
    }
#define X(name)                                                                   \
    {                                                                             \
        PyObject* a = PyDict_GetItemString(args[0], #name);                       \
        void* v = a ? PyLong_AsVoidPtr(a) : nullptr;                              \
        if (!v) {                                                                 \
            if (!PyErr_Occurred()) PyErr_SetString(PyExc_KeyError, #name);        \
            return nullptr;                                                       \
        }                                                                         \
        p_##name = reinterpret_cast<decltype(p_##name)>(v);                       \
    }
    SLIMK_FUNCTIONS(X)
#undef X
    Py_INCREF(args[1]);
    Py_XDECREF(g_check);
    g_check = args[1];
    Py_RETURN_NONE;
}

template <PyObject* (*F)(PyObject*, PyObject* const*, Py_ssize_t)>
constexpr PyCFunction fast() { return reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(F)); }

PyMethodDef g_methods[] = {
    {"bind", fast<bind>(), METH_FASTCALL, "bind(addresses, check)"},
    {"linear", fast<linear>(), METH_FASTCALL, "linear(x, weight, out_dtype, bias) -> tensor, or None for the general path"},
    {"linear16", fast<linear16>(), METH_FASTCALL, "linear16(x, weight, out_dtype, bias) -> tensor or None"},
    {"linear4", fast<linear4>(), METH_FASTCALL, "linear4(x, weight, out_dtype, bias) -> tensor or None"},
    {"quantize", fast<quantize>(), METH_FASTCALL, "quantize(x, group_size, copies, rowsum) -> (q, s_a, rowsum) or None"},
    {"gemm", fast<gemm>(), METH_FASTCALL, "gemm(qa, weight, out_dtype) -> tensor or None"},
    {"rules", fast<rules>(), METH_FASTCALL, "rules(M, N, K, group_size, zp) -> what a call's shape decides (zp 0: symmetric levels, 1: uniform, 2: per group)"},
    {"grouped", fast<grouped>(), METH_FASTCALL, "grouped(problems, out_dtype) -> list of tensors or None"},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "_native", "Native host side of the layer calls.", -1, g_methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__native() {
#define X(name) if (!(n_##name = PyUnicode_InternFromString(#name))) return nullptr;
    SLIMK_NAMES(X)
#undef X
    return PyModule_Create(&g_module);
}
