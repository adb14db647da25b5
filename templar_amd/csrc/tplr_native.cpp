// The per-parameter calls' host path (templar_amd._native): what templar_amd/compress.py does around one library call
// - look at the inputs, allocate the outputs, launch on torch's current stream - in one native call.
//
// A miner or validator that keeps the reference's loop makes these calls for every parameter of a model, and the kernels
// behind them take a few microseconds each: in Python an allocation costs 1.3-1.7 us, the current stream 2 us, a
// no_grad context 1 us, every pointer list a microsecond per peer, and `encode` + `compress` of a 2048 x 2048 parameter
// took 27 us of host time around 19 us of kernels.
//
// Every function serves plain inputs only - exact torch tensors, fp32 (codes: uint8), contiguous, on the GPU, the shapes
// the kernels take - and answers None for anything else: the caller then converts and calls again, or raises.  The
// arithmetic is the library's alone; its entry points are handed over by address (bind), so that the library in use is
// the one templar_amd._lib has loaded.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/core/Tensor.h>
#include <ATen/ops/empty.h>
#include <ATen/ops/empty_strided.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/object_ptr.h>

#include <chrono>
#include <vector>

#include "../../include/tplr_hip.h"

namespace {

// ---- the library's entry points ---------------------------------------------------------------
#define TPLR_NATIVE_ENTRIES(X)                                                                            \
    X(tplr_status_string) X(tplr_dct2d_fwd) X(tplr_dct2d_inv) X(tplr_dct1d) X(tplr_topk_pack)                \
    X(tplr_encode_topk_pack) X(tplr_aggregate_param) X(tplr_decompress_codes) X(tplr_decompress_rows)        \
    X(tplr_clip_scales) X(tplr_peer_sumsq) X(tplr_quantize) X(tplr_dequantize_lists) X(tplr_unchunk)                \
    X(tplr_check_rows) X(tplr_dct2d_dense)
#define X(name) decltype(&::name) p_##name = nullptr;
TPLR_NATIVE_ENTRIES(X)
#undef X
PyObject* error_class = nullptr;    // templar_amd._lib.TplrHipError
PyObject* float32_dtype = nullptr;  // torch.float32

PyObject* bind(PyObject*, PyObject* const* args, Py_ssize_t n) {
    // bind({entry point: address}, error class, torch.float32)
    if (n != 3 || !PyDict_Check(args[0])) {
        PyErr_SetString(PyExc_TypeError, "bind(addresses, error, float32)");
        return nullptr;
    }
#define X(name)                                                                  \
    {                                                                            \
        PyObject* a = PyDict_GetItemString(args[0], #name);                      \
        void* p = a ? PyLong_AsVoidPtr(a) : nullptr;                             \
        if (!p) {                                                                \
            if (!PyErr_Occurred()) PyErr_SetString(PyExc_KeyError, #name);       \
            return nullptr;                                                      \
        }                                                                        \
        p_##name = reinterpret_cast<decltype(&::name)>(p);                       \
    }
    TPLR_NATIVE_ENTRIES(X)
#undef X
    Py_XDECREF(error_class);
    Py_XDECREF(float32_dtype);
    error_class = Py_NewRef(args[1]);
    float32_dtype = Py_NewRef(args[2]);
    Py_RETURN_NONE;
}

PyObject* failed(int status, const char* what) {
    PyErr_Format(error_class, "%s: %s (status %d)", what, p_tplr_status_string(status), status);
    return nullptr;
}

// ---- inputs and outputs -----------------------------------------------------------------------
// A plain device tensor of this type, or nullptr.
const at::Tensor* plain(PyObject* o, c10::ScalarType type) {
    if (!THPVariable_CheckExact(o)) return nullptr;
    const at::Tensor& t = THPVariable_Unpack(o);
    return t.is_cuda() && t.scalar_type() == type && t.layout() == c10::kStrided ? &t : nullptr;
}

const at::Tensor* plain_f32(PyObject* o) { return plain(o, c10::ScalarType::Float); }

// An operation on this tensor would be plain dispatch to the device: no tangent, no transform (vmap, jvp), tracer or mode would
// see it.  For what has been torch's own operation: a launch in its place is invisible to those.
bool nobody_else(const at::Tensor& t) {
    using c10::DispatchKey;
    const c10::DispatchKeySet plain_keys({DispatchKey::Dense, DispatchKey::CUDA, DispatchKey::AutogradCUDA, DispatchKey::ADInplaceOrView,
                                          DispatchKey::AutocastCUDA, DispatchKey::BackendSelect});
    const c10::DispatchKeySet usual = plain_keys | c10::default_included_set;
    const c10::impl::LocalDispatchKeySet tls = c10::impl::tls_local_dispatch_key_set();
    return ((t.key_set() | tls.included_).raw_repr() & ~usual.raw_repr()) == 0 && !t._fw_grad(0).defined();
}

at::Tensor fresh(at::IntArrayRef sizes, c10::ScalarType type, const at::Tensor& like) {
    return at::empty(sizes, at::TensorOptions().dtype(type).device(like.device()));
}

constexpr uint32_t kUnset = 0xffffffffu;  // as a float a NaN, which the quantiser's scale never is

// launches go to the tensor's device and that device's current stream
struct Launch {
    int before, here;
    explicit Launch(const at::Tensor& t) : before(c10::hip::current_device()), here(t.device().index()) {
        if (before != here) c10::hip::set_device(here);
    }
    ~Launch() {
        if (before != here) c10::hip::set_device(before);
    }
    void* stream() const { return c10::hip::getCurrentHIPStream(here).stream(); }
    // other Python threads run meanwhile
    struct Released {
        PyThreadState* state = PyEval_SaveThread();
        ~Released() { PyEval_RestoreThread(state); }
    };
    // wait for the stream
    void wait() const {
        Released released;
        c10::hip::getCurrentHIPStream(here).unwrap().synchronize();
    }
    // wait until kernels of the stream have stored something else than kUnset in each of n words of pinned memory, which they do
    // with system-scope stores; for the stream where half a millisecond does not bring them (work queued before, an error).
    // The interpreter is given up once for all of them: beside a busy thread it comes back a switch interval later.
    void wait_for(const uint32_t* words, int64_t n) const {
        Released released;
        const auto give_up = std::chrono::steady_clock::now() + std::chrono::microseconds(500);
        for (int64_t i = 0; i < n; ++i)
            while (__atomic_load_n(words + i, __ATOMIC_ACQUIRE) == kUnset)
                if (std::chrono::steady_clock::now() > give_up) {
                    c10::hip::getCurrentHIPStream(here).unwrap().synchronize();
                    return;
                }
    }
};

bool to_int(PyObject* o, int64_t& out) {
    const long long v = PyLong_AsLongLong(o);  // (through __index__)
    if (v == -1 && PyErr_Occurred()) {
        PyErr_Clear();
        return false;
    }
    out = v;
    return true;
}

// min(topk, n), at least 2, rounded down to even (src/tplr/compress.py:352-367)
int64_t clamp_k(int64_t n, int64_t topk) {
    int64_t k = topk < n ? topk : n;
    k = k > 2 ? k : 2;
    return k - (k & 1);
}

constexpr int64_t kEdge = 64;

// xshape as (Y, X, 64, 64)
bool chunk_shape(PyObject* o, int64_t& Y, int64_t& X) {
    if (!PyTuple_Check(o) || PyTuple_GET_SIZE(o) != 4) return false;  // (torch.Size is a tuple)
    int64_t h, w;
    return to_int(PyTuple_GET_ITEM(o, 0), Y) && to_int(PyTuple_GET_ITEM(o, 1), X) && to_int(PyTuple_GET_ITEM(o, 2), h) &&
           to_int(PyTuple_GET_ITEM(o, 3), w) && h == kEdge && w == kEdge && Y > 0 && X > 0;
}

// The (edge, edge) basis of a chunk edge, plain and on the tensor's device, or nullptr.
const float* basis_of(PyObject* bases, int64_t edge, const at::Tensor& x) {
    PyObject* key = PyLong_FromLongLong(edge);
    PyObject* found = key ? PyDict_GetItemWithError(bases, key) : nullptr;
    Py_XDECREF(key);
    const at::Tensor* b = found ? plain_f32(found) : nullptr;
    PyErr_Clear();
    return b && b->dim() == 2 && b->size(0) == edge && b->size(1) == edge && b->is_contiguous() && b->device() == x.device()
               ? b->const_data_ptr<float>()
               : nullptr;
}

// ---- encode(x, use_dct=True) ------------------------------------------------------------------
// encode(x, shape_dict, bases): the transforms of a registered 2-D parameter, or of a 1-D one in chunks of 64
PyObject* encode(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 3) return PyErr_SetString(PyExc_TypeError, "encode(x, shape_dict, bases)"), nullptr;
    const at::Tensor* x = plain_f32(args[0]);
    if (!x || !PyDict_Check(args[1]) || !PyDict_Check(args[2]) || x->numel() == 0 || x->dim() < 1 || x->dim() > 2) Py_RETURN_NONE;
    int64_t edges[2] = {0, 0};
    for (int64_t d = 0; d < x->dim(); ++d) {
        PyObject* key = PyLong_FromLongLong(x->size(d));
        PyObject* edge = key ? PyDict_GetItemWithError(args[1], key) : nullptr;
        Py_XDECREF(key);
        if (!edge || !to_int(edge, edges[d])) {
            PyErr_Clear();
            Py_RETURN_NONE;
        }
    }
    Launch on(*x);
    if (x->dim() == 1) {
        if (!x->is_contiguous() || edges[0] != kEdge) Py_RETURN_NONE;
        at::Tensor out = fresh({x->size(0) / kEdge, kEdge}, c10::ScalarType::Float, *x);
        if (int st = p_tplr_dct1d(x->const_data_ptr<float>(), x->size(0) / kEdge, 0, out.data_ptr<float>(), on.stream()))
            return failed(st, "tplr_dct1d");
        return THPVariable_Wrap(std::move(out));
    }
    const int64_t R = x->size(0), C = x->size(1), h = edges[0], w = edges[1];
    if (h != kEdge || w != kEdge) {
        if (h < 1 || w < 1 || h > kEdge || w > kEdge || R % h || C % w || !x->is_contiguous()) Py_RETURN_NONE;
        const float *bh = basis_of(args[2], h, *x), *bw = basis_of(args[2], w, *x);
        if (!bh || !bw) Py_RETURN_NONE;
        at::Tensor out = fresh({R / h, C / w, h, w}, c10::ScalarType::Float, *x);
        if (int st = p_tplr_dct2d_dense(x->const_data_ptr<float>(), R, C, static_cast<int>(h), static_cast<int>(w), bh, bw, 0, 1,
                                        out.data_ptr<float>(), on.stream()))
            return failed(st, "tplr_dct2d_dense");
        return THPVariable_Wrap(std::move(out));
    }
    if (x->stride(1) != 1 || x->stride(0) < C) Py_RETURN_NONE;
    at::Tensor out = fresh({R / kEdge, C / kEdge, kEdge, kEdge}, c10::ScalarType::Float, *x);
    if (int st = p_tplr_dct2d_fwd(x->const_data_ptr<float>(), R, C, x->stride(0), out.data_ptr<float>(), on.stream()))
        return failed(st, "tplr_dct2d_fwd");
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// ---- decode -----------------------------------------------------------------------------------
// the (Y, X, 64, 64) view of a row-major (R, C) tensor, without gaps between its elements or with
bool chunk_view(const at::Tensor& x) {
    return x.dim() == 4 && x.size(2) == kEdge && x.size(3) == kEdge && x.stride(3) == 1 && x.stride(1) == kEdge &&
           x.stride(2) >= x.size(1) * kEdge && (x.stride(0) == kEdge * x.stride(2) || x.size(0) == 1);
}

// decode(x, use_dct, bases): chunks or rows of 64 back into their tensor
PyObject* decode(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 3) return PyErr_SetString(PyExc_TypeError, "decode(x, use_dct, bases)"), nullptr;
    const at::Tensor* x = plain_f32(args[0]);
    if (!x || x->numel() == 0) Py_RETURN_NONE;
    if (args[1] != Py_True) {  // a change of shape: of a view of the tensor itself, the tensor; of whole chunks a copy
        if (x->requires_grad()) Py_RETURN_NONE;
        if (chunk_view(*x)) return THPVariable_Wrap(x->as_strided({x->size(0) * kEdge, x->size(1) * kEdge}, {x->stride(2), 1}));
        if (x->dim() != 4 || !x->is_contiguous()) Py_RETURN_NONE;
        // (one column of chunks is the tensor already: a view)
        if (x->size(1) > 1 && x->size(2) == kEdge && x->size(3) == kEdge && nobody_else(*x) &&
            reinterpret_cast<uintptr_t>(x->const_data_ptr()) % 16 == 0) {
            const int64_t R = x->size(0) * kEdge, C = x->size(1) * kEdge;
            Launch on(*x);
            at::Tensor out = fresh({R, C}, c10::ScalarType::Float, *x);
            const int st = p_tplr_unchunk(x->const_data_ptr<float>(), R, C, out.data_ptr<float>(), on.stream());
            if (st == 0) return THPVariable_Wrap(std::move(out));
            if (st != TPLR_E_TOOMANY) return failed(st, "tplr_unchunk");
        }
        return THPVariable_Wrap(x->permute({0, 2, 1, 3}).reshape({x->size(0) * x->size(2), x->size(1) * x->size(3)}));
    }
    Launch on(*x);
    if (x->dim() == 4 && x->size(2) == kEdge && x->size(3) == kEdge) {
        const int64_t R = x->size(0) * kEdge, C = x->size(1) * kEdge;
        if (!x->is_contiguous()) Py_RETURN_NONE;
        at::Tensor out = fresh({R, C}, c10::ScalarType::Float, *x);
        if (int st = p_tplr_dct2d_inv(x->const_data_ptr<float>(), R, C, out.data_ptr<float>(), C, on.stream()))
            return failed(st, "tplr_dct2d_inv");
        return THPVariable_Wrap(std::move(out));
    }
    if (x->dim() == 4 && x->size(2) <= kEdge && x->size(3) <= kEdge && x->is_contiguous() && PyDict_Check(args[2])) {
        const int64_t h = x->size(2), w = x->size(3), R = x->size(0) * h, C = x->size(1) * w;
        const float *bh = basis_of(args[2], h, *x), *bw = basis_of(args[2], w, *x);
        if (!bh || !bw) Py_RETURN_NONE;
        at::Tensor out = fresh({R, C}, c10::ScalarType::Float, *x);
        if (int st = p_tplr_dct2d_dense(x->const_data_ptr<float>(), R, C, static_cast<int>(h), static_cast<int>(w), bh, bw, 1, 0,
                                        out.data_ptr<float>(), on.stream()))
            return failed(st, "tplr_dct2d_dense");
        return THPVariable_Wrap(std::move(out));
    }
    if (x->dim() == 2 && x->size(1) == kEdge && x->is_contiguous()) {
        at::Tensor out = fresh({x->numel()}, c10::ScalarType::Float, *x);
        if (int st = p_tplr_dct1d(x->const_data_ptr<float>(), x->size(0), 1, out.data_ptr<float>(), on.stream()))
            return failed(st, "tplr_dct1d");
        return THPVariable_Wrap(std::move(out));
    }
    Py_RETURN_NONE;
    END_HANDLE_TH_ERRORS
}

// ---- the quantiser ----------------------------------------------------------------------------
// (codes, quant_params) of fp32 values; a new reference, or nullptr with an exception set
PyObject* quantised(const at::Tensor& val, int64_t n_bins, double range, const Launch& on) {
    const int64_t n = val.numel();
    at::Tensor codes = fresh(val.sizes(), c10::ScalarType::Byte, val);
    at::Tensor shift = fresh({}, c10::ScalarType::Float, val), lookup = fresh({n_bins}, c10::ScalarType::Float, val);
    // a workgroup per 1024 values (one load per thread), one per compute unit at most
    const int64_t slices = n / 1024 < 1 ? 1 : n / 1024 > 256 ? 256 : n / 1024;
    at::Tensor work = fresh({slices * (2 + 2 * n_bins) + 1}, c10::ScalarType::Double, val);
    // the scale is the one figure that travels to the host (float(scale), src/tplr/compress.py:620): the second launch
    // stores it in pinned memory as it begins, and only that store is waited for
    at::Tensor scale = at::empty({1}, at::TensorOptions().dtype(c10::ScalarType::Float).pinned_memory(true));
    uint32_t* const word = reinterpret_cast<uint32_t*>(scale.data_ptr<float>());
    __atomic_store_n(word, kUnset, __ATOMIC_RELAXED);
    if (int st = p_tplr_quantize(val.const_data_ptr<float>(), n, static_cast<int>(n_bins), static_cast<float>(range),
                                 static_cast<int>(slices), work.data_ptr<double>(), codes.data_ptr<uint8_t>(),
                                 shift.data_ptr<float>(), scale.data_ptr<float>(), lookup.data_ptr<float>(), on.stream()))
        return failed(st, "tplr_quantize");
    on.wait_for(word, 1);
    return Py_BuildValue("(N(NdLNO))", THPVariable_Wrap(std::move(codes)), THPVariable_Wrap(std::move(shift)),
                         static_cast<double>(*scale.const_data_ptr<float>()), static_cast<long long>(n_bins / 2),
                         THPVariable_Wrap(std::move(lookup)), float32_dtype);
}

bool can_quantise(const at::Tensor& v, int64_t n_bins) {
    return v.numel() >= 4 && v.numel() % 4 == 0 && n_bins >= 1 && n_bins <= 256 && v.is_contiguous() &&
           reinterpret_cast<uintptr_t>(v.const_data_ptr()) % 16 == 0;
}

// quantize(values, n_bins, range) -> (codes, quant_params)
PyObject* quantize(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    int64_t bins;
    if (n != 3) return PyErr_SetString(PyExc_TypeError, "quantize(values, n_bins, range)"), nullptr;
    const at::Tensor* v = plain_f32(args[0]);
    const double range = PyFloat_AsDouble(args[2]);
    if (range == -1.0 && PyErr_Occurred()) {
        PyErr_Clear();
        Py_RETURN_NONE;
    }
    if (!v || !to_int(args[1], bins) || !can_quantise(*v, bins)) Py_RETURN_NONE;
    Launch on(*v);
    return quantised(*v, bins, range, on);
    END_HANDLE_TH_ERRORS
}

// dequantize(codes list, quant_params list) -> list of fp32 tensors: one parameter's codes of several peers
PyObject* dequantize(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 2 || !PyList_Check(args[0]) || !PyList_Check(args[1])) Py_RETURN_NONE;
    const Py_ssize_t P = PyList_GET_SIZE(args[0]);
    if (P < 1 || P > TPLR_MAX_PEERS || PyList_GET_SIZE(args[1]) < P) Py_RETURN_NONE;
    const uint8_t* codes[TPLR_MAX_PEERS];
    const float *lookup[TPLR_MAX_PEERS], *shift[TPLR_MAX_PEERS];
    float* out[TPLR_MAX_PEERS];
    const at::Tensor* first = nullptr;
    int64_t bins = 0;
    for (Py_ssize_t p = 0; p < P; ++p) {
        const at::Tensor* c = plain(PyList_GET_ITEM(args[0], p), c10::ScalarType::Byte);
        PyObject* qp = PyList_GET_ITEM(args[1], p);
        if (!c || !c->is_contiguous() || !PyTuple_Check(qp) || PyTuple_GET_SIZE(qp) != 5) Py_RETURN_NONE;
        const at::Tensor* s = plain_f32(PyTuple_GET_ITEM(qp, 0));
        const at::Tensor* l = plain_f32(PyTuple_GET_ITEM(qp, 3));
        if (!s || !l || s->dim() != 0 || l->dim() != 1 || !l->is_contiguous() || PyTuple_GET_ITEM(qp, 4) != float32_dtype)
            Py_RETURN_NONE;
        if (p == 0) first = c, bins = l->numel();
        if (c->numel() != first->numel() || l->numel() != bins || c->device() != first->device() ||
            s->device() != first->device() || l->device() != first->device() ||
            reinterpret_cast<uintptr_t>(c->const_data_ptr()) % 4 != 0)
            Py_RETURN_NONE;
        codes[p] = c->const_data_ptr<uint8_t>();
        lookup[p] = l->const_data_ptr<float>();
        shift[p] = s->const_data_ptr<float>();
    }
    const int64_t count = first->numel();
    if (count == 0 || count % 4 || bins < 1 || bins > 256) Py_RETURN_NONE;
    THPObjectPtr list(PyList_New(P));  // (an allocation that throws releases the ones before it)
    if (!list) return nullptr;
    for (Py_ssize_t p = 0; p < P; ++p) {
        at::Tensor o = fresh(THPVariable_Unpack(PyList_GET_ITEM(args[0], p)).sizes(), c10::ScalarType::Float, *first);
        out[p] = o.data_ptr<float>();
        PyList_SET_ITEM(list.get(), p, THPVariable_Wrap(std::move(o)));
    }
    Launch on(*first);
    if (int st = p_tplr_dequantize_lists(codes, static_cast<int>(P), count, lookup, shift, static_cast<int>(bins), out, on.stream()))
        return failed(st, "tplr_dequantize_lists");
    return list.release();
    END_HANDLE_TH_ERRORS
}

// ---- compress ---------------------------------------------------------------------------------
// compress(x, topk, n_bins, range) -> (idx, val, xshape, totalk[, quant_params]); n_bins None: no quantiser
PyObject* compress(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    int64_t topk, bins = 0;
    if (n != 4) return PyErr_SetString(PyExc_TypeError, "compress(x, topk, n_bins, range)"), nullptr;
    const at::Tensor* x = plain_f32(args[0]);
    const bool coded = args[2] != Py_None;
    if (!x || x->numel() == 0 || x->dim() < 1 || x->dim() == 3 || x->dim() > 4 || !to_int(args[1], topk) ||
        (coded && !to_int(args[2], bins)))
        Py_RETURN_NONE;
    const bool chunks = x->dim() == 4;
    const int64_t totalk = chunks ? x->size(2) * x->size(3) : x->size(x->dim() - 1);
    const int64_t k = clamp_k(totalk, topk), rows = x->numel() / totalk;
    if (totalk > TPLR_MAX_ROW || k > totalk) Py_RETURN_NONE;
    const double range = coded ? PyFloat_AsDouble(args[3]) : 0.0;
    if (PyErr_Occurred()) {
        PyErr_Clear();
        Py_RETURN_NONE;
    }
    if (coded && (bins < 1 || bins > 256 || rows * k % 4)) Py_RETURN_NONE;
    // the un-transformed chunk view of a row-major tensor, as encode(use_dct=False) returns it: select straight from it
    const bool view = chunk_view(*x);
    if (view ? k > 128 : !x->is_contiguous()) Py_RETURN_NONE;
    at::Tensor idx = fresh({rows * (k / 2) * 3}, c10::ScalarType::Byte, *x);
    at::Tensor val = chunks ? fresh({x->size(0), x->size(1), k}, c10::ScalarType::Float, *x)
                     : x->dim() == 2 ? fresh({x->size(0), k}, c10::ScalarType::Float, *x)
                                     : fresh({k}, c10::ScalarType::Float, *x);
    Launch on(*x);
    const int st = view ? p_tplr_encode_topk_pack(x->const_data_ptr<float>(), x->size(0) * kEdge, x->size(1) * kEdge, x->stride(2),
                                                  static_cast<int>(k), 0, idx.data_ptr<uint8_t>(), val.data_ptr<float>(), on.stream())
                        : p_tplr_topk_pack(x->const_data_ptr<float>(), rows, totalk, static_cast<int>(k), idx.data_ptr<uint8_t>(),
                                           val.data_ptr<float>(), on.stream());
    if (st) return failed(st, view ? "tplr_encode_topk_pack" : "tplr_topk_pack");
    THPObjectPtr xshape(PyObject_GetAttrString(args[0], "shape"));
    if (!xshape) return nullptr;
    if (!coded)
        return Py_BuildValue("(NNOL)", THPVariable_Wrap(std::move(idx)), THPVariable_Wrap(std::move(val)), xshape.get(),
                             static_cast<long long>(totalk));
    THPObjectPtr q(quantised(val, bins, range, on));
    if (!q) return nullptr;
    return Py_BuildValue("(NOOLO)", THPVariable_Wrap(std::move(idx)), PyTuple_GET_ITEM(q.get(), 0), xshape.get(),
                         static_cast<long long>(totalk), PyTuple_GET_ITEM(q.get(), 1));
    END_HANDLE_TH_ERRORS
}

// ---- decompress, batch_decompress -------------------------------------------------------------
// One parameter's payloads in device memory, found plain; `like` is one of the tensors.
struct Payloads {
    const uint8_t* idx[TPLR_MAX_PEERS];
    const float* val[TPLR_MAX_PEERS];
    int peers;
    int64_t k;
    const at::Tensor* like;
};

// The coefficients chunk after chunk, contiguous on every route: a caller may flatten them in place (view) or hand them
// on as chunks, and what decode(use_dct=False) makes of them is a tensor of its own (a row-major layout would save that
// copy, but share the storage).
at::Tensor chunk_tensor(int64_t Y, int64_t X, const at::Tensor& like) {
    return fresh({Y, X, kEdge, kEdge}, c10::ScalarType::Float, like);
}

// norms (n_norms of them) with scale as scratch, or scale (nullable) the factors themselves
PyObject* scatter_chunks(const Payloads& pl, const float* norms, int64_t n_norms, float* scale, int64_t Y, int64_t X, const Launch& on) {
    at::Tensor out = chunk_tensor(Y, X, *pl.like);
    if (int st = p_tplr_aggregate_param(pl.idx, pl.val, norms, static_cast<int>(n_norms), scale, pl.peers, static_cast<int>(pl.k),
                                        Y * kEdge, X * kEdge, out.data_ptr<float>(), 0, on.stream()))
        return failed(st, "tplr_aggregate_param");
    return THPVariable_Wrap(std::move(out));
}

// aggregate(p, idx list, val list, xshape, block_norms | None, clip): the payloads of P peers on p's device, scatter-mean
// with the clip factors min(1, median / (norm + 1e-8)) of the given norms, or of the values' own -> (Y, X, 64, 64)
// coefficients
PyObject* aggregate(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 6) return PyErr_SetString(PyExc_TypeError, "aggregate(p, idx, val, xshape, norms, clip)"), nullptr;
    const at::Tensor* like = plain_f32(args[0]);
    if (!like || !PyList_Check(args[1]) || !PyList_Check(args[2])) Py_RETURN_NONE;
    int64_t Y, X;
    const Py_ssize_t P = PyList_GET_SIZE(args[2]);
    if (P < 1 || P > TPLR_MAX_PEERS || PyList_GET_SIZE(args[1]) != P || !chunk_shape(args[3], Y, X)) Py_RETURN_NONE;
    const bool clip = args[5] == Py_True;
    Payloads pl;
    pl.peers = static_cast<int>(P);
    pl.k = 0;
    pl.like = like;
    for (Py_ssize_t p = 0; p < P; ++p) {
        const at::Tensor* i = plain(PyList_GET_ITEM(args[1], p), c10::ScalarType::Byte);
        const at::Tensor* v = plain_f32(PyList_GET_ITEM(args[2], p));
        if (!i || !v || i->dim() != 1 || !i->is_contiguous() || !v->is_contiguous() || v->dim() < 1) Py_RETURN_NONE;
        if (p == 0) pl.k = v->size(v->dim() - 1);
        if (pl.k < 2 || pl.k % 2 || pl.k > 4096 || v->size(v->dim() - 1) != pl.k || v->numel() != Y * X * pl.k ||
            i->numel() * 2 != Y * X * pl.k * 3 || v->device() != like->device() || i->device() != like->device())
            Py_RETURN_NONE;
        pl.idx[p] = i->const_data_ptr<uint8_t>();
        pl.val[p] = v->const_data_ptr<float>();
    }
    Launch on(*like);
    at::Tensor scale;
    const float* given = nullptr;
    int64_t n_given = 0;
    if (clip) {
        if (args[4] != Py_None) {
            const at::Tensor* norms = plain_f32(args[4]);
            // (the median is that of every entry given, the factors of the first P are used: :535, :554)
            if (!norms || norms->dim() != 1 || norms->numel() < P || norms->numel() > TPLR_MAX_PEERS || !norms->is_contiguous() ||
                norms->device() != like->device())
                Py_RETURN_NONE;
            n_given = norms->numel();
            given = norms->const_data_ptr<float>();
            scale = fresh({n_given}, c10::ScalarType::Float, *like);
        } else {
            const int64_t count = Y * X * pl.k;
            // about 32 K values per block, so that one large tensor still spreads over the device
            const int64_t slices = count / 32768 < 1 ? 1 : count / 32768 > 256 ? 256 : count / 32768;
            at::Tensor ss = fresh({P, slices}, c10::ScalarType::Float, *like);
            scale = fresh({P}, c10::ScalarType::Float, *like);
            if (int st = p_tplr_peer_sumsq(pl.val, pl.peers, count, static_cast<int>(slices), ss.data_ptr<float>(), on.stream()))
                return failed(st, "tplr_peer_sumsq");
            if (int st = p_tplr_clip_scales(ss.const_data_ptr<float>(), pl.peers, static_cast<int>(slices),
                                            scale.data_ptr<float>(), nullptr, on.stream()))
                return failed(st, "tplr_clip_scales");
        }
    }
    return scatter_chunks(pl, given, n_given, clip ? scale.data_ptr<float>() : nullptr, Y, X, on);
    END_HANDLE_TH_ERRORS
}

// decompress(p, idx, val, xshape, quant_params | None): one payload on p's device, as dense coefficients of xshape.
// None also where an index lies outside its row: the caller finds out which and raises.
PyObject* decompress(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 5) return PyErr_SetString(PyExc_TypeError, "decompress(p, idx, val, xshape, quant_params)"), nullptr;
    const at::Tensor* like = plain_f32(args[0]);
    const at::Tensor* idx = plain(args[1], c10::ScalarType::Byte);
    if (!like || !idx || !idx->is_contiguous() || idx->device() != like->device() || !PyTuple_Check(args[3])) Py_RETURN_NONE;
    const bool coded = args[4] != Py_None;
    const at::Tensor* sent = coded ? plain(args[2], c10::ScalarType::Byte) : plain_f32(args[2]);
    if (!sent || sent->dim() < 1 || sent->numel() == 0 || !sent->is_contiguous() || sent->device() != like->device()) Py_RETURN_NONE;
    const int64_t k = sent->size(sent->dim() - 1), count = sent->numel();
    if (k < 2 || k % 2 || k > 4096 || idx->numel() * 2 != count * 3) Py_RETURN_NONE;
    // the shape: (Y, X, h, w) or rows
    std::vector<int64_t> shape;
    int64_t elements = 1;
    for (Py_ssize_t d = 0; d < PyTuple_GET_SIZE(args[3]); ++d) {
        int64_t s;
        if (!to_int(PyTuple_GET_ITEM(args[3], d), s) || s < 1) Py_RETURN_NONE;
        shape.push_back(s);
        elements *= s;
    }
    if (shape.empty() || shape.size() == 3 || shape.size() > 4) Py_RETURN_NONE;
    const int64_t row_len = shape.size() == 4 ? shape[2] * shape[3] : shape.back();
    const bool chunks = shape.size() == 4 && shape[2] == kEdge && shape[3] == kEdge;
    if (count / k * row_len != elements || row_len > TPLR_MAX_ROW || (!chunks && k > 64)) Py_RETURN_NONE;
    at::Tensor values;
    const float* val = nullptr;
    Launch on(*like);
    if (coded) {
        PyObject* qp = args[4];
        if (!PyTuple_Check(qp) || PyTuple_GET_SIZE(qp) != 5 || PyTuple_GET_ITEM(qp, 4) != float32_dtype || count % 4) Py_RETURN_NONE;
        const at::Tensor* s = plain_f32(PyTuple_GET_ITEM(qp, 0));
        const at::Tensor* l = plain_f32(PyTuple_GET_ITEM(qp, 3));
        if (!s || !l || s->dim() != 0 || l->dim() != 1 || l->numel() < 1 || l->numel() > 256 || !l->is_contiguous() ||
            s->device() != like->device() || l->device() != like->device() ||
            reinterpret_cast<uintptr_t>(sent->const_data_ptr()) % 4 != 0)
            Py_RETURN_NONE;
        if (chunks && k <= 64 && shape[0] * shape[1] <= 0xfffff0) {
            at::Tensor out = chunk_tensor(shape[0], shape[1], *like);
            if (int st = p_tplr_decompress_codes(idx->const_data_ptr<uint8_t>(), sent->const_data_ptr<uint8_t>(),
                                                 l->const_data_ptr<float>(), s->const_data_ptr<float>(), static_cast<int>(l->numel()),
                                                 static_cast<int>(k), shape[0] * kEdge, shape[1] * kEdge, out.data_ptr<float>(), 0,
                                                 on.stream()))
                return failed(st, "tplr_decompress_codes");
            return THPVariable_Wrap(std::move(out));
        }
        values = fresh({count}, c10::ScalarType::Float, *like);
        const uint8_t* codes = sent->const_data_ptr<uint8_t>();
        const float *lookup = l->const_data_ptr<float>(), *shift = s->const_data_ptr<float>();
        float* out = values.data_ptr<float>();
        if (int st = p_tplr_dequantize_lists(&codes, 1, count, &lookup, &shift, static_cast<int>(l->numel()), &out, on.stream()))
            return failed(st, "tplr_dequantize_lists");
        val = out;
    } else {
        val = sent->const_data_ptr<float>();
    }
    if (chunks) {
        Payloads pl;
        pl.peers = 1;
        pl.k = k;
        pl.like = like;
        pl.idx[0] = idx->const_data_ptr<uint8_t>();
        pl.val[0] = val;
        return scatter_chunks(pl, nullptr, 0, nullptr, shape[0], shape[1], on);
    }
    at::Tensor out = fresh(shape, c10::ScalarType::Float, *like);
    // (the reference's scatter raises on an index outside its row as well.)  The check is a launch ahead of the scatter, a
    // workgroup per 32 K entries, and only its words are waited for.
    const int64_t n_words = count >> 15 < 1 ? 1 : count >> 15 > 64 ? 64 : count >> 15;
    at::Tensor seen = at::empty({n_words}, at::TensorOptions().dtype(c10::ScalarType::Int).pinned_memory(true));
    uint32_t* const words = reinterpret_cast<uint32_t*>(seen.data_ptr<int32_t>());
    for (int64_t i = 0; i < n_words; ++i) __atomic_store_n(words + i, kUnset, __ATOMIC_RELAXED);
    if (int st = p_tplr_check_rows(idx->const_data_ptr<uint8_t>(), count / k, static_cast<int>(k), row_len, words,
                                   static_cast<int>(n_words), on.stream()))
        return failed(st, "tplr_check_rows");
    const int st = p_tplr_decompress_rows(idx->const_data_ptr<uint8_t>(), val, count / k, static_cast<int>(k), row_len,
                                          out.data_ptr<float>(), nullptr, on.stream());
    on.wait_for(words, n_words);  // (all of them: the memory is given back behind this)
    bool outside = false;
    for (int64_t i = 0; i < n_words; ++i) outside |= words[i] != 0;
    if (st) return failed(st, "tplr_decompress_rows");
    if (outside) Py_RETURN_NONE;
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

PyMethodDef methods[] = {
    {"bind", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(bind)), METH_FASTCALL, nullptr},
    {"encode", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(encode)), METH_FASTCALL, nullptr},
    {"decode", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(decode)), METH_FASTCALL, nullptr},
    {"compress", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(compress)), METH_FASTCALL, nullptr},
    {"quantize", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(quantize)), METH_FASTCALL, nullptr},
    {"dequantize", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(dequantize)), METH_FASTCALL, nullptr},
    {"aggregate", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(aggregate)), METH_FASTCALL, nullptr},
    {"decompress", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(decompress)), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_native", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__native() { return PyModule_Create(&module); }
