// Host path of the torch modules in native code: one call per layer forward that checks the
// activations, allocates the output, finds the stream's scratch and launches through the C
// ABI of libexl3_hip.so. The same steps in Python (tensor methods, three size queries and a
// ctypes call with 18 arguments) took 22 us per call, nearly four times the GPU time of a
// small layer (5120 -> 1024, one row: 5.8 us); calls now follow each other at 6.8 us.
//
// The module also owns the scratch buffers and counters of every (device, stream).
// Everything runs under the GIL.
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/PyInterpreter.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/object_ptr.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/TracerMode.h>
#include <ATen/autocast_mode.h>
#include <ATen/core/grad_mode.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>

#include <algorithm>
#include <cstdint>
#include <initializer_list>
#include <map>
#include <memory>
#include <string>
#include <utility>
#include <vector>

#include "../../include/exl3_hip.h"

namespace {

// Raises what ponyexl3_amd._lib.check raises for a status code.
void check_status(int rc, const char* what) {
    if (rc == EXL3_OK) return;
    PyObject* mod = PyImport_ImportModule("ponyexl3_amd._lib");
    PyObject* r = mod ? PyObject_CallMethod(mod, "check", "is", rc, what) : nullptr;
    Py_XDECREF(mod);
    Py_XDECREF(r);
    throw python_error();
}

[[noreturn]] void value_error(const std::string& msg) {
    PyErr_SetString(PyExc_ValueError, msg.c_str());
    throw python_error();
}

const uint16_t* half_ptr(const at::Tensor& t) {
    return t.defined() ? static_cast<const uint16_t*>(t.const_data_ptr()) : nullptr;
}
const int32_t* int_ptr(const at::Tensor& t) {
    return t.defined() ? static_cast<const int32_t*>(t.const_data_ptr()) : nullptr;
}
uint16_t* half_out(const at::Tensor& t) { return static_cast<uint16_t*>(t.mutable_data_ptr()); }

// (kernels that copy 16 bytes at a time)
bool aligned16(std::initializer_list<const at::Tensor*> tensors) {
    uintptr_t bits = 0;
    for (const at::Tensor* t : tensors) bits |= reinterpret_cast<uintptr_t>(t->const_data_ptr());
    return (bits & 15) == 0;
}

at::Tensor tensor_or_none(PyObject* o, const char* name) {
    if (o == Py_None) return {};
    if (!THPVariable_Check(o)) value_error(std::string(name) + " must be a torch.Tensor");
    return THPVariable_Unpack(o);
}

// ---------------------------------------------------------------------------
// Scratch of one (device, stream): launches on one stream are ordered, so they can share
// buffers; two streams of a device running EXL3 layers at the same time must not (the
// counters and partial rows of one launch would be read by the other). A buffer that is
// replaced by a larger one stays allocated: a HIP graph captured earlier still replays
// launches that point into it. Buffers grow by half at least, which bounds what is kept.
struct Scratch {
    at::Tensor buf[3];
    // Counters made while the stream was being captured: the fill that zeroes them is part of that
    // graph and may not have run when another graph or an eager call uses them. Until an eager
    // call has cleared them, every further capture records a fill of its own.
    bool counters_unset = false;
    unsigned long long cleared_in = 0;
};
enum { kWorkspace = 0, kGemmWorkspace = 1, kCounters = 2 };

std::map<std::pair<int, void*>, Scratch>& scratch_map() {
    static auto* m = new std::map<std::pair<int, void*>, Scratch>;  // never destroyed: outlives the HIP runtime
    return *m;
}
std::vector<at::Tensor>& retired() {
    static auto* v = new std::vector<at::Tensor>;
    return *v;
}

struct StreamContext {
    int device;
    void* stream;
    Scratch& scratch;
    explicit StreamContext(int dev)
        : device(dev),
          stream(c10::hip::getCurrentHIPStream(static_cast<c10::DeviceIndex>(dev)).stream()),
          scratch(scratch_map()[{dev, stream}]) {}

    // `n` bytes of scratch, or an int32 array of at least n zeroed when created (the kernels
    // leave it zero)
    const at::Tensor& get(int kind, size_t n) {
        at::Tensor& t = scratch.buf[kind];
        if (!t.defined() || static_cast<size_t>(t.numel()) < n) {
            size_t want = std::max(n, t.defined() ? static_cast<size_t>(t.numel()) * 3 / 2 : 0);
            want = std::max<size_t>(want, kind == kCounters ? 4096 : size_t(1) << 20);
            if (kind == kCounters) want += want & 1;  // whole 64-bit accumulators
            if (t.defined()) retired().push_back(t);
            const auto opt = at::TensorOptions()
                                 .device(at::Device(at::kCUDA, static_cast<c10::DeviceIndex>(device)))
                                 .dtype(kind == kCounters ? at::kInt : at::kByte);
            t = kind == kCounters ? at::zeros({static_cast<int64_t>(want)}, opt)
                                  : at::empty({static_cast<int64_t>(want)}, opt);
            if (kind == kCounters) scratch.counters_unset = capturing(&scratch.cleared_in);
        } else if (kind == kCounters && scratch.counters_unset) {
            unsigned long long id = 0;
            if (!capturing(&id)) {
                t.zero_();
                scratch.counters_unset = false;
            } else if (id != scratch.cleared_in) {
                t.zero_();
                scratch.cleared_in = id;
            }
        }
        return t;
    }

    // whether the stream is being captured, and into which graph
    bool capturing(unsigned long long* id) const {
        hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
        return hipStreamGetCaptureInfo(static_cast<hipStream_t>(stream), &status, id) == hipSuccess &&
               status == hipStreamCaptureStatusActive;
    }
};

// scratch(kind, device index, n) -> tensor of the device's current stream, or None where
// there is none yet and n < 0
PyObject* py_scratch(PyObject*, PyObject* args) {
    HANDLE_TH_ERRORS
    int kind, device;
    long long n;
    if (!PyArg_ParseTuple(args, "iiL", &kind, &device, &n)) throw python_error();
    if (kind < 0 || kind > 2) value_error("unknown scratch kind");
    StreamContext ctx(device);
    if (n < 0) {
        if (!ctx.scratch.buf[kind].defined()) Py_RETURN_NONE;
        return THPVariable_Wrap(ctx.get(kind, 0));
    }
    return THPVariable_Wrap(ctx.get(kind, static_cast<size_t>(n)));
    END_HANDLE_TH_ERRORS
}

// Refuses what a kernel cannot read at a tensor's address; undefined tensors pass.
void require(const at::Tensor& t, const char* name, std::initializer_list<at::ScalarType> types, int64_t numel,
             const at::Tensor& like) {
    if (!t.defined()) return;
    const std::string n(name);
    if (!t.is_cuda()) value_error(n + " must live on the GPU (got device " + t.device().str() + ")");
    if (t.device() != like.device()) value_error(n + " must live on " + like.device().str());
    if (!t.is_contiguous()) value_error(n + " must be contiguous");
    if (std::find(types.begin(), types.end(), t.scalar_type()) == types.end())
        value_error(n + " must not be " + c10::toString(t.scalar_type()));
    if (t.numel() != numel) value_error(n + " has " + std::to_string(t.numel()) + " elements, not " + std::to_string(numel));
}

// ---------------------------------------------------------------------------
// A linear layer or a sibling-fused group.
struct LinearLayer {
    at::Tensor trellis, suh, svh, bias, group_sub, block_sub;
    std::vector<int64_t> member_out;  // out_features of each sibling; empty = one linear
    int k = 0, cb = 0, in_tiles = 0, out_tiles = 0, n_sub = 1;
    int64_t in_features() const { return int64_t(in_tiles) * 16; }
    int64_t out_features() const { return int64_t(out_tiles) * 16; }
};

// x: contiguous fp16 (rows, in) on the layer's device, y: (rows, out)
void linear_run(const LinearLayer& l, const at::Tensor& x, int64_t rows64, const at::Tensor& y, bool fused) {
    if (rows64 == 0) return;
    if (rows64 > INT32_MAX) value_error("too many rows");
    const int rows = static_cast<int>(rows64);
    const int n_in = l.in_tiles * 16, n_out = l.out_tiles * 16;
    const int small_rows = exl3_gemv_max_rows();
    StreamContext ctx(x.device().index());
    const uint16_t* xp = half_ptr(x);
    uint16_t* yp = half_out(y);
    const uint16_t* tr = half_ptr(l.trellis);
    if (l.n_sub > 1 && rows > (fused ? exl3_linear_small_max_rows() : small_rows)) {
        bool one_launch = true;  // members end on 256-column blocks
        int64_t total = 0;
        for (int64_t n : l.member_out) {
            one_launch = one_launch && n % 256 == 0;
            total += n;
        }
        if (l.member_out.size() != static_cast<size_t>(l.n_sub) || total != n_out)
            value_error("member_out must list the out_features of the stacked members");
        const at::Tensor xh = at::empty({rows64, l.n_sub, n_in}, x.options());
        // (not fused: the chain of the separate entry points, bit for bit)
        check_status((fused ? exl3_rotate : exl3_had128_pre)(xp, rows, n_in, half_ptr(l.suh), l.n_sub, half_out(xh),
                                                             ctx.stream),
                     "exl3_rotate");
        // (past exl3_linear_rows()' rows the members of a stack that takes the rows kernel end on 256-column blocks, the ones
        // it was measured against the GEMM with)
        const bool fits = fused && l.group_sub.defined() && exl3_linear_rows_faster(tr, rows, l.in_tiles, l.out_tiles, l.k, l.cb);
        const bool fits_long = fused && l.group_sub.defined() && one_launch &&
                               exl3_linear_rows_long_faster(tr, rows, l.in_tiles, l.out_tiles, l.k, l.cb);
        if (fits || fits_long) {
            const size_t bytes = exl3_linear_rows_workspace_bytes(rows, n_in, n_out);
            void* ws = bytes ? ctx.get(kWorkspace, bytes).mutable_data_ptr() : nullptr;
            check_status((fits ? exl3_linear_rows : exl3_linear_rows_long)(
                             half_ptr(xh), rows, l.n_sub, tr, l.in_tiles, l.out_tiles, l.k, l.cb, int_ptr(l.group_sub),
                             half_ptr(l.svh), half_ptr(l.bias), yp, ws, bytes, ctx.stream),
                         "exl3_linear_rows");
            return;
        }
        if (one_launch) {
            // one GEMM launch over all members, each block reading its member's rotation, then
            // the output transform
            const at::Tensor block_sub =
                l.block_sub.defined() ? l.block_sub : l.group_sub.slice(0, 0, l.group_sub.numel(), 2).contiguous();
            const size_t bytes = exl3_linear_prefill_workspace_bytes(rows, n_in, n_out);
            const at::Tensor& ws = ctx.get(kWorkspace, bytes);
            check_status(exl3_linear_prefill(half_ptr(xh), rows, l.n_sub, tr, l.in_tiles, l.out_tiles, l.k, l.cb,
                                             int_ptr(block_sub), half_ptr(l.svh), half_ptr(l.bias), yp,
                                             ws.mutable_data_ptr(), ws.numel(), ctx.stream),
                         "exl3_linear_prefill");
            return;
        }
        int tn0 = 0;
        for (size_t i = 0; i < l.member_out.size(); i++) {
            if (l.member_out[i] % 128) value_error("member out_features must be multiples of 128");
            const int tn = static_cast<int>(l.member_out[i] / 16);
            const size_t bytes = exl3_gemm_workspace_bytes(rows, l.in_tiles, tn);
            void* ws = bytes ? ctx.get(kGemmWorkspace, bytes).mutable_data_ptr() : nullptr;
            check_status(exl3_gemm(half_ptr(xh) + i * n_in, rows, size_t(l.n_sub) * n_in, tr, l.in_tiles, l.out_tiles,
                                   l.k, l.cb, tn0, tn, yp + size_t(16) * tn0, n_out, ws, bytes, ctx.stream),
                         "exl3_gemm");
            tn0 += tn;
        }
        check_status(exl3_had128_post(yp, 0, 1, size_t(rows) * n_out, rows, n_out, half_ptr(l.svh), half_ptr(l.bias),
                                      yp, ctx.stream),
                     "exl3_had128_post");
        return;
    }
    const size_t bytes = exl3_linear_workspace_bytes(rows, n_in, n_out, l.n_sub);
    const at::Tensor& ws = ctx.get(kWorkspace, bytes);
    int32_t* cnt = nullptr;
    size_t cnt_len = 0;
    if (fused) {
        // one-launch kernel: a 64-bit accumulator per (row, output column) = two ints each;
        // medium-batch kernel: one counter per 128-column group. Two more for the status word.
        const size_t n = rows <= small_rows ? size_t(2) * rows * n_out : n_out / 128;
        const at::Tensor& c = ctx.get(kCounters, n + 2);
        cnt = static_cast<int32_t*>(c.mutable_data_ptr());
        cnt_len = c.numel();
    }
    check_status(exl3_linear_forward(xp, rows, tr, l.in_tiles, l.out_tiles, l.k, l.cb, half_ptr(l.suh), l.n_sub,
                                     int_ptr(l.group_sub), half_ptr(l.svh), half_ptr(l.bias), yp,
                                     ws.mutable_data_ptr(), ws.numel(), cnt, cnt_len, ctx.stream),
                 "exl3_linear_forward");
}

// Activations as the kernels take them: fp16, contiguous, last dimension `features`.
at::Tensor activations(PyObject* arg, int64_t features) {
    if (!THPVariable_Check(arg)) value_error("x must be a torch.Tensor");
    at::Tensor x = THPVariable_Unpack(arg);
    if (x.dim() < 1 || x.size(-1) != features)
        value_error("expected last dim " + std::to_string(features) + ", got " +
                    (x.dim() < 1 ? std::string("a scalar") : std::to_string(x.size(-1))));
    if (!x.is_cuda()) value_error("x must live on the GPU (got device " + x.device().str() + ")");
    if (x.scalar_type() != at::kHalf) x = x.to(at::kHalf);
    return x.is_contiguous() ? x : x.contiguous();
}

struct PyLinear {
    PyObject_HEAD
    LinearLayer* layer;
};

int linear_init(PyObject* self, PyObject* args, PyObject*) {
    try {
        PyObject *trellis, *suh, *svh, *bias, *group_sub, *block_sub, *members;
        int k, cb;
        if (!PyArg_ParseTuple(args, "OiiOOOOOO", &trellis, &k, &cb, &suh, &svh, &bias, &group_sub, &block_sub, &members))
            return -1;
        auto l = std::make_unique<LinearLayer>();
        l->trellis = tensor_or_none(trellis, "trellis");
        if (!l->trellis.defined() || l->trellis.dim() != 3) value_error("trellis must be 3D (in_tiles, out_tiles, 16*K)");
        l->suh = tensor_or_none(suh, "suh");
        l->svh = tensor_or_none(svh, "svh");
        l->bias = tensor_or_none(bias, "bias");
        l->group_sub = tensor_or_none(group_sub, "group_sub");
        l->block_sub = tensor_or_none(block_sub, "block_sub");
        l->k = k;
        l->cb = cb;
        l->in_tiles = static_cast<int>(l->trellis.size(0));
        l->out_tiles = static_cast<int>(l->trellis.size(1));
        l->n_sub = l->suh.defined() && l->suh.dim() == 2 ? static_cast<int>(l->suh.size(0)) : 1;
        if (k < 1 || k > 8 || l->trellis.size(2) != 16 * k) value_error("trellis must be 3D (in_tiles, out_tiles, 16*K)");
        require(l->trellis, "trellis", {at::kShort, at::kUInt16}, l->trellis.numel(), l->trellis);
        require(l->suh, "suh", {at::kHalf}, l->n_sub * l->in_features(), l->trellis);
        require(l->svh, "svh", {at::kHalf}, l->out_features(), l->trellis);
        require(l->bias, "bias", {at::kHalf}, l->out_features(), l->trellis);
        require(l->group_sub, "group_sub", {at::kInt}, l->out_features() / 128, l->trellis);
        require(l->block_sub, "block_sub", {at::kInt}, (l->out_features() + 255) / 256, l->trellis);
        if (members != Py_None) {
            PyObject* seq = PySequence_Fast(members, "member_out must be a sequence");
            if (!seq) return -1;
            for (Py_ssize_t i = 0; i < PySequence_Fast_GET_SIZE(seq); i++)
                l->member_out.push_back(PyLong_AsLongLong(PySequence_Fast_GET_ITEM(seq, i)));
            Py_DECREF(seq);
            if (PyErr_Occurred()) return -1;
        }
        delete reinterpret_cast<PyLinear*>(self)->layer;
        reinterpret_cast<PyLinear*>(self)->layer = l.release();
        return 0;
    } catch (python_error& e) {
        e.restore();
        return -1;
    } catch (const std::exception& e) {
        PyErr_SetString(PyExc_RuntimeError, e.what());
        return -1;
    }
}

void linear_dealloc(PyObject* self) {
    delete reinterpret_cast<PyLinear*>(self)->layer;
    Py_TYPE(self)->tp_free(self);
}

// layer(x): (..., in) -> (..., out) fp16, or for a group a tuple of its members' outputs
// (views of one buffer)
PyObject* linear_call(PyObject* self, PyObject* args, PyObject* kwargs) {
    HANDLE_TH_ERRORS
    const LinearLayer* l = reinterpret_cast<PyLinear*>(self)->layer;
    if (!l || PyTuple_GET_SIZE(args) != 1 || kwargs) value_error("a layer takes one positional argument");
    const at::Tensor x = activations(PyTuple_GET_ITEM(args, 0), l->in_features());
    c10::OptionalDeviceGuard guard(x.device());
    at::DimVector shape(x.sizes());
    shape.back() = l->out_features();
    at::Tensor y = at::empty(shape, x.options());
    linear_run(*l, x, x.numel() / l->in_features(), y, true);
    if (l->member_out.empty()) return THPVariable_Wrap(std::move(y));
    PyObject* out = PyTuple_New(static_cast<Py_ssize_t>(l->member_out.size()));
    if (!out) throw python_error();
    int64_t at_col = 0;
    for (size_t i = 0; i < l->member_out.size(); i++) {
        PyTuple_SET_ITEM(out, static_cast<Py_ssize_t>(i), THPVariable_Wrap(y.narrow(-1, at_col, l->member_out[i])));
        at_col += l->member_out[i];
    }
    return out;
    END_HANDLE_TH_ERRORS
}

// layer.rows(x2d, fused): operator form, x checked by the caller
PyObject* linear_rows(PyObject* self, PyObject* args) {
    HANDLE_TH_ERRORS
    PyObject* x_arg;
    int fused;
    if (!PyArg_ParseTuple(args, "Op", &x_arg, &fused)) throw python_error();
    const LinearLayer* l = reinterpret_cast<PyLinear*>(self)->layer;
    if (!l) value_error("not initialised");
    const at::Tensor x = activations(x_arg, l->in_features());
    c10::OptionalDeviceGuard guard(x.device());
    const int64_t rows = x.numel() / l->in_features();
    at::Tensor y = at::empty({rows, l->out_features()}, x.options());
    linear_run(*l, x, rows, y, fused != 0);
    return THPVariable_Wrap(std::move(y));
    END_HANDLE_TH_ERRORS
}

PyMethodDef linear_methods[] = {{"rows", linear_rows, METH_VARARGS, nullptr}, {nullptr, nullptr, 0, nullptr}};

PyTypeObject linear_type = {PyVarObject_HEAD_INIT(nullptr, 0)};

// ---------------------------------------------------------------------------
// Routed experts of a MoE block (stacked trellises).
struct ExpertStack {
    at::Tensor gu_trellis, gu_suh, gu_svh, dn_trellis, dn_suh, dn_svh;
    int k = 0, cb = 0, activation = 0;
    int experts() const { return static_cast<int>(gu_suh.size(0)); }
    int dim() const { return static_cast<int>(gu_suh.size(2)); }
    int hidden() const { return static_cast<int>(dn_suh.size(1)); }
};

// x (tokens, D) fp16, indices (tokens, top_k) int32, both contiguous -> y: (tokens, top_k, D),
// or with scores (fp16, like indices) the weighted sums (tokens, D).
void experts_run(const ExpertStack& m, const at::Tensor& x, const at::Tensor& indices, const at::Tensor& scores,
                 bool prefill, const at::Tensor& y) {
    const int64_t tokens = indices.size(0), top_k = indices.size(1);
    if (tokens == 0 || top_k == 0) return;
    if (tokens * top_k > INT32_MAX) value_error("too many (token, slot) pairs");
    const int E = m.experts(), D = m.dim(), H = m.hidden(), kk = static_cast<int>(top_k);
    StreamContext ctx(x.device().index());
    // the prefill kernels read everything 16 bytes at a time; the slot kernels take any address
    if (prefill && aligned16({&x, &m.gu_trellis, &m.gu_suh, &m.gu_svh, &m.dn_trellis, &m.dn_suh, &m.dn_svh})) {
        const int t = static_cast<int>(tokens);
        // 4 D + 2 H bytes per (token, slot): up to gigabytes, which go back to the allocator (it
        // hands them out again in the order of this stream) and do not become the stream's scratch
        const at::Tensor ws = at::empty({static_cast<int64_t>(exl3_moe_prefill_workspace_bytes(t, kk, E, D, H))},
                                        x.options().dtype(at::kByte));
        check_status(exl3_moe_prefill(half_ptr(x), t, int_ptr(indices), kk, half_ptr(m.gu_trellis), half_ptr(m.gu_suh),
                                      half_ptr(m.gu_svh), half_ptr(m.dn_trellis), half_ptr(m.dn_suh),
                                      half_ptr(m.dn_svh), E, D, H, m.k, m.cb, m.activation, half_ptr(scores),
                                      half_out(y), ws.mutable_data_ptr(), ws.numel(), ctx.stream),
                     "exl3_moe_prefill");
        return;
    }
    const at::Tensor slots = scores.defined() ? at::empty({tokens, top_k, D}, x.options()) : y;
    const int64_t chunk = std::max<int64_t>(1, 4096 / top_k);
    for (int64_t t0 = 0; t0 < tokens; t0 += chunk) {
        const int t = static_cast<int>(std::min(chunk, tokens - t0));
        const at::Tensor& ws = ctx.get(kWorkspace, exl3_moe_workspace_bytes(t, kk, D, H));
        // counter memory for the gate/up reduction through accumulators; the length tells the
        // library so. Two more ints make the last one the status word.
        const size_t n_cnt = size_t(t) * kk * (size_t(4) * H + D / 128) + 2;
        const at::Tensor& cnt = ctx.get(kCounters, n_cnt);
        check_status(exl3_moe_forward(half_ptr(x) + t0 * D, t, int_ptr(indices) + t0 * top_k, kk,
                                      half_ptr(m.gu_trellis), half_ptr(m.gu_suh), half_ptr(m.gu_svh),
                                      half_ptr(m.dn_trellis), half_ptr(m.dn_suh), half_ptr(m.dn_svh), E, D, H, m.k,
                                      m.cb, m.activation, half_out(slots) + t0 * top_k * D, ws.mutable_data_ptr(),
                                      ws.numel(), static_cast<int32_t*>(cnt.mutable_data_ptr()), n_cnt, ctx.stream),
                     "exl3_moe_forward");
    }
    if (scores.defined())
        check_status(exl3_moe_combine(half_ptr(slots), half_ptr(scores), static_cast<int>(tokens), kk, D, half_out(y),
                                      ctx.stream),
                     "exl3_moe_combine");
}

struct PyExperts {
    PyObject_HEAD
    ExpertStack* stack;
};

int experts_init(PyObject* self, PyObject* args, PyObject*) {
    try {
        PyObject* t[6];
        int k, cb, activation;
        if (!PyArg_ParseTuple(args, "OOOOOOiii", &t[0], &t[1], &t[2], &t[3], &t[4], &t[5], &k, &cb, &activation)) return -1;
        auto m = std::make_unique<ExpertStack>();
        at::Tensor* to[6] = {&m->gu_trellis, &m->gu_suh, &m->gu_svh, &m->dn_trellis, &m->dn_suh, &m->dn_svh};
        for (int i = 0; i < 6; i++) {
            *to[i] = tensor_or_none(t[i], "expert weights");
            if (!to[i]->defined() || !to[i]->is_cuda() || !to[i]->is_contiguous())
                value_error("expert weights must be contiguous tensors on the GPU");
        }
        if (m->gu_suh.dim() != 3 || m->dn_suh.dim() != 2 || k < 1 || k > 8) value_error("expert weights of unexpected shape");
        const int64_t e = m->experts(), d = m->dim(), h = m->hidden();
        require(m->gu_trellis, "gu_trellis", {at::kShort, at::kUInt16}, e * 2 * h * d / 16 * k, m->gu_trellis);
        require(m->dn_trellis, "dn_trellis", {at::kShort, at::kUInt16}, e * h * d / 16 * k, m->gu_trellis);
        require(m->gu_suh, "gu_suh", {at::kHalf}, e * 2 * d, m->gu_trellis);
        require(m->gu_svh, "gu_svh", {at::kHalf}, e * 2 * h, m->gu_trellis);
        require(m->dn_suh, "dn_suh", {at::kHalf}, e * h, m->gu_trellis);
        require(m->dn_svh, "dn_svh", {at::kHalf}, e * d, m->gu_trellis);
        m->k = k;
        m->cb = cb;
        m->activation = activation;
        delete reinterpret_cast<PyExperts*>(self)->stack;
        reinterpret_cast<PyExperts*>(self)->stack = m.release();
        return 0;
    } catch (python_error& e) {
        e.restore();
        return -1;
    } catch (const std::exception& e) {
        PyErr_SetString(PyExc_RuntimeError, e.what());
        return -1;
    }
}

void experts_dealloc(PyObject* self) {
    delete reinterpret_cast<PyExperts*>(self)->stack;
    Py_TYPE(self)->tp_free(self);
}

// experts.slots(x (B, S, D), indices (B, S, top_k), prefill) -> (B, S, top_k, D)
PyObject* experts_slots(PyObject* self, PyObject* args) {
    HANDLE_TH_ERRORS
    PyObject *x_arg, *idx_arg;
    int prefill;
    if (!PyArg_ParseTuple(args, "OOp", &x_arg, &idx_arg, &prefill)) throw python_error();
    const ExpertStack& m = *reinterpret_cast<PyExperts*>(self)->stack;
    const at::Tensor x = activations(x_arg, m.dim());
    c10::OptionalDeviceGuard guard(x.device());
    if (!THPVariable_Check(idx_arg)) value_error("indices must be a torch.Tensor");
    at::Tensor idx = THPVariable_Unpack(idx_arg);
    if (idx.dim() != 3) value_error("indices must be (B, S, top_k)");
    if (!idx.is_cuda()) value_error("indices must live on the GPU (got device " + idx.device().str() + ")");
    const int64_t B = idx.size(0), S = idx.size(1), kk = idx.size(2);
    if (x.numel() != B * S * m.dim()) value_error("x and indices disagree on the number of tokens");
    if (idx.scalar_type() != at::kInt) idx = idx.to(at::kInt);
    idx = idx.reshape({B * S, kk}).contiguous();
    at::Tensor y = at::empty({B, S, kk, m.dim()}, x.options());
    experts_run(m, x, idx, {}, prefill != 0, y);
    return THPVariable_Wrap(std::move(y));
    END_HANDLE_TH_ERRORS
}

// Up to this many tokens the router's product runs in exl3_moe_gate, above it in the gate
// module: its kernel is made for one round trip to memory, not for throughput.
constexpr int64_t kGateMaxTokens = 32;
constexpr int64_t kGateGridTokens = 16 * 65535;

// Router table, experts and weighted sum of a call on the slot kernels: one call, whose tables and slot
// rows lie in the stream's scratch behind the kernels' workspace. x (tokens, D), logits fp16 (tokens,
// n_router) and shared logits or null: device addresses; or w (and w_shared): the gate weights that they
// are computed from. False where the slot kernels do not take the call at once.
bool experts_decode(const ExpertStack& m, StreamContext& ctx, const at::Tensor& x, int64_t tokens, const uint16_t* logits,
                    const uint16_t* shared, const at::Tensor& w, const at::Tensor& w_shared, int64_t n_router, int top_k,
                    bool has_shared, int norm, const at::Tensor& y) {
    const int E = m.experts(), D = m.dim(), H = m.hidden(), kk = top_k + has_shared;
    if (n_router + has_shared > E || n_router > 1024 || (has_shared && n_router != E - 1) || top_k > n_router ||
        tokens * kk > 4096 || !aligned16({&y}))
        return false;
    const int t = static_cast<int>(tokens);
    size_t at = 0;
    auto take = [&at](size_t bytes) {
        const size_t o = at;
        at += (bytes + 255) / 256 * 256;
        return o;
    };
    const size_t ws_bytes = exl3_moe_workspace_bytes(t, kk, D, H);
    const size_t o_ws = take(ws_bytes), o_logits = take(w.defined() ? tokens * (n_router + has_shared) * 2 : 0),
                 o_idx = take(tokens * kk * 4), o_scores = take(tokens * kk * 2), o_rows = take(tokens * kk * D * 2);
    char* base = static_cast<char*>(ctx.get(kWorkspace, at).mutable_data_ptr());
    const size_t n_cnt = exl3_moe_decode_counters(t, kk, D, H);
    const at::Tensor& cnt = ctx.get(kCounters, n_cnt);
    if (w.defined()) {
        uint16_t* out = reinterpret_cast<uint16_t*>(base + o_logits);
        check_status(exl3_moe_gate(half_ptr(x), t, D, half_ptr(w), static_cast<int>(n_router), half_ptr(w_shared), out,
                                   has_shared ? out + tokens * n_router : nullptr, ctx.stream),
                     "exl3_moe_gate");
        logits = out;
        shared = has_shared ? out + tokens * n_router : nullptr;
    }
    check_status(exl3_moe_decode(half_ptr(x), t, logits, shared, static_cast<int>(n_router), top_k, norm,
                                 half_ptr(m.gu_trellis), half_ptr(m.gu_suh), half_ptr(m.gu_svh), half_ptr(m.dn_trellis),
                                 half_ptr(m.dn_suh), half_ptr(m.dn_svh), E, D, H, m.k, m.cb, m.activation,
                                 reinterpret_cast<int32_t*>(base + o_idx), reinterpret_cast<uint16_t*>(base + o_scores),
                                 reinterpret_cast<uint16_t*>(base + o_rows), half_out(y), base + o_ws, ws_bytes,
                                 static_cast<int32_t*>(cnt.mutable_data_ptr()), n_cnt, ctx.stream),
                 "exl3_moe_decode");
    return true;
}

PyObject* import_class(const char* module, const char* name) {
    PyObject* mod = PyImport_ImportModule(module);
    PyObject* cls = mod ? PyObject_GetAttrString(mod, name) : nullptr;
    Py_XDECREF(mod);
    if (!cls) throw python_error();
    return cls;
}
// (no guarded static: an import may hand the GIL to a thread that would wait for the guard with it)
PyObject* linear_module_class() {
    static PyObject* cls = nullptr;
    if (!cls) cls = import_class("torch.nn", "Linear");
    return cls;
}

// Whether something is to see or change the torch operations of a call: function modes (the one
// behind torch.set_default_device only touches factory functions and is no reason), dispatch
// modes, autocast, a function transform, tracing.
bool operations_watched() {
    const int64_t modes = at::impl::PythonTorchFunctionTLS::stack_len();
    for (int64_t i = 0; i < modes; i++) {
        static PyObject* device_mode = nullptr;
        if (!device_mode) device_mode = import_class("torch.utils._device", "DeviceContext");
        PyObject* mode = at::impl::PythonTorchFunctionTLS::get_stack_at(i)->ptr(getPyInterpreter());
        if (reinterpret_cast<PyObject*>(Py_TYPE(mode)) != device_mode) return true;
    }
    return c10::impl::TorchDispatchModeTLS::any_modes_set() || at::autocast::is_autocast_enabled(at::kCUDA) ||
           c10::impl::tls_local_dispatch_key_set().included_.has(c10::DispatchKey::FuncTorchDynamicLayerFrontMode) ||
           at::tracer::impl::is_dispatch_enabled();
}

// A tensor that its memory describes: no subclass (whose data may live elsewhere and whose
// operations may mean something else), no forward-mode tangent, no pending negation.
bool plain_tensor(PyObject* o) {
    if (!THPVariable_CheckExact(o)) return false;
    const at::Tensor& t = THPVariable_Unpack(o);
    return !t._fw_grad(0).defined() && !t.is_neg();
}

// The weight of a plain bias-free fp16 torch.nn.Linear without hooks on the device of `x`, as
// exl3_moe_gate takes it (both 16-byte aligned); undefined if `gate` is anything else.
at::Tensor plain_gate_weight(PyObject* gate, const at::Tensor& x) {
    if (reinterpret_cast<PyObject*>(Py_TYPE(gate)) != linear_module_class()) return {};
    PyObject** dict = _PyObject_GetDictPtr(gate);
    if (!dict || !*dict) return {};
    static PyObject* const hook_names[] = {
        PyUnicode_InternFromString("_forward_hooks"), PyUnicode_InternFromString("_forward_pre_hooks"),
        PyUnicode_InternFromString("_backward_hooks"), PyUnicode_InternFromString("_backward_pre_hooks")};
    static PyObject *const forward_name = PyUnicode_InternFromString("forward"),
                    *const params_name = PyUnicode_InternFromString("_parameters"),
                    *const bias_name = PyUnicode_InternFromString("bias"),
                    *const weight_name = PyUnicode_InternFromString("weight");
    for (PyObject* name : hook_names) {
        PyObject* h = PyDict_GetItem(*dict, name);
        if (!h || PyObject_Size(h) != 0) return {};
    }
    if (PyDict_GetItem(*dict, forward_name)) return {};  // replaced on the instance
    PyObject* params = PyDict_GetItem(*dict, params_name);
    if (!params || !PyDict_Check(params)) return {};
    PyObject* bias = PyDict_GetItem(params, bias_name);
    PyObject* weight = PyDict_GetItem(params, weight_name);
    if ((bias && bias != Py_None) || !weight || !plain_tensor(weight)) return {};
    const at::Tensor& w = THPVariable_Unpack(weight);
    if (w.device() != x.device() || w.scalar_type() != at::kHalf || w.dim() != 2 || w.size(1) != x.size(-1) ||
        !w.is_contiguous() || !aligned16({&w, &x}))
        return {};
    return w;
}

// Whether exl3_moe_route can read what a gate module returned for the tokens of `x`: `width`
// logits per token, or any number if that is 0.
bool usable_logits(PyObject* o, const at::Tensor& x, int64_t width) {
    if (!plain_tensor(o)) return false;
    const at::Tensor& t = THPVariable_Unpack(o);
    return t.device() == x.device() && !t.requires_grad() && t.dim() >= 1 && t.is_contiguous() &&
           (t.scalar_type() == at::kHalf || t.scalar_type() == at::kFloat) &&
           t.numel() == x.numel() / x.size(-1) * (width ? width : t.size(-1));
}

// The tests above as the block applies them, for any device of x.
PyObject* py_operations_watched(PyObject*, PyObject*) {
    HANDLE_TH_ERRORS
    return PyBool_FromLong(operations_watched());
    END_HANDLE_TH_ERRORS
}

PyObject* py_plain_gate_weight(PyObject*, PyObject* args) {
    HANDLE_TH_ERRORS
    PyObject *gate, *x;
    if (!PyArg_ParseTuple(args, "OO", &gate, &x)) throw python_error();
    if (!THPVariable_Check(x)) value_error("x must be a torch.Tensor");
    const at::Tensor w = plain_gate_weight(gate, THPVariable_Unpack(x));
    if (!w.defined()) Py_RETURN_NONE;
    return THPVariable_Wrap(w);
    END_HANDLE_TH_ERRORS
}

PyObject* py_usable_logits(PyObject*, PyObject* args) {
    HANDLE_TH_ERRORS
    PyObject *logits, *x;
    long long width;
    if (!PyArg_ParseTuple(args, "OOL", &logits, &x, &width)) throw python_error();
    if (!THPVariable_Check(x) || THPVariable_Unpack(x).numel() == 0) value_error("x must be a torch.Tensor with elements");
    return PyBool_FromLong(usable_logits(logits, THPVariable_Unpack(x), width));
    END_HANDLE_TH_ERRORS
}

// experts.block(x (..., D), gate, shared gate or None, top_k, norm, prefill) -> (..., D): the
// router (the gates are modules of the caller's; called, or if they are plain Linears and
// there are few tokens, computed here), experts and weighted sum. Where the native route does
// not apply (other types, sizes beyond its kernels, values that carry a gradient or a tangent,
// operations that a mode or transform is to see) it returns
// (logits, shared logits or None) if the gates have been called, None if not.
PyObject* experts_block(PyObject* self, PyObject* args) {
    HANDLE_TH_ERRORS
    PyObject *x_arg, *gate, *shared_gate;
    int top_k, norm, prefill;
    if (!PyArg_ParseTuple(args, "OOOipp", &x_arg, &gate, &shared_gate, &top_k, &norm, &prefill)) throw python_error();
    const ExpertStack& m = *reinterpret_cast<PyExperts*>(self)->stack;
    if (!THPVariable_Check(x_arg) || !plain_tensor(x_arg) || operations_watched()) Py_RETURN_NONE;
    at::Tensor x = THPVariable_Unpack(x_arg);
    const bool has_shared = shared_gate != Py_None;
    const int D = m.dim();
    if (!x.is_cuda() || x.scalar_type() != at::kHalf || x.dim() < 1 || x.size(-1) != D || x.requires_grad() ||
        x.numel() == 0 || top_k < 1 || top_k > 64 || (prefill && m.experts() > 1024))
        Py_RETURN_NONE;
    const int64_t tokens = x.numel() / D;
    c10::OptionalDeviceGuard guard(x.device());
    if (!x.is_contiguous()) x = x.contiguous();
    StreamContext ctx(x.device().index());

    at::Tensor logits, shared, w_shared;  // shared logits, or the weight that the router's kernel takes for them
    const bool grad = at::GradMode::is_enabled();
    if (tokens <= kGateMaxTokens) {
        const at::Tensor w = plain_gate_weight(gate, x);
        const at::Tensor ws = has_shared ? plain_gate_weight(shared_gate, x) : at::Tensor();
        if (w.defined() && !(grad && w.requires_grad()) &&
            (!has_shared || (ws.defined() && ws.size(0) == 1 && !(grad && ws.requires_grad())))) {
            const int64_t E = w.size(0);
            if (!prefill) {
                at::Tensor y = at::empty(x.sizes(), x.options());
                if (experts_decode(m, ctx, x, tokens, nullptr, nullptr, w, ws, E, top_k, has_shared, norm, y))
                    return THPVariable_Wrap(std::move(y));
            }
            const at::Tensor out = at::empty({tokens * (E + has_shared)}, x.options());
            logits = out.narrow(0, 0, tokens * E).view({tokens, E});
            if (has_shared) shared = out.narrow(0, tokens * E, tokens);
            check_status(exl3_moe_gate(half_ptr(x), static_cast<int>(tokens), D, half_ptr(w), static_cast<int>(E),
                                       half_ptr(ws), half_out(logits), has_shared ? half_out(shared) : nullptr,
                                       ctx.stream),
                         "exl3_moe_gate");
        }
    }
    if (!logits.defined()) {
        THPObjectPtr x3(THPVariable_Wrap(x.view({1, tokens, D})));
        THPObjectPtr l(PyObject_CallFunctionObjArgs(gate, x3.get(), nullptr));
        if (!l) throw python_error();
        bool ok = usable_logits(l.get(), x, 0);
        // (a grid of exl3_moe_gate holds kGateGridTokens; more reach the slot kernels where the caller has moved the line)
        if (has_shared && ok && (prefill || tokens <= kGateGridTokens) && THPVariable_Unpack(l.get()).scalar_type() == at::kHalf &&
            THPVariable_Unpack(l.get()).size(-1) == m.experts() - 1 && top_k < m.experts()) {
            w_shared = plain_gate_weight(shared_gate, x);
            if (w_shared.defined() && (w_shared.size(0) != 1 || (grad && w_shared.requires_grad()))) w_shared = at::Tensor();
        }
        THPObjectPtr s;
        if (w_shared.defined() && !prefill) {
            // the slot kernels' router takes logits: one row of the gate's kernel, where the module's product is a library
            // call that takes 2 to 5 us more in front of the experts (55 x 1280 15 us more: block 54.3 -> 38.9)
            shared = at::empty({tokens}, x.options());
            check_status(exl3_moe_gate(half_ptr(x), static_cast<int>(tokens), D, half_ptr(w_shared), 1, nullptr,
                                       half_out(shared), nullptr, ctx.stream),
                         "exl3_moe_gate");
            w_shared = at::Tensor();
        } else if (has_shared && !w_shared.defined()) {
            s = THPObjectPtr(PyObject_CallFunctionObjArgs(shared_gate, x3.get(), nullptr));
            if (!s) throw python_error();
        }
        ok = ok && (!s || (usable_logits(s.get(), x, 1) && THPVariable_Unpack(s.get()).scalar_type() ==
                                                                             THPVariable_Unpack(l.get()).scalar_type()));
        if (!ok) return PyTuple_Pack(2, l.get(), has_shared ? s.get() : Py_None);
        logits = THPVariable_Unpack(l.get());
        if (s) shared = THPVariable_Unpack(s.get());
    }
    const int64_t n_experts = logits.size(-1);
    if (n_experts + has_shared > m.experts() || n_experts > 1024 || (has_shared && n_experts != m.experts() - 1) ||
        top_k > n_experts) {
        THPObjectPtr l(THPVariable_Wrap(logits.view({1, tokens, n_experts})));
        THPObjectPtr s(has_shared ? THPVariable_Wrap(shared.view({1, tokens, 1})) : Py_NewRef(Py_None));
        return PyTuple_Pack(2, l.get(), s.get());
    }
    at::Tensor y = at::empty(x.sizes(), x.options());
    if (!prefill && logits.scalar_type() == at::kHalf &&
        experts_decode(m, ctx, x, tokens, half_ptr(logits), half_ptr(shared), {}, {}, n_experts, top_k, has_shared, norm, y))
        return THPVariable_Wrap(std::move(y));
    const int64_t kk = top_k + has_shared;
    // indices and scores in one allocation
    const at::Tensor routing = at::empty({tokens * kk * 6}, x.options().dtype(at::kByte));
    const at::Tensor idx = routing.narrow(0, 0, tokens * kk * 4).view(at::kInt).view({tokens, kk});
    const at::Tensor scores = routing.narrow(0, tokens * kk * 4, tokens * kk * 2).view(at::kHalf).view({tokens, kk});
    if (w_shared.defined())
        check_status(exl3_moe_route_shared(half_ptr(logits), half_ptr(x), D, half_ptr(w_shared), static_cast<int>(tokens),
                                           static_cast<int>(n_experts), top_k, norm,
                                           static_cast<int32_t*>(idx.mutable_data_ptr()), half_out(scores), ctx.stream),
                     "exl3_moe_route_shared");
    else
        check_status(exl3_moe_route(logits.const_data_ptr(), logits.scalar_type() == at::kFloat,
                                    has_shared ? shared.const_data_ptr() : nullptr, static_cast<int>(tokens),
                                    static_cast<int>(n_experts), top_k, norm,
                                    static_cast<int32_t*>(idx.mutable_data_ptr()), half_out(scores), ctx.stream),
                     "exl3_moe_route");
    experts_run(m, x, idx, scores, prefill != 0, y);
    return THPVariable_Wrap(std::move(y));
    END_HANDLE_TH_ERRORS
}

PyMethodDef experts_methods[] = {{"slots", experts_slots, METH_VARARGS, nullptr},
                                 {"block", experts_block, METH_VARARGS, nullptr},
                                 {nullptr, nullptr, 0, nullptr}};

PyTypeObject experts_type = {PyVarObject_HEAD_INIT(nullptr, 0)};

// A tensor argument as the operators of ponyexl3_amd.ops take it (their messages).
at::Tensor operand(PyObject* o, const char* name, std::initializer_list<at::ScalarType> types, const char* type_name) {
    const std::string n(name);
    if (!THPVariable_Check(o)) value_error(n + " must be a torch.Tensor");
    const at::Tensor& t = THPVariable_Unpack(o);
    if (!t.is_cuda()) value_error(n + " must live on the GPU (got device " + t.device().str() + ")");
    if (!t.is_contiguous()) value_error(n + " must be contiguous");
    if (std::find(types.begin(), types.end(), t.scalar_type()) == types.end())
        value_error(n + " must be " + type_name + ", got " + c10::toString(t.scalar_type()));
    return t;
}

// public_weight(trellis, K, codebook, suh or None, svh or None, first tile column, tile columns or -1 for the
// rest, transposed) -> (in, 16 n) or transposed, fp16. 11 us of host time per call in Python.
PyObject* py_public_weight(PyObject*, PyObject* args) {
    HANDLE_TH_ERRORS
    PyObject *trellis_arg, *suh_arg, *svh_arg;
    int k, cb, tn_offset, tn_count, transposed;
    if (!PyArg_ParseTuple(args, "OiiOOiip", &trellis_arg, &k, &cb, &suh_arg, &svh_arg, &tn_offset, &tn_count, &transposed))
        throw python_error();
    const at::Tensor trellis = operand(trellis_arg, "trellis", {at::kShort, at::kUInt16}, "a 16-bit integer tensor");
    if (trellis.dim() != 3) value_error("trellis must be 3D (in_tiles, out_tiles, 16*K)");
    if (k < 1 || k > 8) value_error("K must be in [1, 8], got " + std::to_string(k));
    if (trellis.size(2) != 16 * k)
        value_error("packed size " + std::to_string(trellis.size(2)) + " != expected " + std::to_string(16 * k) + " for K=" +
                    std::to_string(k));
    const int in_tiles = static_cast<int>(trellis.size(0)), out_tiles = static_cast<int>(trellis.size(1));
    if (tn_count == -1) tn_count = out_tiles - tn_offset;
    if (tn_offset < 0 || tn_count < 0 || int64_t(tn_offset) + tn_count > out_tiles) value_error("slice exceeds output features");
    const int64_t n_in = int64_t(in_tiles) * 16, n_out = int64_t(tn_count) * 16;
    if (n_in % 128 || n_out % 128)
        value_error("in/out features must be multiples of 128 for the Hadamard transform");
    at::Tensor scale[2];
    for (int i = 0; i < 2; i++) {
        PyObject* o = i ? svh_arg : suh_arg;
        if (o == Py_None) continue;
        const char* name = i ? "svh" : "suh";
        scale[i] = operand(o, name, {at::kHalf}, "float16");
        if (scale[i].numel() != (i ? n_out : n_in)) value_error(std::string(name) + " length does not match the feature dim");
    }
    c10::OptionalDeviceGuard guard(trellis.device());
    at::Tensor w = transposed ? at::empty({n_out, n_in}, trellis.options().dtype(at::kHalf))
                              : at::empty({n_in, n_out}, trellis.options().dtype(at::kHalf));
    if (w.numel()) {
        void* stream = c10::hip::getCurrentHIPStream(trellis.device().index()).stream();
        check_status(exl3_public_weight(half_ptr(trellis), in_tiles, out_tiles, k, cb, half_ptr(scale[0]), half_ptr(scale[1]),
                                        tn_offset, tn_count, transposed, half_out(w), stream),
                     "exl3_public_weight");
    }
    return THPVariable_Wrap(std::move(w));
    END_HANDLE_TH_ERRORS
}

PyMethodDef module_methods[] = {{"public_weight", py_public_weight, METH_VARARGS, nullptr},
                                {"scratch", py_scratch, METH_VARARGS, nullptr},
                                {"plain_gate_weight", py_plain_gate_weight, METH_VARARGS, nullptr},
                                {"operations_watched", py_operations_watched, METH_NOARGS, nullptr},
                                {"usable_logits", py_usable_logits, METH_VARARGS, nullptr},
                                {nullptr, nullptr, 0, nullptr}};

PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "_exl3_host", nullptr, -1, module_methods};

}  // namespace

PyMODINIT_FUNC PyInit__exl3_host() {
    linear_type.tp_name = "ponyexl3_amd._exl3_host.Linear";
    linear_type.tp_basicsize = sizeof(PyLinear);
    linear_type.tp_flags = Py_TPFLAGS_DEFAULT;
    linear_type.tp_new = PyType_GenericNew;
    linear_type.tp_init = linear_init;
    linear_type.tp_dealloc = linear_dealloc;
    linear_type.tp_call = linear_call;
    linear_type.tp_methods = linear_methods;
    experts_type.tp_name = "ponyexl3_amd._exl3_host.Experts";
    experts_type.tp_basicsize = sizeof(PyExperts);
    experts_type.tp_flags = Py_TPFLAGS_DEFAULT;
    experts_type.tp_new = PyType_GenericNew;
    experts_type.tp_init = experts_init;
    experts_type.tp_dealloc = experts_dealloc;
    experts_type.tp_methods = experts_methods;
    if (PyType_Ready(&linear_type) < 0 || PyType_Ready(&experts_type) < 0) return nullptr;
    PyObject* m = PyModule_Create(&module_def);
    if (!m) return nullptr;
    Py_INCREF(&linear_type);
    if (PyModule_AddObject(m, "Linear", reinterpret_cast<PyObject*>(&linear_type)) < 0) return nullptr;
    Py_INCREF(&experts_type);
    if (PyModule_AddObject(m, "Experts", reinterpret_cast<PyObject*>(&experts_type)) < 0) return nullptr;
    return m;
}
