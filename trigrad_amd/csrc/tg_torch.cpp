// tg_torch.cpp -- the call a training loop or a viewer makes for every frame, without the interpreter between its steps.
//
// A small frame is bound by the host: 60 us of kernels, and 165 us of host work per forward and backward pass when the
// checks, the buffers and both halves of the autograd function are Python.  This module is that work in C++: it checks the
// tensors, finds the plan of a frame of this kind, allocates, calls tg_frame_forward, and records an autograd node
// whose backward pass is tg_frame_backward.  What is not the ordinary case is left to the Python route (trigrad_amd._C.frame_forward)
// by returning None: a kind of frame not seen before on this stream, a scene whose number of keys has left the range its
// plan was made for, a wait of the kernels that expired, arguments the checks there have an error for.
//
// Plans are per kind of frame (sizes, options, a rounded number of triangles), frame states (what tg_bin_frame keeps between
// calls) per device and stream; both are made by the Python route, handed over, and bounded in number.
#define PY_SSIZE_T_CLEAN
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_variable.h>

#include <ATen/TensorSubclassLikeUtils.h>
#include <ATen/ops/empty.h>
#include <ATen/ops/zeros_like.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/hip/HIPStream.h>

#include <algorithm>
#include <array>
#include <cstring>
#include <deque>
#include <map>
#include <memory>
#include <mutex>

#include "tg_gradient_copies.hpp"

namespace {

using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

struct Library {
    int (*forward)(tg_frame *) = nullptr;
    int (*backward)(const tg_frame *) = nullptr;
    int (*wait)(const uint32_t *, int, uint32_t, void *) = nullptr;
    void (*force_tickets)(int) = nullptr;
    const char *(*last_error)() = nullptr;
} lib;

void check(int code, const char *what) {
    if (code == 0) return;
    const char *text = lib.last_error();
    throw std::runtime_error(std::string(what) + " failed with code " + std::to_string(code) + ": " + (text ? text : ""));
}

// The part of a call that a plan holds: struct tg_frame from n_vertices on.  The counts come with the frame: a viewer that
// moves through a split scene, or a training loop that adds triangles, has others in every frame.  A plan's sizes are made
// for the number of triangles rounded up (round_count), and no size a frame needs grows when its count gets smaller.  Only triangles
// with two vertices or more each may have records (tg_frame_has_records), which take room: their plans are others.
constexpr size_t kKindBytes = sizeof(tg_frame) - offsetof(tg_frame, n_vertices);
struct Plan {
    std::array<char, kKindBytes> kind;
    int64_t frame_bytes = 0, keys_low = 0, keys_high = 0;  // K outside [low, high]: the next frame's plan is made anew
    void fill(tg_frame &f, int64_t n_vertices, int64_t n_triangles, int64_t max_layers) const {
        std::memset(&f, 0, sizeof f);
        std::memcpy(reinterpret_cast<char *>(&f) + offsetof(tg_frame, n_vertices), kind.data(), kKindBytes);
        f.n_vertices = n_vertices;
        f.n_triangles = n_triangles;
        f.max_layers = max_layers;
    }
};
using PlanKey = std::array<int64_t, 11>;

// As _round_count of the Python side: itself below 32, else up to a multiple of a sixteenth to a thirty-second of itself.
int64_t round_count(int64_t n) {
    int bits = 0;
    for (int64_t m = n; m; m >>= 1) bits++;
    const int64_t step = (int64_t)1 << std::max(bits - 5, 0);
    return std::min<int64_t>((n + step - 1) / step * step, 0x7fffffff);
}

struct State {
    at::Tensor memory;
    int64_t bytes = 0;
    int64_t epoch = 0;
    std::mutex launches;  // one frame at a time on a stream's state
};

// A frame's four words in pinned memory; [2] is the list kernels' status once the blending has begun.
struct Status {
    at::Tensor words;
    uint32_t *at = nullptr;
    void *stream = nullptr;
    int64_t frame = 0;
    std::atomic<bool> checked{false};
    volatile uint32_t &word() const { return const_cast<volatile uint32_t *>(at)[2]; }
    void verify() {
        if (checked) return;
        if (word() == TG_FRAME_PENDING) check(lib.wait(at, 2, TG_FRAME_PENDING, stream), "tg_frame_wait");
        checked = true;
        if (word() == 0) return;
        lib.force_tickets(1);
        throw std::runtime_error("tg_frame_forward: look-back wait timed out (status " + std::to_string(word()) + "); the lists of frame " +
                                 std::to_string(frame) + " are invalid and its image is NaN.  Later frames number their tiles by ticket.");
    }
};

// Never destroyed: the tensors in here must not outlive the runtime that frees them.
struct Registry {
    std::mutex mutex;
    std::map<PlanKey, std::shared_ptr<const Plan>> plans;
    std::map<std::pair<int, void *>, std::shared_ptr<State>> states;
    std::mutex pending_mutex;
    std::deque<std::shared_ptr<Status>> pending;
    int64_t frames = 0;
};
Registry &registry() {
    static Registry *r = new Registry;
    return *r;
}

// Raises if the lists of an earlier frame are invalid; looks at the words that have arrived, or (wait) waits for them.
void verify_pending(bool wait) {
    Registry &r = registry();
    std::lock_guard<std::mutex> lock(r.pending_mutex);
    while (!r.pending.empty()) {
        const std::shared_ptr<Status> s = r.pending.front();
        if (!wait && s->word() == TG_FRAME_PENDING) return;
        r.pending.pop_front();
        s->verify();
    }
}

// The status words of a call that failed: kernels launched before the failure may still write them.
void keep_until_idle(const std::shared_ptr<Status> &status) {
    if (hipStreamSynchronize(static_cast<hipStream_t>(status->stream)) == hipSuccess) return;
    (void)hipGetLastError();
    static auto *kept = new std::deque<std::shared_ptr<Status>>;  // never given back: nobody knows when the kernels end
    static std::mutex mutex;
    std::lock_guard<std::mutex> lock(mutex);
    kept->push_back(status);
}

struct Frame : torch::CustomClassHolder {
    std::shared_ptr<const Plan> plan;
    std::shared_ptr<Status> status;
    at::Tensor image, depthmap, kept;
    int64_t n_keys = 0, max_layers = 0;
};

at::TensorOptions on(const at::Tensor &like, at::ScalarType type) { return at::TensorOptions().device(like.device()).dtype(type); }

// Renders; false: a case for the Python route (nothing is left under way).
bool render(Frame &frame, const std::shared_ptr<State> &state, void *stream, const at::Tensor &vertices, const at::Tensor &indices,
            const at::Tensor &colors, const at::Tensor &opacities) {
    Registry &r = registry();
    tg_frame f;
    frame.plan->fill(f, vertices.size(0), indices.size(0), frame.max_layers);
    frame.image = at::empty({f.height, f.width, 4}, on(vertices, at::kFloat));
    frame.depthmap = at::empty({f.height, f.width}, on(vertices, at::kFloat));
    frame.kept = at::empty({f.kept_bytes}, on(vertices, at::kByte));
    const at::Tensor scratch = at::empty({f.scratch_bytes}, on(vertices, at::kByte));
    auto status = std::make_shared<Status>();
    status->words = at::empty({4}, at::TensorOptions().dtype(at::kInt).pinned_memory(true));
    status->at = static_cast<uint32_t *>(status->words.data_ptr());
    status->stream = stream;
    const at::Tensor v = vertices.contiguous(), i = indices.contiguous(), c = colors.contiguous(), o = opacities.contiguous();
    f.vertices = v.data_ptr<float>();
    f.indices = i.data_ptr<int32_t>();
    f.colors = c.data_ptr<float>();
    f.opacities = o.data_ptr<float>();
    f.image = frame.image.data_ptr<float>();
    f.depthmap = frame.depthmap.data_ptr<float>();
    f.kept = frame.kept.data_ptr();
    f.scratch = scratch.data_ptr();
    f.host = status->at;
    f.stream = stream;
    f.phases = TG_FRAME_BIN | TG_FRAME_LISTS | TG_FRAME_RASTER | TG_FRAME_WAIT;
    {
        std::lock_guard<std::mutex> lock(state->launches);
        f.frame = state->memory.data_ptr();
        f.frame_bytes = state->bytes;
        f.epoch = ++state->epoch;
        if (const int code = lib.forward(&f)) {
            try {
                check(code, "tg_frame_forward");
            } catch (...) {
                // whether the call's scan ran is not known: the digit totals and epochs start anew, as in a fresh state
                state->memory.zero_();
                keep_until_idle(status);
                throw;
            }
        }
    }
    frame.n_keys = f.n_keys;
    if (f.counted != TG_FRAME_COUNTED || f.n_keys > f.key_capacity) {
        // the status words are to stay until the blending has begun
        if (status->word() == TG_FRAME_PENDING) check(lib.wait(status->at, 2, TG_FRAME_PENDING, stream), "tg_frame_wait");
        return false;
    }
    frame.status = status;
    std::lock_guard<std::mutex> lock(r.pending_mutex);
    status->frame = ++r.frames;
    r.pending.push_back(status);
    return true;
}

struct Render : torch::autograd::Function<Render> {
    // the frame is rendered already: a case for the Python route must not leave a node behind
    static variable_list forward(AutogradContext *ctx, const at::Tensor &vertices, const at::Tensor &indices, const at::Tensor &colors,
                                 const at::Tensor &opacities, const c10::intrusive_ptr<Frame> &frame) {
        ctx->set_materialize_grads(false);
        ctx->save_for_backward({vertices, indices, colors, opacities, frame->image, frame->depthmap, frame->kept});
        variable_list out{frame->image, frame->depthmap};
        frame->image.reset();
        frame->depthmap.reset();
        frame->kept.reset();  // released with the node's saved tensors, not with the node
        ctx->saved_data["frame"] = c10::IValue::make_capsule(frame);
        return out;
    }

    static variable_list backward(AutogradContext *ctx, const variable_list &grads) {
        const variable_list saved = ctx->get_saved_variables();
        const auto capsule = ctx->saved_data["frame"].toCapsule();
        const Frame &frame = *static_cast<const Frame *>(capsule.get());
        const at::Tensor v = saved[0].contiguous(), i = saved[1].contiguous(), c = saved[2].contiguous(), o = saved[3].contiguous();
        const c10::DeviceGuard guard(v.device());
        const at::Tensor grad_image = grads[0].defined() ? grads[0].contiguous() : at::zeros_like(saved[4]);
        const at::Tensor grad_depthmap = grads[1].defined() ? grads[1].contiguous() : at::Tensor();
        const int64_t n = v.size(0);
        const at::Tensor gradients = at::empty({8 * n}, on(v, at::kFloat));  // (V,4) | (V,3) | (V,) behind each other
        tg_frame f;
        frame.plan->fill(f, n, i.size(0), frame.max_layers);
        f.n_keys = frame.n_keys;
        const int copies = tg::gradient_copies(f);
        f.phases = TG_FRAME_GRADIENT_COPIES | (int64_t)copies << 16;
        const at::Tensor block = copies ? at::empty({copies * 8 * n}, on(v, at::kFloat)) : gradients;
        f.vertices = v.data_ptr<float>();
        f.indices = i.data_ptr<int32_t>();
        f.colors = c.data_ptr<float>();
        f.opacities = o.data_ptr<float>();
        f.image = saved[4].data_ptr<float>();
        f.depthmap = saved[5].data_ptr<float>();
        f.kept = saved[6].data_ptr();
        f.stream = c10::hip::getCurrentHIPStream(v.device().index()).stream();
        f.grad_image = grad_image.data_ptr<float>();
        f.grad_depthmap = grad_depthmap.defined() ? grad_depthmap.data_ptr<float>() : nullptr;
        f.gradients = gradients.data_ptr<float>();
        f.block = block.data_ptr<float>();
        check(lib.backward(&f), "tg_frame_backward");
        frame.status->verify();  // everything is launched, and the kernels look at the word themselves
        return {gradients.as_strided({n, 4}, {4, 1}, 0), at::Tensor(), gradients.as_strided({n, 3}, {3, 1}, 4 * n),
                gradients.as_strided({n}, {1}, 7 * n), at::Tensor()};
    }
};

PyObject *key_counts = nullptr;  // dict: device index -> K of its last frame

bool fits(const at::Tensor &t, const at::Tensor &with, at::ScalarType type, int64_t rows, int64_t columns) {
    return t.device() == with.device() && t.scalar_type() == type && t.dim() == (columns ? 2 : 1) && t.size(0) == rows &&
           (!columns || t.size(1) == columns);
}

// render(vertices, indices, colors, opacities, width, height, tile_width, tile_height, threshold, record_timing, per_pixel_sort,
// max_layers) -> (image, depthmap), or None for the Python route.
PyObject *py_render(PyObject *, PyObject *const *args, Py_ssize_t n) {
    HANDLE_TH_ERRORS  // torch's own exception types: OutOfMemoryError, and what a saved-tensor hook raised
    if (n != 12) Py_RETURN_NONE;
    for (int k = 0; k < 4; k++)
        if (!THPVariable_Check(args[k])) Py_RETURN_NONE;
    for (int k = 4; k < 8; k++)
        if (!PyLong_CheckExact(args[k])) Py_RETURN_NONE;
    if (!PyFloat_CheckExact(args[8]) || args[9] != Py_False || !PyBool_Check(args[10]) || !PyLong_CheckExact(args[11])) Py_RETURN_NONE;
    const at::Tensor &vertices = THPVariable_Unpack(args[0]), &indices = THPVariable_Unpack(args[1]),
                     &colors = THPVariable_Unpack(args[2]), &opacities = THPVariable_Unpack(args[3]);
    if (!vertices.is_cuda() || vertices.dim() != 2 || indices.dim() != 2) Py_RETURN_NONE;
    // tracing, functorch transforms, dispatch modes, fake tensors and forward-mode tangents: the Python function records or refuses them
    if (c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::Tracer)) Py_RETURN_NONE;
    for (const at::Tensor *t : {&vertices, &indices, &colors, &opacities})
        if (at::isTensorSubclassLike(*t) || t->_fw_grad(0).defined()) Py_RETURN_NONE;
    const int64_t n_vertices = vertices.size(0), n_triangles = indices.size(0);
    if (n_triangles < 1 || !fits(vertices, vertices, at::kFloat, n_vertices, 4) || !fits(indices, vertices, at::kInt, n_triangles, 3) ||
        !fits(colors, vertices, at::kFloat, n_vertices, 3) || !fits(opacities, vertices, at::kFloat, n_vertices, 0))
        Py_RETURN_NONE;
    const bool backward =
        at::GradMode::is_enabled() && (vertices.requires_grad() || colors.requires_grad() || opacities.requires_grad());
    const double threshold = PyFloat_AS_DOUBLE(args[8]);
    int64_t threshold_bits;
    std::memcpy(&threshold_bits, &threshold, sizeof threshold_bits);
    int64_t layers = PyLong_AsLongLong(args[11]);
    if (layers <= 0) layers = n_triangles + 1;  // no limit
    const PlanKey key = {vertices.device().index(), round_count(n_triangles), PyLong_AsLongLong(args[4]), PyLong_AsLongLong(args[5]),
                         PyLong_AsLongLong(args[6]), PyLong_AsLongLong(args[7]), threshold_bits, args[10] == Py_True,
                         layers == n_triangles + 1 ? 0 : layers, backward, n_vertices >= 2 * n_triangles};
    if (PyErr_Occurred()) {  // an integer beyond 64 bits
        PyErr_Clear();
        Py_RETURN_NONE;
    }
    const c10::DeviceGuard guard(vertices.device());
    void *stream = c10::hip::getCurrentHIPStream(vertices.device().index()).stream();
    auto frame = c10::make_intrusive<Frame>();
    frame->max_layers = layers;
    std::shared_ptr<State> state;
    {
        Registry &r = registry();
        std::lock_guard<std::mutex> lock(r.mutex);
        const auto plan = r.plans.find(key);
        const auto found = r.states.find({(int)vertices.device().index(), stream});
        if (plan == r.plans.end() || found == r.states.end()) Py_RETURN_NONE;
        frame->plan = plan->second;
        state = found->second;
    }
    if (state->bytes < frame->plan->frame_bytes || state->epoch >= 0x3FFFFFF0) Py_RETURN_NONE;
    bool rendered;
    variable_list out;
    PyThreadState *unlocked = PyEval_SaveThread();
    try {
        verify_pending(false);
        {
            const at::NoGradGuard no_grad;
            rendered = render(*frame, state, stream, vertices, indices, colors, opacities);
        }
        if (rendered) {
            if (backward)
                out = Render::apply(vertices, indices, colors, opacities, frame);
            else
                out = {frame->image, frame->depthmap};
        }
    } catch (...) {
        PyEval_RestoreThread(unlocked);
        throw;
    }
    PyEval_RestoreThread(unlocked);
    if (!rendered || frame->n_keys < frame->plan->keys_low || frame->n_keys > frame->plan->keys_high) {
        std::lock_guard<std::mutex> lock(registry().mutex);
        registry().plans.erase(key);
    }
    if (!rendered) Py_RETURN_NONE;
    if (key_counts) {
        PyObject *device = PyLong_FromLong(vertices.device().index()), *count = PyLong_FromLongLong(frame->n_keys);
        if (device && count) PyDict_SetItem(key_counts, device, count);
        Py_XDECREF(device);
        Py_XDECREF(count);
    }
    PyObject *result = PyTuple_New(2);
    if (!result) return nullptr;
    PyTuple_SET_ITEM(result, 0, THPVariable_Wrap(std::move(out[0])));
    PyTuple_SET_ITEM(result, 1, THPVariable_Wrap(std::move(out[1])));
    return result;
    END_HANDLE_TH_ERRORS
}

// bind(addresses of tg_frame_forward, tg_frame_backward, tg_frame_wait, tg_force_tickets, tg_last_error; dict of key counts)
PyObject *py_bind(PyObject *, PyObject *args) {
    unsigned long long a[5];
    PyObject *counts;
    if (!PyArg_ParseTuple(args, "KKKKKO!", &a[0], &a[1], &a[2], &a[3], &a[4], &PyDict_Type, &counts)) return nullptr;
    Py_INCREF(counts);
    Py_XDECREF(key_counts);
    key_counts = counts;
    lib.forward = reinterpret_cast<int (*)(tg_frame *)>(a[0]);
    lib.backward = reinterpret_cast<int (*)(const tg_frame *)>(a[1]);
    lib.wait = reinterpret_cast<int (*)(const uint32_t *, int, uint32_t, void *)>(a[2]);
    lib.force_tickets = reinterpret_cast<void (*)(int)>(a[3]);
    lib.last_error = reinterpret_cast<const char *(*)()>(a[4]);
    Py_RETURN_NONE;
}

// remember(key of eleven integers, plan bytes, frame bytes, keys_low, keys_high): a plan for frames of this kind
PyObject *py_remember(PyObject *, PyObject *args) {
    PlanKey key = {};
    long long k[11], frame_bytes, low, high;
    const char *bytes;
    Py_ssize_t size;
    if (!PyArg_ParseTuple(args, "(LLLLLLLLLLL)y#LLL", &k[0], &k[1], &k[2], &k[3], &k[4], &k[5], &k[6], &k[7], &k[8], &k[9], &k[10], &bytes,
                          &size, &frame_bytes, &low, &high))
        return nullptr;
    if ((size_t)size != kKindBytes) {
        PyErr_SetString(PyExc_ValueError, "the plan's constant part has another size");
        return nullptr;
    }
    for (int j = 0; j < 11; j++) key[j] = k[j];
    auto plan = std::make_shared<Plan>();
    std::memcpy(plan->kind.data(), bytes, kKindBytes);
    plan->frame_bytes = frame_bytes;
    plan->keys_low = low;
    plan->keys_high = high;
    std::lock_guard<std::mutex> lock(registry().mutex);
    if (registry().plans.size() >= 256) registry().plans.clear();
    registry().plans[key] = plan;
    Py_RETURN_NONE;
}

// add_state(device index, stream, zeroed byte tensor, usable bytes): frame state for a stream
PyObject *py_add_state(PyObject *, PyObject *args) {
    int device;
    unsigned long long stream;
    PyObject *memory;
    long long bytes;
    if (!PyArg_ParseTuple(args, "iKOL", &device, &stream, &memory, &bytes)) return nullptr;
    if (!THPVariable_Check(memory)) {
        PyErr_SetString(PyExc_TypeError, "the state is a tensor");
        return nullptr;
    }
    auto state = std::make_shared<State>();
    state->memory = THPVariable_Unpack(memory);
    state->bytes = bytes;
    std::lock_guard<std::mutex> lock(registry().mutex);
    if (registry().states.size() >= 256) registry().states.clear();
    registry().states[{device, reinterpret_cast<void *>(stream)}] = state;
    Py_RETURN_NONE;
}

// state_bytes(device index, stream) -> usable bytes of the stream's state with epochs left, 0 without one
PyObject *py_state_bytes(PyObject *, PyObject *args) {
    int device;
    unsigned long long stream;
    if (!PyArg_ParseTuple(args, "iK", &device, &stream)) return nullptr;
    std::lock_guard<std::mutex> lock(registry().mutex);
    const auto found = registry().states.find({device, reinterpret_cast<void *>(stream)});
    return PyLong_FromLongLong(found == registry().states.end() || found->second->epoch >= 0x3FFFFFF0 ? 0 : found->second->bytes);
}

PyObject *py_forget(PyObject *, PyObject *) {
    std::lock_guard<std::mutex> lock(registry().mutex);
    registry().plans.clear();
    Py_RETURN_NONE;
}

PyObject *py_verify(PyObject *, PyObject *wait) {
    HANDLE_TH_ERRORS
    const bool waits = wait == Py_True;
    PyThreadState *unlocked = PyEval_SaveThread();
    try {
        verify_pending(waits);
    } catch (...) {
        PyEval_RestoreThread(unlocked);
        throw;
    }
    PyEval_RestoreThread(unlocked);
    Py_RETURN_NONE;
    END_HANDLE_TH_ERRORS
}

PyMethodDef methods[] = {{"render", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(py_render)), METH_FASTCALL, nullptr},
                         {"bind", py_bind, METH_VARARGS, nullptr},
                         {"remember", py_remember, METH_VARARGS, nullptr},
                         {"add_state", py_add_state, METH_VARARGS, nullptr},
                         {"state_bytes", py_state_bytes, METH_VARARGS, nullptr},
                         {"forget", py_forget, METH_NOARGS, nullptr},
                         {"verify", py_verify, METH_O, nullptr},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "trigrad_torch", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_trigrad_torch() { return PyModule_Create(&module); }
