// Host glue of TrainableCQT for the common case: the autograd node, the block
// views and the launch of one direction in one C++ call (host code only; the
// kernels are libflashcqt.so's, reached through the C ABI function pointers that
// Python passes in). A training step on 16 slices spends 75 us on the GPU and
// spent 225 us on the host, most of it in Python: the view per block, the
// autograd Functions and the GIL hand-overs of the backward pass. fwd and bwd
// return None for every call that is not plain (another device or type, tensor
// subclasses, function or dispatch modes, functorch, tracing, forward-mode
// tangents, stream capture, a workspace that has to grow); trainable.py's own
// path, which has the same results, then takes it.
#include <atomic>
#include <mutex>
#include <string>
#include <vector>

#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPGraphsC10Utils.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/extension.h>

#include "../../include/flashcqt.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

struct Group {
    int64_t bands, M, off;
};

struct Engine : torch::CustomClassHolder {
    // tables (device pointers into table_mem), C ABI entry points, layout
    fcqt_tables tab;
    const int32_t *route, *route_b, *scat, *scat_a, *ovf, *ovf_a;
    decltype(&fcqt_analysis) analysis_fn;
    decltype(&fcqt_synthesis) synthesis_fn;
    Tensor table_mem;
    c10::Device device{c10::kCUDA, 0};
    std::vector<Group> groups;
    int64_t octave_groups = 0;

    // the engine's current buffer set (leading rows serve any smaller batch);
    // Python publishes every change, so nothing here outlives a replaced set
    std::mutex mu;
    // a direction's launches stay together: they share the set (Python holds it too,
    // as a context manager, around the launches of the calls that fwd and bwd decline)
    std::mutex launching;
    int64_t rows = 0;
    Tensor X, W, F, FA;
    std::atomic<bool> captured{false};

    // adjoint: with FA, which the gradient of an analysis scatters into (a
    // synthesis and its gradient use X, W and F alone)
    bool ready(int64_t batch, bool adjoint) {
        std::lock_guard<std::mutex> lock(mu);
        return rows >= batch && (!adjoint || FA.defined());
    }
    // X and W, or a scatter buffer and W, of at least `batch` rows: the engine's
    // own, or buffers of this call when the set is gone or too small (a backward
    // pass after the engine released it)
    void buffers(int64_t batch, Tensor Engine::*which, int64_t row, Tensor& a, Tensor& w) {
        if (c10::hip::currentStreamCaptureStatusMayInitCtx() != c10::hip::CaptureStatus::None) captured = true;
        {
            std::lock_guard<std::mutex> lock(mu);
            if (rows >= batch && (this->*which).defined()) {
                a = this->*which;
                w = W;
                return;
            }
        }
        const auto opt = table_mem.options().dtype(at::kFloat);
        a = which == &Engine::X ? at::empty({batch, row, 2}, opt) : at::zeros({batch, row, 2}, opt);
        w = at::empty({batch, FCQT_L, 2}, opt);
    }
};

using Ref = c10::intrusive_ptr<Engine>;

// Raise flash_cqt._native.NativeError from any thread.
[[noreturn]] void raise_native(int status, const char* what) {
    py::gil_scoped_acquire gil;
    try {
        py::module_::import("flash_cqt._native").attr("check")(status, what);
    } catch (py::error_already_set& e) {
        e.restore();
    }
    python_error err;
    err.persist();
    throw std::move(err);
}

hipStream_t launch_stream(const Engine& e) {
    if (c10::hip::current_device() != e.device.index()) {
        // the same error as the Python path
        py::gil_scoped_acquire gil;
        try {
            py::module_::import("flash_cqt._native").attr("stream_handle")(e.device.index());
        } catch (py::error_already_set& err) {
            err.restore();
        }
        python_error err;
        err.persist();
        throw std::move(err);
    }
    return c10::hip::getCurrentHIPStream(e.device.index()).stream();
}

// x [B, N] fp32 -> [B, ncoef] complex64
Tensor analysis(Engine& e, const Tensor& x, const int32_t* table) {
    const int64_t batch = x.size(0);
    const hipStream_t stream = launch_stream(e);
    Tensor xs, w;
    e.buffers(batch, &Engine::X, FCQT_XSTRIDE, xs, w);
    Tensor kc = at::empty({batch, e.tab.ncoef}, x.options().dtype(at::kComplexFloat));
    std::unique_lock<std::mutex> lock(e.launching);
    const int s = e.analysis_fn(&e.tab, table, x.data_ptr<float>(), static_cast<float*>(kc.data_ptr()), nullptr,
                                FCQT_INTERLEAVED, xs.data_ptr<float>(), w.data_ptr<float>(), batch, stream);
    lock.unlock();
    if (s) raise_native(s, "analysis");
    return kc;
}

// kc [B, ncoef] complex64 -> [B, N] fp32
Tensor synthesis(Engine& e, const Tensor& kc, const int32_t* table, const int32_t* ovf, Tensor Engine::*fbuf) {
    const int64_t batch = kc.size(0);
    const hipStream_t stream = launch_stream(e);
    Tensor f, w;
    e.buffers(batch, fbuf, FCQT_FROW, f, w);
    Tensor y = at::empty({batch, FCQT_N}, kc.options().dtype(at::kFloat));
    std::unique_lock<std::mutex> lock(e.launching);
    const int s = e.synthesis_fn(&e.tab, table, ovf, static_cast<const float*>(kc.data_ptr()), nullptr,
                                 FCQT_INTERLEAVED, f.data_ptr<float>(), w.data_ptr<float>(), y.data_ptr<float>(),
                                 batch, stream);
    lock.unlock();
    if (s) raise_native(s, "synthesis");
    return y;
}

Ref engine_of(AutogradContext* ctx) {
    return c10::static_intrusive_pointer_cast<Engine>(ctx->saved_data["engine"].toCapsule());
}

struct Analysis : torch::autograd::Function<Analysis> {
    static Tensor forward(AutogradContext* ctx, const Tensor& x, const Ref& e) {
        ctx->saved_data["engine"] = c10::IValue::make_capsule(e);
        return analysis(*e, x, e->route);
    }
    static variable_list backward(AutogradContext* ctx, const variable_list& g) {
        const Ref e = engine_of(ctx);
        const Tensor gk = g[0].to(at::kComplexFloat).resolve_conj().contiguous();
        return {synthesis(*e, gk, e->scat_a, e->ovf_a, &Engine::FA), Tensor()};
    }
};

struct Synthesis : torch::autograd::Function<Synthesis> {
    static Tensor forward(AutogradContext* ctx, const Tensor& kc, const Ref& e) {
        ctx->saved_data["engine"] = c10::IValue::make_capsule(e);
        return synthesis(*e, kc, e->scat, e->ovf, &Engine::F);
    }
    static variable_list backward(AutogradContext* ctx, const variable_list& g) {
        const Ref e = engine_of(ctx);
        const Tensor gy = g[0].to(at::kFloat).resolve_neg().contiguous();
        return {analysis(*e, gy, e->route_b), Tensor()};
    }
};

// A call under none of the modes that want to see its operations.
bool plain_call() {
    return !c10::impl::TorchDispatchModeTLS::any_modes_set() && !at::impl::torch_function_mode_enabled() &&
           !torch::jit::tracer::isTracing() &&
           !c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode) &&
           !c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::Functionalize) &&
           c10::hip::currentStreamCaptureStatusMayInitCtx() == c10::hip::CaptureStatus::None;
}

// No subclass, wrapper, lazy conjugation or negation: its values are its memory.
bool own_values(const Tensor& t) {
    static const c10::DispatchKeySet odd({c10::DispatchKey::Python, c10::DispatchKey::FuncTorchBatched,
                                          c10::DispatchKey::FuncTorchGradWrapper, c10::DispatchKey::Functionalize,
                                          c10::DispatchKey::Conjugate, c10::DispatchKey::Negative,
                                          c10::DispatchKey::ZeroTensor});
    return t.defined() && !t.key_set().has_any(odd) && t.layout() == c10::kStrided;
}

// A strided tensor of the given GPU and type with values of its own, no tangent.
bool plain_tensor(const c10::Device& device, const Tensor& t, at::ScalarType type) {
    return own_values(t) && t.device() == device && t.scalar_type() == type && !t._fw_grad(0).defined();
}

// (octave blocks, side blocks) of x [..., N], or None
py::object fwd(const Ref& e, const Tensor& x) {
    if (!plain_call() || !plain_tensor(e->device, x, at::kFloat)) return py::none();
    const int64_t dim = x.dim();
    if (dim < 1 || x.size(-1) != FCQT_N || x.numel() == 0 || !x.is_contiguous()) return py::none();
    const bool grad = x.requires_grad() && at::GradMode::is_enabled();
    if (!e->ready(x.numel() / FCQT_N, grad)) return py::none();
    std::vector<Tensor> blocks, side;
    {
        py::gil_scoped_release nogil;
        const Tensor kc = Analysis::apply(dim == 2 ? x : x.view({-1, FCQT_N}), e);
        std::vector<int64_t> shape(x.sizes().begin(), x.sizes().end() - 1);
        shape.resize(dim + 1);
        for (size_t i = 0; i < e->groups.size(); ++i) {
            const Group& g = e->groups[i];
            shape[dim - 1] = g.bands;
            shape[dim] = g.M;
            // one narrow per group: single views, which autograd lets a caller modify in place
            ((int64_t)i < e->octave_groups ? blocks : side).push_back(kc.narrow(1, g.off, g.bands * g.M).view(shape));
        }
    }
    return py::make_tuple(blocks, side);
}

// The [B, ncoef] buffer whose consecutive group views the parts are, else an undefined tensor.
// A part that is a leaf of its own, that keeps its gradient or has hooks on it, or whose gradient is
// wanted where the buffer's is not, is no such view: its gradient would go past it.
Tensor base_of(const Engine& e, const std::vector<Tensor>& parts, int64_t batch) {
    if (!parts[0].is_view()) return {};
    const Tensor base(parts[0]._base());
    if (base.device() != e.device || base.scalar_type() != at::kComplexFloat || base.dim() != 2 ||
        base.size(0) != batch || base.size(1) != e.tab.ncoef || !base.is_contiguous() ||
        base.key_set().has(c10::DispatchKey::Conjugate))
        return {};
    const auto* ptr = static_cast<const char*>(base.data_ptr());
    const bool grad = at::GradMode::is_enabled();
    for (size_t i = 0; i < parts.size(); ++i) {
        const Tensor& c = parts[i];
        const Group& g = e.groups[i];
        if (grad && (c.requires_grad() != base.requires_grad() ||
                     (c.requires_grad() &&
                      (c.is_leaf() || c.retains_grad() || !torch::autograd::impl::hooks(c).empty()))))
            return {};
        if (!c.is_view() || !c._base().is_same(base) || static_cast<const char*>(c.data_ptr()) != ptr + 8 * g.off)
            return {};
        int64_t want = e.tab.ncoef;                    // strides of the leading dimensions, last first
        for (int64_t d = c.dim() - 3; d >= 0; --d) {
            if (c.size(d) != 1 && c.stride(d) != want) return {};
            want *= c.size(d);
        }
        if (c.stride(-1) != 1 || (g.bands != 1 && c.stride(-2) != g.M)) return {};
    }
    return base;
}

// The flat SlicedCQT coefficient buffer of `rows` slices that the parts are all
// the blocks of, in order, as its fwd returned them, or None.
py::object block_base(const Ref& e, const std::vector<Tensor>& parts, int64_t rows) {
    if (parts.size() != e->groups.size() || !own_values(parts[0]) || !parts[0].is_view()) return py::none();
    const Tensor base(parts[0]._base());
    if (!own_values(base) || base.device() != e->device || base.scalar_type() != at::kComplexFloat || base.dim() != 1 ||
        base.numel() != rows * e->tab.ncoef || !base.is_contiguous())
        return py::none();
    const auto* ptr = static_cast<const char*>(base.data_ptr());
    for (size_t i = 0; i < parts.size(); ++i) {
        const Tensor& c = parts[i];
        const Group& g = e->groups[i];
        if (!own_values(c) || !c.is_view() || !c._base().is_same(base) || !c.is_contiguous() ||
            c.numel() != rows * g.bands * g.M || static_cast<const char*>(c.data_ptr()) != ptr + 8 * rows * g.off)
            return py::none();
    }
    return py::cast(base);
}

// y [..., N] of the blocks, or None
py::object bwd(const Ref& e, const std::vector<Tensor>& parts) {
    if (!plain_call() || parts.size() != e->groups.size()) return py::none();
    const int64_t dim = parts[0].defined() ? parts[0].dim() : 0;
    if (dim < 2) return py::none();
    const auto lead = parts[0].sizes().slice(0, dim - 2);
    int64_t batch = 1;
    for (int64_t d : lead) batch *= d;
    for (size_t i = 0; i < parts.size(); ++i) {
        const Tensor& c = parts[i];
        if (!plain_tensor(e->device, c, at::kComplexFloat) || c.dim() != dim || c.sizes().slice(0, dim - 2) != lead ||
            c.size(-2) != e->groups[i].bands || c.size(-1) != e->groups[i].M)
            return py::none();
    }
    if (batch < 1 || !e->ready(batch, false)) return py::none();
    Tensor y;
    {
        py::gil_scoped_release nogil;
        Tensor flat = base_of(*e, parts, batch);
        if (!flat.defined()) {
            std::vector<Tensor> rows;
            for (const Tensor& c : parts) rows.push_back(c.reshape({batch, -1}));
            flat = at::cat(rows, -1);
        }
        y = Synthesis::apply(flat, e);
        if (lead.size() != 1) {
            std::vector<int64_t> shape(lead.begin(), lead.end());
            shape.push_back(FCQT_N);
            y = y.view(shape);
        }
    }
    return py::cast(y);
}

// A Python error raised below, as pybind11 passes it on.
template <typename F, typename... A>
py::object guarded(F f, const A&... a) {
    try {
        return f(a...);
    } catch (python_error& e) {
        e.restore();
        throw py::error_already_set();
    }
}

// Copies of the tensors (t.clone() each) with one launch of fcqt_copy_buffers, or
// None where one of them is not a plain dense tensor of the current GPU or they
// pass that launch's 64 GiB.
py::object clones(const std::vector<Tensor>& ts, int64_t copy_fn) {
    if (ts.empty() || ts.size() > FCQT_COPY_MAX || !plain_call()) return py::none();
    const c10::Device device(c10::kCUDA, c10::hip::current_device());
    const void* src[FCQT_COPY_MAX];
    void* dst[FCQT_COPY_MAX];
    int64_t bytes[FCQT_COPY_MAX];
    size_t total = 0;
    for (const Tensor& t : ts) {
        if (!plain_tensor(device, t, t.scalar_type()) || !t.is_non_overlapping_and_dense() || t.numel() == 0)
            return py::none();
        total += t.nbytes() + FCQT_COPY_SHARE;         // a buffer's last workgroup may be short
    }
    if (total > FCQT_COPY_BYTES) return py::none();
    std::vector<Tensor> out;
    for (size_t i = 0; i < ts.size(); ++i) {
        out.push_back(at::empty_like(ts[i]));
        src[i] = ts[i].data_ptr();
        dst[i] = out[i].data_ptr();
        bytes[i] = (int64_t)ts[i].nbytes();
    }
    if (int s = reinterpret_cast<decltype(&fcqt_copy_buffers)>(copy_fn)(
            src, dst, bytes, (int)ts.size(), c10::hip::getCurrentHIPStream(device.index()).stream()))
        raise_native(s, "copy_buffers");
    return py::cast(out);
}

const void* address(int64_t p) { return reinterpret_cast<const void*>(p); }

}  // namespace

PYBIND11_MODULE(_fcqt_torch, m) {
    // what the loader compares with the library and the running torch
    m.attr("abi_version") = FCQT_ABI_VERSION;
    m.attr("torch_version") = FCQT_TORCH_VERSION;
    m.def("clones", [](const std::vector<Tensor>& ts, int64_t copy_fn) { return guarded(clones, ts, copy_fn); });
    // [t.as_strided(size, stride, offset) for size, stride, offset in args]
    m.def("strided_views", [](const Tensor& t, const std::vector<std::tuple<std::vector<int64_t>, std::vector<int64_t>,
                                                                            int64_t>>& args) {
        std::vector<Tensor> out;
        for (const auto& a : args) out.push_back(t.as_strided(std::get<0>(a), std::get<1>(a), std::get<2>(a)));
        return out;
    });
    py::class_<Engine, Ref>(m, "Engine")
        .def(py::init([](const std::vector<int64_t>& tables, int64_t ntasks, int64_t ncoef, int64_t coef_span,
                         int64_t analysis_fn, int64_t synthesis_fn, const Tensor& table_mem,
                         const std::vector<std::vector<int64_t>>& groups, int64_t octave_groups) {
            TORCH_CHECK(tables.size() == 10 && table_mem.is_cuda(), "flash_cqt engine tables");
            Ref e = c10::make_intrusive<Engine>();
            e->tab.tw_pass = static_cast<const float*>(address(tables[0]));
            e->tab.tw_half = static_cast<const float*>(address(tables[1]));
            e->tab.tw_stage = static_cast<const float*>(address(tables[2]));
            e->tab.tasks = static_cast<const int32_t*>(address(tables[3]));
            e->tab.ntasks = (int32_t)ntasks;
            e->tab.ncoef = ncoef;
            e->tab.coef_span = coef_span;
            const int32_t** rec[] = {&e->route, &e->route_b, &e->scat, &e->scat_a, &e->ovf, &e->ovf_a};
            for (int i = 0; i < 6; ++i) *rec[i] = static_cast<const int32_t*>(address(tables[4 + i]));
            e->analysis_fn = reinterpret_cast<decltype(&fcqt_analysis)>(analysis_fn);
            e->synthesis_fn = reinterpret_cast<decltype(&fcqt_synthesis)>(synthesis_fn);
            e->table_mem = table_mem;
            e->device = table_mem.device();
            for (const auto& g : groups) e->groups.push_back({g.at(0), g.at(1), g.at(2)});
            e->octave_groups = octave_groups;
            return e;
        }))
        .def("set_workspace",
             [](const Ref& e, int64_t rows, const Tensor& x, const Tensor& w, const Tensor& f,
                const std::optional<Tensor>& fa) {
                 std::lock_guard<std::mutex> lock(e->mu);
                 e->rows = rows;
                 e->X = x;
                 e->W = w;
                 e->F = f;
                 e->FA = fa ? *fa : Tensor();
             })
        .def("clear_workspace",
             [](const Ref& e) {
                 std::lock_guard<std::mutex> lock(e->mu);
                 e->rows = 0;
                 e->X = e->W = e->F = e->FA = Tensor();
                 e->captured = false;
             })
        // waiting without the GIL: the holder may need it to get on
        .def("__enter__", [](const Ref& e) { e->launching.lock(); }, py::call_guard<py::gil_scoped_release>())
        .def("__exit__", [](const Ref& e, const py::args&) { e->launching.unlock(); })
        .def_property_readonly("captured", [](const Ref& e) { return e->captured.load(); })
        .def("block_base", [](const Ref& e, const std::vector<Tensor>& parts, int64_t rows) {
            return block_base(e, parts, rows);
        })
        .def("fwd", [](const Ref& e, const Tensor& x) { return guarded(fwd, e, x); })
        .def("bwd", [](const Ref& e, const std::vector<Tensor>& parts) { return guarded(bwd, e, parts); });
}
