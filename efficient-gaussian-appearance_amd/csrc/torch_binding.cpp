// The differentiable entry points (diff_rasterize, neural_decode) as C++ autograd functions over the C ABI
// (include/efgs.h): input checks, native structs, workspaces and gradient outputs are made here, without Python objects
// and without the interpreter's lock. Small frames are bound by the host: with the same steps in Python (a Python
// autograd function, ctypes structs, a view per gradient) a training pass over 10k Gaussians at 256 x 192 took 237 us
// for 113 us of kernels, 115 us now; over 100k at 800 x 800 248 -> 156 us; the decode of 1M primitives, forward and
// backward, 143 -> 92 us.
//
// Reference counterpart: B/torch_bindings/rasterization.py:86-196 (the Python autograd function around _C.forward and
// _C.backward).
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/utils/pybind.h>
#include <torch/extension.h>

#include <array>
#include <map>
#include <mutex>
#include <string>
#include <utility>
#include <vector>

#include "../../include/efgs.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

// One device allocation per call, handed out by the library's bump allocator; requests beyond it get tensors of their
// own. The region follows the largest total requested so far (per call kind and device, with 1/16 headroom), so in
// steady state a call makes a single allocation.
class Workspace {
  public:
    enum Kind { forward = 0, backward = 1, decode = 2, forward_no_backward = 3 };

    Workspace(Kind kind, at::Device device) : key_(kind, device.index()), options_(at::TensorOptions().dtype(at::kByte).device(device)) {
        size_t capacity = 0;
        {
            std::lock_guard<std::mutex> lock(mutex());
            capacity = sizes()[key_];
        }
        tensors_.push_back(at::empty({static_cast<int64_t>(capacity > 256 ? capacity : 256)}, options_));
        ws_ = efgs_workspace{tensors_[0].data_ptr(), capacity, 0, 0, &Workspace::fallback, this};
    }
    Workspace(const Workspace&) = delete;
    Workspace& operator=(const Workspace&) = delete;

    efgs_workspace* context() { return &ws_; }

    // records the call's total for the next region; the tensors back every buffer that was handed out
    std::vector<Tensor> finish() {
        std::lock_guard<std::mutex> lock(mutex());
        size_t& size = sizes()[key_];
        if (ws_.requested > size) size = (ws_.requested + ws_.requested / 16 + 255) / 256 * 256;
        return std::move(tensors_);
    }

  private:
    static void* fallback(void* self, size_t bytes) noexcept {
        try {
            Workspace* w = static_cast<Workspace*>(self);
            w->tensors_.push_back(at::empty({static_cast<int64_t>(bytes > 0 ? bytes : 1)}, w->options_));
            return w->tensors_.back().data_ptr();
        } catch (...) {  // (out of memory: the library reports the failed allocation)
            return nullptr;
        }
    }
    static std::mutex& mutex() {
        static std::mutex m;
        return m;
    }
    static std::map<std::pair<int, int>, size_t>& sizes() {
        static std::map<std::pair<int, int>, size_t> s;
        return s;
    }

    std::pair<int, int> key_;
    at::TensorOptions options_;
    std::vector<Tensor> tensors_;
    efgs_workspace ws_{};
};

void check_status(int rc) {
    if (rc == EFGS_OK) return;
    const char* message = efgs_last_error();
    TORCH_CHECK(false, "efgs: ", message && *message ? message : "error", " (status ", rc, ")");
}

void* current_stream(at::Device device) { return c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(device.index()).stream(); }

template <typename T>
T* pointer(const Tensor& t) {
    return t.numel() > 0 ? static_cast<T*>(t.data_ptr()) : nullptr;
}

void check_parameter(const char* name, const Tensor& t, at::Device device) {
    if (t.numel() == 0) return;
    TORCH_CHECK_VALUE(t.scalar_type() == at::kFloat, "efgs: ", name, " must be float32, got ", t.dtype());
    TORCH_CHECK_VALUE(t.device() == device, "efgs: ", name, " is on ", t.device(), ", expected ", device);
    TORCH_CHECK_VALUE(t.is_contiguous(), "efgs: ", name, " must be contiguous");
}

// contiguous float32 on `device` (the tensor itself when it already is)
Tensor as_float(const Tensor& t, at::Device device) { return t.detach().to(device, at::kFloat).contiguous(); }

// the camera tensors of RasterizerSettings in the rendering device's memory, and the native struct that points to them
struct Camera {
    efgs_settings native{};
    Tensor w2c, position, background;
};

enum Input { in_means, in_scales, in_rotations, in_opacities, in_precomputed, in_base, in_residual, in_mlp, n_inputs };

efgs_primitives native_primitives(const std::vector<Tensor>& t) {
    efgs_primitives p{};
    p.n_primitives = t[in_means].size(0);
    p.means = static_cast<const float*>(t[in_means].data_ptr());
    p.scales = static_cast<const float*>(t[in_scales].data_ptr());
    p.rotations = static_cast<const float*>(t[in_rotations].data_ptr());
    p.opacities = static_cast<const float*>(t[in_opacities].data_ptr());
    p.precomputed_colors = pointer<const float>(t[in_precomputed]);
    p.base_colors = pointer<const float>(t[in_base]);
    p.residual_params = pointer<const float>(t[in_residual]);
    p.mlp_weights = pointer<const float>(t[in_mlp]);
    return p;
}

// what the backward keeps of its forward beside the saved tensors
struct Frame : torch::CustomClassHolder {
    efgs_rasterizer* rasterizer = nullptr;
    Camera camera;
    efgs_frame frame{};
    std::array<int64_t, 4> counts{};  // primitives, visible primitives, instances, tiles
    std::vector<Tensor> buffers;
    Tensor densification;
    int64_t rows = 0;
    bool differentiable = false;
};

// The gradients of a backward that is itself being differentiated (create_graph with an upstream that requires a
// gradient) hang on the upstream by an identity whose own backward raises: the kernels have no second derivatives, and a
// graph without this edge would give zeros for them. The message is the one that Python autograd functions marked
// once_differentiable give, which programs may look for.
struct FirstOrderOnly : torch::autograd::Function<FirstOrderOnly> {
    static Tensor forward(AutogradContext*, const Tensor& /*upstream*/, const Tensor& grad) { return grad.variable_data(); }  // (no view: it may be changed in place)
    static variable_list backward(AutogradContext*, variable_list) {
        TORCH_CHECK(false, "trying to differentiate twice a function that was marked with @once_differentiable");
    }
};

variable_list first_order_only(variable_list grads, const Tensor& upstream) {
    if (at::GradMode::is_enabled() && upstream.requires_grad())
        for (Tensor& g : grads)
            if (g.defined()) g = FirstOrderOnly::apply(upstream, g);
    return grads;
}

struct Rasterize : torch::autograd::Function<Rasterize> {
    static Tensor forward(AutogradContext* ctx, const Tensor& means, const Tensor& scales, const Tensor& rotations, const Tensor& opacities,
                          const Tensor& precomputed, const Tensor& base, const Tensor& residual, const Tensor& mlp_weights,
                          c10::intrusive_ptr<Frame> state) {
        const at::Device device = means.device();
        const Tensor mlp = mlp_weights.numel() > 0 ? as_float(mlp_weights, mlp_weights.device())
                                                   : at::empty({0}, at::TensorOptions().dtype(at::kFloat).device(device));
        const std::vector<Tensor> inputs = {means, scales, rotations, opacities, precomputed, base, residual, mlp};
        TORCH_CHECK_VALUE(device.is_cuda(), "efgs: the rasterizer runs on a GPU device");
        static const char* const names[] = {"means", "scales", "rotations", "opacities", "precomputed_colors", "base_colors", "residual_params"};
        for (int i = 0; i < in_mlp; i++) check_parameter(names[i], inputs[i], device);
        if (mlp.numel() > 0) {
            const int64_t expected = efgs_mlp_param_count(state->rasterizer);
            TORCH_CHECK_VALUE(mlp.numel() == expected && mlp.device() == device, "efgs: mlp_weights must hold ", expected, " parameters on ",
                              device, ", got ", mlp.numel());
        }
        const Tensor& dinfo = state->densification;
        state->rows = dinfo.defined() && dinfo.numel() > 0 ? dinfo.size(0) : 0;
        if (state->rows > 0 && state->differentiable)
            TORCH_CHECK_VALUE(dinfo.scalar_type() == at::kFloat && dinfo.is_contiguous() && dinfo.size(-1) == means.size(0) && dinfo.device() == device,
                              "efgs: densification_info must be a contiguous float32 (2|3, N) tensor on the rendering device");
        const c10::DeviceGuard guard(device);
        Camera& cam = state->camera;
        cam.w2c = as_float(cam.w2c, device);
        cam.position = as_float(cam.position, device);
        cam.background = as_float(cam.background, device);
        TORCH_CHECK_VALUE(cam.w2c.numel() >= 12, "efgs: w2c needs at least 3 rows of 4 entries");
        cam.native.w2c = static_cast<const float*>(cam.w2c.data_ptr());
        cam.native.cam_position = static_cast<const float*>(cam.position.data_ptr());
        cam.native.bg_color = static_cast<const float*>(cam.background.data_ptr());
        const Tensor image = at::empty({3, cam.native.height, cam.native.width}, at::TensorOptions().dtype(at::kFloat).device(device));
        const efgs_primitives prims = native_primitives(inputs);
        if (!state->differentiable) {
            Workspace workspace(Workspace::forward_no_backward, device);
            check_status(efgs_forward_no_backward(state->rasterizer, &prims, &cam.native, static_cast<float*>(image.data_ptr()), efgs_workspace_alloc,
                                                  workspace.context(), state->counts.data(), current_stream(device)));
            workspace.finish();
            return image;
        }
        Workspace workspace(Workspace::forward, device);
        check_status(efgs_forward(state->rasterizer, &prims, &cam.native, static_cast<float*>(image.data_ptr()), efgs_workspace_alloc,
                                  workspace.context(), &state->frame, current_stream(device)));
        state->buffers = workspace.finish();
        const efgs_frame& f = state->frame;
        state->counts = {f.n_primitives, f.n_visible, f.n_instances, static_cast<int64_t>(f.grid_width) * f.grid_height};
        ctx->saved_data["frame"] = c10::IValue::make_capsule(state);
        ctx->saved_data["mlp_numel"] = mlp_weights.numel();
        ctx->save_for_backward({image, means, scales, rotations, opacities, precomputed, base, residual, mlp});
        return image;
    }

    static variable_list backward(AutogradContext* ctx, variable_list upstream) {
        const variable_list saved = ctx->get_saved_variables();  // (checks that no saved tensor was modified in place)
        variable_list grads;
        {
            at::NoGradGuard no_grad;
            grads = gradients(ctx, saved, upstream[0]);
        }
        return first_order_only(std::move(grads), upstream[0]);
    }

    static variable_list gradients(AutogradContext* ctx, const variable_list& saved, const Tensor& upstream) {
        const auto state = c10::static_intrusive_pointer_cast<Frame>(ctx->saved_data["frame"].toCapsule());
        const Tensor& image = saved[0];
        const at::Device device = image.device();
        const Tensor grad_image = upstream.contiguous();
        TORCH_CHECK_VALUE(grad_image.sizes() == image.sizes() && grad_image.scalar_type() == at::kFloat && grad_image.device() == device,
                          "efgs: the image gradient must be a float32 tensor of the image's shape on its device");
        const c10::DeviceGuard guard(device);
        const std::vector<Tensor> inputs(saved.begin() + 1, saved.end());
        // every gradient output is fully written by the backward
        const auto options = at::TensorOptions().dtype(at::kFloat).device(device);
        variable_list out;
        for (int i = 0; i < in_mlp; i++) out.push_back(at::empty(inputs[i].sizes(), options));
        out.push_back(at::empty({ctx->saved_data["mlp_numel"].toInt()}, options));
        efgs_gradients g{};
        g.means = static_cast<float*>(out[in_means].data_ptr());
        g.scales = static_cast<float*>(out[in_scales].data_ptr());
        g.rotations = static_cast<float*>(out[in_rotations].data_ptr());
        g.opacities = static_cast<float*>(out[in_opacities].data_ptr());
        g.precomputed_colors = pointer<float>(out[in_precomputed]);
        g.base_colors = pointer<float>(out[in_base]);
        g.residual_params = pointer<float>(out[in_residual]);
        g.mlp_weights = pointer<float>(out[in_mlp]);
        g.densification_info = state->rows > 0 ? static_cast<float*>(state->densification.data_ptr()) : nullptr;
        g.densification_rows = static_cast<int>(state->rows);
        const efgs_primitives prims = native_primitives(inputs);
        Workspace workspace(Workspace::backward, device);
        check_status(efgs_backward(state->rasterizer, &prims, &state->camera.native, &state->frame, static_cast<const float*>(image.data_ptr()),
                                   static_cast<const float*>(grad_image.data_ptr()), &g, efgs_workspace_alloc, workspace.context(),
                                   current_stream(device)));
        workspace.finish();
        for (int i = in_precomputed; i < n_inputs; i++)
            if (out[i].numel() == 0) out[i] = Tensor();
        out.push_back(Tensor());  // (the frame)
        return out;
    }
};

Tensor given_or_empty(const c10::optional<Tensor>& t, at::Device device) {
    return t.has_value() ? *t : at::empty({0}, at::TensorOptions().dtype(at::kFloat).device(device));
}

// The image and the frame's counts (primitives, visible primitives, instances, tiles). The arguments from w2c on are
// RasterizerSettings' fields in order, then the optional colour inputs.
std::pair<Tensor, std::array<int64_t, 4>> diff_rasterize(uintptr_t rasterizer, const Tensor& means, const Tensor& scales, const Tensor& rotations,
                                                         const Tensor& opacities, const Tensor& densification, const Tensor& w2c,
                                                         const Tensor& position, const Tensor& background, int appearance_degree, int width,
                                                         int height, double focal_x, double focal_y, double center_x, double center_y,
                                                         double near_plane, double far_plane, bool proper_antialiasing, bool render_base,
                                                         bool render_residual, const c10::optional<Tensor>& precomputed,
                                                         const c10::optional<Tensor>& base, const c10::optional<Tensor>& residual,
                                                         const c10::optional<Tensor>& mlp) {
    auto state = c10::make_intrusive<Frame>();
    state->rasterizer = reinterpret_cast<efgs_rasterizer*>(rasterizer);
    state->densification = densification;
    state->camera.w2c = w2c;
    state->camera.position = position;
    state->camera.background = background;
    efgs_settings& s = state->camera.native;
    s.appearance_degree = appearance_degree;
    s.width = width;
    s.height = height;
    s.focal_x = static_cast<float>(focal_x);
    s.focal_y = static_cast<float>(focal_y);
    s.center_x = static_cast<float>(center_x);
    s.center_y = static_cast<float>(center_y);
    s.near_plane = static_cast<float>(near_plane);
    s.far_plane = static_cast<float>(far_plane);
    s.proper_antialiasing = proper_antialiasing ? 1 : 0;
    s.render_base = render_base ? 1 : 0;
    s.render_residual = render_residual ? 1 : 0;
    const at::Device device = means.device();
    const Tensor pre = given_or_empty(precomputed, device), base_colors = given_or_empty(base, device);
    const Tensor residual_params = given_or_empty(residual, device), mlp_weights = given_or_empty(mlp, device);
    for (const Tensor* t : {&means, &scales, &rotations, &opacities, &pre, &base_colors, &residual_params, &mlp_weights})
        state->differentiable = state->differentiable || (at::GradMode::is_enabled() && t->requires_grad());
    Tensor image = Rasterize::apply(means, scales, rotations, opacities, pre, base_colors, residual_params, mlp_weights, state);
    return {std::move(image), state->counts};
}

struct NeuralDecode : torch::autograd::Function<NeuralDecode> {
    static Tensor forward(AutogradContext* ctx, const Tensor& features, const Tensor& dirs, const Tensor& mlp_weights, const Tensor& base,
                          int64_t rasterizer, int64_t degree) {
        const at::Device device = features.device();
        const c10::DeviceGuard guard(device);
        const Tensor half = mlp_weights.detach().to(at::kHalf).contiguous();
        const int64_t n = dirs.size(0);
        const Tensor out = at::empty({n, 3}, at::TensorOptions().dtype(at::kFloat).device(device));
        check_status(efgs_neural_decode_forward(reinterpret_cast<efgs_rasterizer*>(rasterizer), n, pointer<const float>(features),
                                                pointer<const float>(base), pointer<const float>(dirs), pointer<const uint16_t>(half),
                                                static_cast<int>(degree), pointer<float>(out), current_stream(device)));
        ctx->saved_data["rasterizer"] = rasterizer;
        ctx->saved_data["degree"] = degree;
        ctx->saved_data["mlp_numel"] = mlp_weights.numel();
        ctx->save_for_backward({features, dirs, half, base});
        return out;
    }

    static variable_list backward(AutogradContext* ctx, variable_list upstream) {
        const variable_list saved = ctx->get_saved_variables();
        variable_list grads;
        {
            at::NoGradGuard no_grad;
            grads = gradients(ctx, saved, upstream[0]);
        }
        return first_order_only(std::move(grads), upstream[0]);
    }

    static variable_list gradients(AutogradContext* ctx, const variable_list& saved, const Tensor& upstream) {
        const Tensor &features = saved[0], &dirs = saved[1], &half = saved[2], &base = saved[3];
        const at::Device device = features.device();
        const c10::DeviceGuard guard(device);
        const Tensor grad_out = upstream.contiguous();
        Tensor g_features = at::empty_like(features), g_dirs = at::empty_like(dirs), g_base = at::empty_like(base);
        Tensor g_mlp = at::empty({ctx->saved_data["mlp_numel"].toInt()}, at::TensorOptions().dtype(at::kFloat).device(device));
        Workspace workspace(Workspace::decode, device);
        check_status(efgs_neural_decode_backward(reinterpret_cast<efgs_rasterizer*>(ctx->saved_data["rasterizer"].toInt()), dirs.size(0),
                                                 pointer<const float>(features), pointer<const float>(base), pointer<const float>(dirs),
                                                 pointer<const uint16_t>(half), static_cast<int>(ctx->saved_data["degree"].toInt()),
                                                 pointer<const float>(grad_out), pointer<float>(g_features), pointer<float>(g_base),
                                                 pointer<float>(g_dirs), pointer<float>(g_mlp), efgs_workspace_alloc, workspace.context(),
                                                 current_stream(device)));
        workspace.finish();
        return {features.numel() > 0 ? g_features : Tensor(), g_dirs, g_mlp, base.numel() > 0 ? g_base : Tensor(), Tensor(), Tensor()};
    }
};

Tensor neural_decode(uintptr_t rasterizer, const Tensor& features, const Tensor& dirs, const Tensor& mlp_weights, const Tensor& base, int64_t degree) {
    return NeuralDecode::apply(features, dirs, mlp_weights, base, static_cast<int64_t>(rasterizer), degree);
}

}  // namespace

PYBIND11_MODULE(_native, m) {
    m.doc() = "C++ autograd functions of efgs";
    // (the interpreter's lock is released while they run; C++ errors become the Python exceptions torch maps them to)
    m.def("diff_rasterize", torch::wrap_pybind_function_no_gil(diff_rasterize));
    m.def("neural_decode", torch::wrap_pybind_function_no_gil(neural_decode));
}
