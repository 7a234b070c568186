// Host path of the framework between torch and libmsd_hip.so: a small network is bound by what
// the host does between launches, so the calls that such a program makes again and again run
// here, without the interpreter: one differentiated layer, the forward pass of a network, a
// whole training step up to the gradients, and the optimiser.
//
// Every entry checks its arguments and returns None for whatever it does not take (other types,
// strides, hooks, tensor subclasses, forward mode, a tracer that is running ...); the Python modules then go
// their general way, which also raises the errors.  Nothing is kept between calls.
#include <torch/extension.h>

#include <ATen/SavedTensorHooks.h>
#include <ATen/autocast_mode.h>
#include <ATen/core/grad_mode.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <dlfcn.h>
#include <torch/csrc/autograd/anomaly_mode.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/variable.h>
#include <torch/csrc/jit/frontend/tracer.h>

#include <string>
#include <vector>

#include "../../../include/msd_hip.h"

namespace {

using at::Tensor;
namespace py = pybind11;

// The entry points, looked up in the library that the package has loaded.
#define MSD_ENTRIES(X)                                                                                              \
    X(msd_last_error) X(msd_conv_forward) X(msd_conv_relu_forward) X(msd_conv_layer_backward) X(msd_conv_layer_workspace_bytes)  \
    X(msd_block_forward_ws) X(msd_block_forward_workspace_bytes_of) X(msd_block_backward) X(msd_block_workspace_bytes) X(msd_final_forward)                     \
    X(msd_final_backward) X(msd_final_forward_loss) X(msd_final_workspace_bytes) X(msd_scale_fold) X(msd_adam_step)   \
    X(msd_label_check)
struct Entries {
#define X(name) decltype(&::name) name = nullptr;
    MSD_ENTRIES(X)
#undef X
} lib;

void bind(const std::string &path)
{
    void *h = dlopen(path.c_str(), RTLD_NOW | RTLD_LOCAL);
    TORCH_CHECK(h, "cannot load ", path, ": ", dlerror());
#define X(name)                                                    \
    lib.name = reinterpret_cast<decltype(lib.name)>(dlsym(h, #name)); \
    TORCH_CHECK(lib.name, path, " does not export " #name);
    MSD_ENTRIES(X)
#undef X
}

void check(int rc) { TORCH_CHECK(rc == MSD_OK, lib.msd_last_error()); }

int dtype_of(const Tensor &t) { return t.scalar_type() == at::kFloat ? MSD_F32 : MSD_F64; }

void *stream_on(const at::Device &d) { return c10::hip::getCurrentHIPStream(d.index()).stream(); }

// A dense tensor on the GPU that nothing dispatches on and that carries no tangent of forward mode.
bool plain(const Tensor &t)
{
    return t.defined() && t.is_cuda() && t.layout() == at::kStrided && !t.is_neg() && !t.is_conj() &&
           !t._fw_grad(0).defined() &&
           !t.key_set().has_any(c10::DispatchKeySet({c10::DispatchKey::Python, c10::DispatchKey::FuncTorchBatched,
                                                     c10::DispatchKey::FuncTorchGradWrapper,
                                                     c10::DispatchKey::Functionalize}));
}
// A tracer records autograd functions as calls of their own; it cannot see the calls made here, and
// their results would become constants of the trace.
bool traced() { return torch::jit::tracer::isTracing(); }

bool floating(const Tensor &t) { return t.scalar_type() == at::kFloat || t.scalar_type() == at::kDouble; }
bool like(const Tensor &t, const Tensor &first)
{
    return plain(t) && t.scalar_type() == first.scalar_type() && t.device() == first.device();
}

bool kernel_ok(const Tensor &w, int64_t dim)
{
    if (w.dim() != dim || !w.is_contiguous()) return false;
    for (int64_t i = 2; i < dim; i++)
        if (w.size(i) != 3) return false;
    return true;
}

bool dilation_ok(const Tensor &x, int64_t d)
{
    if (d <= 0) return false;
    for (int64_t i = 2; i < x.dim(); i++)
        if (d > x.size(i)) return false;
    return true;
}

// Every channel plane contiguous (what the final layer's kernels take).
bool planes_ok(const Tensor &t)
{
    if (t.numel() == 0) return false;
    int64_t want = 1;
    for (int64_t i = t.dim() - 1; i >= 2; i--) {
        if (t.size(i) != 1 && t.stride(i) != want) return false;
        want *= t.size(i);
    }
    return true;
}

int64_t voxels(const Tensor &t)
{
    int64_t n = 1;
    for (int64_t i = 2; i < t.dim(); i++) n *= t.size(i);
    return n;
}

Tensor workspace(int64_t bytes, const Tensor &like_t)
{
    TORCH_CHECK(bytes >= 0, lib.msd_last_error());
    return at::empty({bytes > 8 ? bytes : 8}, like_t.options().dtype(at::kByte).requires_grad(false));
}

// ---------------------------------------------------------------------------
// One layer: conv[+ReLU] into the caller's output, differentiated.
// ---------------------------------------------------------------------------

class ConvLayer : public torch::autograd::Function<ConvLayer> {
  public:
    static Tensor forward(torch::autograd::AutogradContext *ctx, const Tensor &x, const Tensor &w, const Tensor &b,
                          const Tensor &out, int64_t dilation, bool relu)
    {
        const auto f = relu ? lib.msd_conv_relu_forward : lib.msd_conv_forward;
        check(f(dtype_of(x), (int)x.dim() - 2, x.size(0), x.size(1), out.size(1), x.sizes().data() + 2, (int)dilation,
                x.data_ptr(), x.strides().data(), w.data_ptr(), b.data_ptr(), out.data_ptr(), out.strides().data(),
                stream_on(x.device())));
        if (relu)
            ctx->save_for_backward({x, w, b, out});
        else
            ctx->save_for_backward({x, w, b});
        ctx->saved_data["dilation"] = dilation;
        ctx->saved_data["relu"] = relu;
        return out;
    }

    static torch::autograd::variable_list backward(torch::autograd::AutogradContext *ctx,
                                                   const torch::autograd::variable_list &grads)
    {
        const auto saved = ctx->get_saved_variables();
        const bool relu = ctx->saved_data["relu"].toBool();
        const int64_t dilation = ctx->saved_data["dilation"].toInt();
        const Tensor &x = saved[0], &w = saved[1], &b = saved[2];
        const Tensor out = relu ? saved[3] : Tensor();
        at::AutoDispatchBelowADInplaceOrView below;
        const c10::DeviceGuard guard(x.device());
        const Tensor g = grads[0].contiguous();
        TORCH_CHECK(plain(g) && g.scalar_type() == x.scalar_type() && g.device() == x.device() && g.dim() == x.dim() &&
                        g.size(0) == x.size(0) && g.size(1) == w.size(0),
                    "conv backward: unexpected output gradient");
        const Tensor gx = ctx->needs_input_grad(0) ? at::empty_like(x) : Tensor();
        const Tensor gw = ctx->needs_input_grad(1) ? at::empty_like(w) : Tensor();
        const Tensor gb = ctx->needs_input_grad(2) ? at::empty_like(b) : Tensor();
        if (gx.defined() || gw.defined() || gb.defined()) {
            Tensor ws;
            int64_t need = 0;
            if (gw.defined() || gb.defined()) {
                need = lib.msd_conv_layer_workspace_bytes(dtype_of(x), (int)x.dim() - 2, x.size(0), x.size(1), w.size(0),
                                                          x.sizes().data() + 2);
                ws = workspace(need, x);
            }
            check(lib.msd_conv_layer_backward(
                relu, dtype_of(x), (int)x.dim() - 2, x.size(0), x.size(1), w.size(0), x.sizes().data() + 2,
                (int)dilation, relu ? out.data_ptr() : nullptr, relu ? out.strides().data() : nullptr, g.data_ptr(),
                g.strides().data(), x.data_ptr(), x.strides().data(), w.data_ptr(),
                gx.defined() ? gx.data_ptr() : nullptr, gx.defined() ? gx.strides().data() : nullptr,
                gw.defined() ? gw.data_ptr() : nullptr, gb.defined() ? gb.data_ptr() : nullptr,
                ws.defined() ? ws.data_ptr() : nullptr, need, stream_on(x.device())));
        }
        return {gx, gw, gb, Tensor(), Tensor(), Tensor()};
    }
};

std::optional<Tensor> conv_layer(const Tensor &x, const Tensor &w, const Tensor &b, const Tensor &out,
                                 int64_t dilation, bool relu)
{
    if (traced() || !plain(x) || !floating(x) || (x.dim() != 4 && x.dim() != 5) || !like(w, x) || !like(b, x) || !like(out, x) ||
        !kernel_ok(w, x.dim()) || w.size(1) != x.size(1) || b.dim() != 1 || !b.is_contiguous() ||
        b.size(0) != w.size(0) || out.dim() != x.dim() || out.size(0) != x.size(0) || out.size(1) != w.size(0) ||
        out.sizes().slice(2) != x.sizes().slice(2) || !dilation_ok(x, dilation) || x.numel() == 0)
        return std::nullopt;
    const c10::DeviceGuard guard(x.device());
    py::gil_scoped_release nogil;
    return ConvLayer::apply(x, w, b, out, dilation, relu);
}

// ---------------------------------------------------------------------------
// The dense block, as the network's forward pass and training step run it.
// ---------------------------------------------------------------------------

struct Block {
    std::vector<int64_t> widths, dilations;
    std::vector<const void *> weights;
    int64_t c_in = 0, channels = 0;

    // false for anything that the native block does not take as it is
    bool set(const Tensor &x, const Tensor &bias, const std::vector<Tensor> &ws, const std::vector<int64_t> &dils)
    {
        if (ws.empty() || ws.size() != dils.size() || !like(bias, x) || bias.dim() != 1 || !bias.is_contiguous())
            return false;
        c_in = channels = x.size(1);
        for (size_t i = 0; i < ws.size(); i++) {
            const Tensor &w = ws[i];
            if (!like(w, x) || !kernel_ok(w, x.dim()) || w.size(1) != channels || w.size(0) < 1 || !dilation_ok(x, dils[i]))
                return false;
            widths.push_back(w.size(0));
            weights.push_back(w.data_ptr());
            channels += w.size(0);
        }
        dilations = dils;
        return bias.size(0) == channels - c_in;
    }

    // A channel stack (or the gradient of one) for the native calls alone.  A wave of the block's
    // kernels reads a short run of 16 channels at a time; where the channels lie a multiple of
    // kCamped bytes apart these runs meet in few of the memory's channels, so such planes are moved
    // apart by kApart bytes (from kFrom bytes on: smaller ones come from the caches).  1024 x 1024, 104
    // channels, a pass of msd_pull.hip: 452 -> 372 us; a training step there, depth 100: 6.7 -> 6.3 ms;
    // 2048 x 2048, two channels per layer, depth 200: 319 -> 272; a forward pass of 256^3, depth 30: 10.0 -> 9.6.
    // Distances of 128 to 66048 bytes did the same in 2D; 128^3, depth 50, gains 1 % with this one and loses 0.5 %
    // with 512 or 66048.  Planes of other sizes gain nothing (1000 x 1056: 396 us with and without).
    Tensor new_stack(const Tensor &x) const
    {
        constexpr int64_t kCamped = 64 * 1024, kFrom = 1 << 20, kApart = 32 * 1024 + 512;
        auto sizes = x.sizes().vec();
        sizes[1] = channels;
        const auto options = x.options().requires_grad(false);
        const int64_t el = x.element_size(), plane = voxels(x);
        if (plane * el % kCamped != 0 || plane * el < kFrom) return at::empty(sizes, options);
        std::vector<int64_t> strides(sizes.size(), 1);
        for (size_t d = sizes.size() - 1; d > 2; d--) strides[d - 1] = strides[d] * sizes[d];
        strides[1] = plane + kApart / el;
        strides[0] = channels * strides[1];
        return at::empty_strided(sizes, strides, options);
    }

    void forward(const Tensor &stack, const Tensor &bias, void *stream) const
    {
        Tensor ws;
        int64_t need = 0;
        for (const int outputs : {14, 7}) {
            const int64_t bytes = lib.msd_block_forward_workspace_bytes_of(
                dtype_of(stack), (int)stack.dim() - 2, stack.size(0), c_in, (int)widths.size(), widths.data(),
                stack.sizes().data() + 2, dilations.data(), outputs);
            if (bytes <= 0 || bytes == need) break;
            need = bytes;
            try {
                ws = workspace(need, stack);
                break;
            } catch (const c10::OutOfMemoryError &) {
                // groups of half as many layers, or none: the layers then run one by one
            }
        }
        check(lib.msd_block_forward_ws(dtype_of(stack), (int)stack.dim() - 2, stack.size(0), c_in, (int)widths.size(),
                                       widths.data(), stack.sizes().data() + 2, dilations.data(), stack.data_ptr(),
                                       stack.strides().data(), weights.data(), bias.data_ptr(),
                                       ws.defined() ? ws.data_ptr() : nullptr, ws.defined() ? need : 0, stream));
    }
};

bool final_ok(const Block &block, const Tensor &x, const Tensor &fw, const Tensor &fb)
{
    return like(fw, x) && like(fb, x) && fw.dim() >= 2 && fw.size(1) == block.channels && fw.is_contiguous() &&
           fw.numel() == fw.size(0) * fw.size(1) && fb.dim() == 1 && fb.size(0) == fw.size(0) && fb.is_contiguous();
}

bool scale_ok(const Tensor &w, const Tensor &b, const Tensor &x, int64_t channels)
{
    return like(w, x) && like(b, x) && w.is_contiguous() && b.is_contiguous() && w.size(0) == channels &&
           w.numel() == channels * channels && b.numel() == channels && !w.requires_grad() && !b.requires_grad();
}

void pointwise(const Tensor &x, const Tensor &w, const Tensor &b, const Tensor &out, int64_t c_out, void *stream)
{
    check(lib.msd_final_forward(dtype_of(x), x.size(0), x.size(1), c_out, voxels(x), x.data_ptr(), x.stride(0),
                                x.stride(1), w.data_ptr(), b.data_ptr(), out.data_ptr(), out.stride(0), out.stride(1),
                                stream));
}

// Output of block + final layer, without gradients.
std::optional<Tensor> net_forward(const Tensor &x, const Tensor &bias, const std::vector<Tensor> &weights,
                                  const std::vector<int64_t> &dilations, const Tensor &fw, const Tensor &fb)
{
    if (traced() || !plain(x) || !floating(x) || (x.dim() != 4 && x.dim() != 5) || x.numel() == 0) return std::nullopt;
    Block block;
    if (!block.set(x, bias, weights, dilations) || !final_ok(block, x, fw, fb)) return std::nullopt;
    const c10::DeviceGuard guard(x.device());
    at::AutoDispatchBelowADInplaceOrView below;
    py::gil_scoped_release nogil;
    void *stream = stream_on(x.device());
    const Tensor stack = block.new_stack(x);
    stack.narrow(1, 0, block.c_in).copy_(x);
    block.forward(stack, bias, stream);
    auto sizes = x.sizes().vec();
    sizes[1] = fw.size(0);
    const Tensor out = at::empty(sizes, x.options().requires_grad(false));
    pointwise(stack, fw, fb, out, fw.size(0), stream);
    return out;
}

// Somebody looks at the graph that a training step would make: hooks on what it saves, a check of
// every gradient for NaN, or autocast, which acts on the products with the output scaling (and which the
// general path refuses for that).
bool watched()
{
    return !at::SavedTensorDefaultHooks::get_tls_state().stack.empty() || torch::autograd::AnomalyMode::is_enabled() ||
           at::autocast::is_autocast_enabled(at::kCUDA);
}

// A parameter whose gradient can be set without autograd: a leaf that nobody watches.
bool settable(const Tensor &p)
{
    if (!p.requires_grad() || !p.is_leaf()) return false;
    auto *meta = torch::autograd::impl::get_autograd_meta(p);
    if (!meta || !meta->hooks_.empty() || meta->post_acc_grad_hooks_) return false;
    if (const auto acc = torch::autograd::impl::try_get_grad_accumulator(p))
        return acc->pre_hooks().empty() && acc->tensor_pre_hooks().empty() && acc->post_hooks().empty();
    return true;
}

// A tensor over a piece of `flat` (what flat.narrow().view() gives, without two dispatched calls).
Tensor piece(const Tensor &flat, int64_t offset, const Tensor &shaped_like)
{
    Tensor t = at::detail::make_tensor<c10::TensorImpl>(c10::Storage(flat.storage()), flat.key_set(), flat.dtype());
    t.unsafeGetTensorImpl()->set_storage_offset(flat.storage_offset() + offset);
    t.unsafeGetTensorImpl()->set_sizes_contiguous(shaped_like.sizes());
    return t;
}

// One training step short of the optimiser: scaling of the input, block, final layer (with the
// frozen output scaling folded into it), loss, and the gradients of all parameters, which
// REPLACE their .grad.  Same launches as the autograd node MSDNetLossFunction makes.  Returns
// (loss, output), or None (and nothing has happened).
std::optional<std::pair<Tensor, Tensor>> train_step(const Tensor &x, const Tensor &sw, const Tensor &sb,
                                                    const Tensor &bias, const std::vector<Tensor> &weights,
                                                    const std::vector<int64_t> &dilations, const Tensor &fw,
                                                    const Tensor &fb, const std::optional<Tensor> &osw,
                                                    const std::optional<Tensor> &osb, const Tensor &target, int kind)
{
    if (traced() || watched() || !plain(x) || !floating(x) || (x.dim() != 4 && x.dim() != 5) || !planes_ok(x) ||
        x.requires_grad())
        return std::nullopt;
    Block block;
    if (!block.set(x, bias, weights, dilations) || !final_ok(block, x, fw, fb)) return std::nullopt;
    const int64_t c_out = fw.size(0), c_in = block.c_in, channels = block.channels;
    if (c_out > 8 || !scale_ok(sw, sb, x, c_in)) return std::nullopt;
    const bool scaled = osw.has_value();
    if (scaled != osb.has_value() || (scaled && !scale_ok(*osw, *osb, x, c_out))) return std::nullopt;
    if (!plain(target) || target.device() != x.device() || target.requires_grad() || target.dim() == 0 ||
        target.size(0) != x.size(0))
        return std::nullopt;
    if (kind == MSD_LOSS_NLL) {
        if (target.scalar_type() != at::kLong || target.dim() != x.dim() - 1 || !target.is_contiguous() ||
            target.sizes().slice(1) != x.sizes().slice(2))
            return std::nullopt;
    } else if (target.scalar_type() != x.scalar_type() || target.dim() != x.dim() || target.size(1) != c_out ||
               target.sizes().slice(2) != x.sizes().slice(2) || !planes_ok(target)) {
        return std::nullopt;
    }
    if (!settable(bias) || !settable(fw) || !settable(fb)) return std::nullopt;
    for (const Tensor &w : weights)
        if (!settable(w)) return std::nullopt;

    const c10::DeviceGuard guard(x.device());
    at::AutoDispatchBelowADInplaceOrView below;
    py::gil_scoped_release nogil;
    void *stream = stream_on(x.device());
    const int dt = dtype_of(x);
    const int64_t nvox = voxels(x), batch = x.size(0);
    const auto options = x.options().requires_grad(false);
    const int depth = (int)weights.size();

    const Tensor stack = block.new_stack(x);
    pointwise(x, sw, sb, stack, c_in, stream);     // the scaled input goes straight into the stack
    block.forward(stack, bias, stream);

    // one buffer for all gradients: bias | weights | final weight | final bias (the block adds to
    // its part, which starts at zero; the final layer overwrites its own)
    int64_t hidden = bias.numel();
    for (const Tensor &w : weights) hidden += w.numel();
    const Tensor flat = at::empty({hidden + (c_out * channels + c_out) * (scaled ? 2 : 1)}, options);
    flat.narrow(0, 0, hidden).zero_();
    char *const base = (char *)flat.data_ptr();
    const int64_t el = flat.element_size();
    char *const g_fw = base + hidden * el, *const g_fb = g_fw + c_out * channels * el;
    char *const s_fw = scaled ? g_fb + c_out * el : g_fw, *const s_fb = s_fw + c_out * channels * el;

    Tensor folded;
    const void *w_eff = fw.data_ptr(), *b_eff = fb.data_ptr();
    if (scaled) {
        folded = at::empty({c_out * (channels + 1)}, options);
        char *fp = (char *)folded.data_ptr();
        check(lib.msd_scale_fold(dt, c_out, channels, osw->data_ptr(), osb->data_ptr(), w_eff, b_eff, fp,
                                 fp + c_out * channels * el, stream));
        w_eff = fp;
        b_eff = fp + c_out * channels * el;
    }
    auto out_sizes = x.sizes().vec();
    out_sizes[1] = c_out;
    const Tensor output = at::empty(out_sizes, options), grad_out = at::empty(out_sizes, options);
    const Tensor loss = at::empty({}, options);
    {
        const int64_t need = lib.msd_final_workspace_bytes(dt, batch, channels, c_out, nvox);
        const Tensor ws = workspace(need, x);
        const int64_t osb_ = output.stride(0), osc = output.stride(1);
        check(lib.msd_final_forward_loss(dt, kind, batch, channels, c_out, nvox, stack.data_ptr(), stack.stride(0),
                                         stack.stride(1), w_eff, b_eff, target.data_ptr(),
                                         kind == MSD_LOSS_NLL ? nvox : target.stride(0),
                                         kind == MSD_LOSS_NLL ? 0 : target.stride(1), output.data_ptr(), osb_, osc,
                                         grad_out.data_ptr(), osb_, osc, s_fw, s_fb, loss.data_ptr(), ws.data_ptr(),
                                         need, stream));
    }
    if (scaled)
        check(lib.msd_scale_fold(dt, c_out, channels, osw->data_ptr(), nullptr, s_fw, s_fb, g_fw, g_fb, stream));

    const Tensor grads = block.new_stack(x);
    check(lib.msd_final_backward(dt, batch, channels, c_out, nvox, nullptr, grads.stride(0), grads.stride(1),
                                 grad_out.data_ptr(), grad_out.stride(0), grad_out.stride(1), w_eff, grads.data_ptr(),
                                 grads.stride(0), grads.stride(1), nullptr, nullptr, nullptr, 0, stream));
    std::vector<void *> gw(depth);
    int64_t offset = bias.numel();
    for (int i = 0; i < depth; i++) {
        gw[i] = base + offset * el;
        offset += weights[i].numel();
    }
    {
        const int64_t need = lib.msd_block_workspace_bytes(dt, (int)x.dim() - 2, batch, c_in, depth,
                                                           block.widths.data(), x.sizes().data() + 2);
        const Tensor ws = workspace(need, x);
        check(lib.msd_block_backward(dt, (int)x.dim() - 2, batch, c_in, depth, block.widths.data(),
                                     x.sizes().data() + 2, block.dilations.data(), stack.data_ptr(),
                                     stack.strides().data(), grads.data_ptr(), grads.strides().data(),
                                     block.weights.data(), gw.data(), base, 0, ws.data_ptr(), need, stream));
    }
    bias.mutable_grad() = piece(flat, 0, bias);
    offset = bias.numel();
    for (const Tensor &w : weights) {
        w.mutable_grad() = piece(flat, offset, w);
        offset += w.numel();
    }
    fw.mutable_grad() = piece(flat, hidden, fw);
    fb.mutable_grad() = piece(flat, hidden + fw.numel(), fb);
    return std::make_pair(loss, output);
}

// ---------------------------------------------------------------------------
// Adam on the state that torch.optim.Adam keeps (step, exp_avg, exp_avg_sq per parameter).
// False (and nothing has happened) for a state that the kernel does not take.
// ---------------------------------------------------------------------------

bool adam_step(const std::vector<Tensor> &params, const py::list &states, bool capturable, double lr, double beta1,
               double beta2, double eps)
{
    static PyObject *const k_step = PyUnicode_InternFromString("step");
    static PyObject *const k_avg = PyUnicode_InternFromString("exp_avg");
    static PyObject *const k_sq = PyUnicode_InternFromString("exp_avg_sq");
    if (params.empty() || params.size() != states.size()) return false;
    const Tensor &first = params[0];
    if (!plain(first) || !floating(first)) return false;
    std::vector<msd_adam_param> table;
    std::vector<float *> host_steps;
    std::vector<Tensor> touched;
    table.reserve(params.size());
    for (size_t i = 0; i < params.size(); i++) {
        const Tensor &p = params[i];
        const Tensor &g = p.grad();
        if (!g.defined()) continue;               // torch's optimiser passes it over as well
        PyObject *const entry = PyList_GET_ITEM(states.ptr(), i);
        if (!PyDict_Check(entry)) return false;
        PyObject *ps = PyDict_GetItem(entry, k_step), *pa = PyDict_GetItem(entry, k_avg), *pq = PyDict_GetItem(entry, k_sq);
        if (!ps || !pa || !pq || !THPVariable_Check(ps) || !THPVariable_Check(pa) || !THPVariable_Check(pq)) return false;
        const Tensor &step = THPVariable_Unpack(ps), &avg = THPVariable_Unpack(pa), &sq = THPVariable_Unpack(pq);
        for (const Tensor *t : {&p, &g, &avg, &sq})
            if (!like(*t, first) || !t->is_contiguous() || t->numel() != p.numel()) return false;
        if (step.scalar_type() != at::kFloat || step.numel() != 1 || p.is_inference()) return false;
        msd_adam_param e{p.data_ptr(), g.data_ptr(), avg.data_ptr(), sq.data_ptr(), nullptr, 0.0, p.numel()};
        if (step.is_cuda()) {
            if (step.device() != first.device()) return false;
            e.device_step = step.data_ptr<float>();
        } else if (step.is_cpu() && !capturable) {   // (torch refuses a capturable step counted on the host)
            float *s = step.data_ptr<float>();
            e.step = (double)*s + 1.0;
            host_steps.push_back(s);
        } else {
            return false;
        }
        table.push_back(e);
        touched.push_back(p);
    }
    if (table.empty()) return true;
    const c10::DeviceGuard guard(first.device());
    check(lib.msd_adam_step(dtype_of(first), (int)table.size(), table.data(), lr, beta1, beta2, eps,
                            stream_on(first.device())));
    for (float *s : host_steps) *s += 1.f;
    for (const Tensor &p : touched) p.unsafeGetTensorImpl()->bump_version();
    return true;
}

// Labels limited to [0, num_labels) and their range so far (a tensor of two int64 on the
// device, updated in place), without waiting for the device.
std::optional<Tensor> label_check(const Tensor &labels, int64_t num_labels, const Tensor &range)
{
    if (!plain(labels) || labels.scalar_type() != at::kLong || !labels.is_contiguous() || labels.numel() == 0 ||
        !plain(range) || range.scalar_type() != at::kLong || range.numel() != 2 || !range.is_contiguous() ||
        range.device() != labels.device())
        return std::nullopt;
    const c10::DeviceGuard guard(labels.device());
    at::AutoDispatchBelowADInplaceOrView below;
    const Tensor out = at::empty(labels.sizes(), labels.options());
    check(lib.msd_label_check(labels.numel(), num_labels, labels.data_ptr<int64_t>(), out.data_ptr<int64_t>(),
                              range.data_ptr<int64_t>(), stream_on(labels.device())));
    return out;
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m)
{
    m.def("bind", &bind);
    m.def("conv_layer", &conv_layer);
    m.def("net_forward", &net_forward);
    m.def("train_step", &train_step);
    m.def("adam_step", &adam_step);
    m.def("label_check", &label_check);
}
