"""The native host path (csrc/host/msd_host.cpp) against the Python path it stands in for: the
same launches, so the same bits where nothing but the route differs."""
import pytest
import torch

from parity import bias_close, rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ndim,size,c_in,c_out,dilation,dtype", [
    (2, (1, 5), 1, 1, 1, torch.float32),           # rows too short for the row kernels
    (2, (96, 96), 12, 1, 3, torch.float32),
    (2, (33, 130), 17, 2, 10, torch.float32),
    (2, (40, 64), 5, 5, 2, torch.float32),         # output channels two at a time
    (3, (8, 9, 33), 3, 1, 2, torch.float32),
    (3, (6, 7, 64), 16, 3, 1, torch.float32),
    (2, (9, 11), 2, 2, 4, torch.float64),
    (3, (5, 6, 7), 2, 1, 2, torch.float64),
])
@pytest.mark.parametrize("relu", [True, False])
def test_a_layer_overwrites_what_the_operators_add_to_zeros(ndim, size, c_in, c_out, dilation, dtype, relu):
    from msd_pytorch_amd import conv2d, conv3d
    function = {(2, True): conv2d.Conv2dReluFunction, (2, False): conv2d.Conv2dFunction,
                (3, True): conv3d.Conv3DReluFunction, (3, False): conv3d.Conv3DFunction}[ndim, relu]
    native = {(2, True): conv2d.conv2d_relu, (2, False): conv2d.conv2d,
              (3, True): conv3d.conv3d_relu, (3, False): conv3d.conv3d}[ndim, relu]
    gen = torch.Generator().manual_seed(7)
    x = torch.randn(2, c_in, *size, generator=gen, dtype=dtype).cuda().requires_grad_()
    w = torch.randn(c_out, c_in, *([3] * ndim), generator=gen, dtype=dtype).cuda().requires_grad_()
    b = torch.randn(c_out, generator=gen, dtype=dtype).cuda().requires_grad_()
    g = torch.randn(2, c_out, *size, generator=gen, dtype=dtype).cuda()
    results = []
    for apply in (native, function.apply):
        # memory that the gradients will be allocated from holds something else than zeros
        dirty = [torch.full_like(t, 7.0) for t in (x, w, b)]
        del dirty
        out = torch.empty_like(g)
        y = apply(x, w, b, out, 1, dilation)
        assert y.data_ptr() == out.data_ptr()
        results.append([y.detach().clone(), *torch.autograd.grad(y, (x, w, b), g)])
    for got, want in zip(*results):
        # one rounding more or less where a gradient is added to a zero that was stored before
        assert rel_err(got, want) <= (1e-6 if dtype == torch.float32 else 1e-14)
    # only what is asked for
    y = native(x.detach(), w, b, torch.empty_like(g), 1, dilation)
    only = torch.autograd.grad(y, (b,), g)
    # (the bias gradient alone is summed by another kernel, in another order)
    terms = g * (y.detach() > 0) if relu else g
    assert bias_close(only[0], results[1][3].cpu(), terms.cpu(), tol=1e-4 if dtype == torch.float32 else 1e-12)


def test_a_layer_raises_like_the_operators():
    from msd_pytorch_amd.conv2d import conv2d_relu
    x, w, b = torch.zeros(1, 2, 4, 4).cuda(), torch.zeros(1, 2, 3, 3).cuda(), torch.zeros(1).cuda()
    with pytest.raises(RuntimeError, match="Dilation cannot be greater"):
        conv2d_relu(x, w, b, torch.zeros(1, 1, 4, 4).cuda(), 1, 5)
    with pytest.raises(RuntimeError, match="same type"):
        conv2d_relu(x, w.double(), b, torch.zeros(1, 1, 4, 4).cuda(), 1, 1)


def _models(task, ndim, depth, width, c_out, count):
    from msd_pytorch_amd import MSDRegressionModel, MSDSegmentationModel
    models = []
    for _ in range(count):
        torch.manual_seed(3)
        if task == "labels":
            m = MSDSegmentationModel(2, c_out, depth, width, dilations=[1, 2, 3], ndim=ndim)
        else:
            m = MSDRegressionModel(2, c_out, depth, width, dilations=[1, 2, 3], loss=task, ndim=ndim)
            m.scale_out.weight.data += 0.3 * torch.randn_like(m.scale_out.weight)
            m.scale_out.bias.data += 0.7
        m.scale_in.weight.data *= 1.7
        m.scale_in.bias.data -= 0.2
        m.msd.final_layer.linear.weight.data.normal_(0, 0.2)
        models.append(m)
    return models


@pytest.mark.parametrize("task,ndim,size,depth,width,c_out", [
    ("L2", 2, (20, 65), 4, 1, 1), ("L1", 2, (32, 64), 5, 2, 3), ("labels", 2, (31, 40), 6, 1, 4),
    ("L2", 3, (6, 9, 36), 4, 1, 2), ("labels", 3, (5, 7, 33), 3, 2, 2),
    ("L2", 2, (16, 64), 62, 1, 1),                 # more parameters than one launch of the optimiser takes
])
def test_training_steps_follow_the_autograd_path(task, ndim, size, depth, width, c_out):
    native, general = _models(task, ndim, depth, width, c_out, 2)
    general._native_step = lambda: False
    general._native_adam = lambda: False
    gen = torch.Generator().manual_seed(5)
    for step in range(3):
        x = torch.randn(2, 2, *size, generator=gen).cuda()
        t = torch.randint(0, c_out, (2, 1, *size), generator=gen).cuda() if task == "labels" \
            else torch.randn(2, c_out, *size, generator=gen).cuda()
        losses = [m.learn(x, t) for m in (native, general)]
        assert abs(losses[0] - losses[1]) <= 1e-5 * abs(losses[1])
        assert native.loss.grad_fn is None and general.loss.grad_fn is not None
        assert rel_err(native.output, general.output) <= 1e-4
        for p, q in zip(native.msd.parameters(), general.msd.parameters()):
            # Adam's first steps are lr * sign(gradient): a rounding of a gradient near zero may
            # move its parameter by up to lr, so the parameters are copied over for the next step
            assert p.grad.shape == q.grad.shape and rel_err(p.grad, q.grad) <= 1e-4
            state, want = native.optimizer.state[p], general.optimizer.state[q]
            assert float(state["step"]) == float(want["step"]) == step + 1
            assert rel_err(state["exp_avg"], want["exp_avg"]) <= 1e-4
            assert rel_err(state["exp_avg_sq"], want["exp_avg_sq"]) <= 2e-4
            assert float((p.detach() - q.detach()).abs().max()) <= 2.1e-3
            p.data.copy_(q.data)


def test_what_the_native_step_leaves_to_the_general_path():
    (model,) = _models("L2", 2, 3, 1, 1, 1)
    x, t = torch.rand(1, 2, 24, 40).cuda(), torch.rand(1, 1, 24, 40).cuda()
    model.learn(x, t)
    assert model.loss.grad_fn is None
    seen = []
    handle = model.msd.msd_block.weight1.register_hook(lambda g: seen.append(tuple(g.shape)))
    model.learn(x, t)                              # a watched parameter
    assert seen == [(1, 3, 3, 3)] and model.loss.grad_fn is not None
    handle.remove()
    model.optimizer = torch.optim.SGD(list(model.msd.parameters())[:2], lr=0.1)
    before = model.msd.final_layer.linear.weight.detach().clone()
    model.learn(x, t)                              # an optimiser of some of the parameters
    assert model.loss.grad_fn is not None and torch.equal(before, model.msd.final_layer.linear.weight)
    model.optimizer = torch.optim.Adam(model.msd.parameters(), weight_decay=0.1)
    model.learn(x, t)
    scheduler = torch.optim.lr_scheduler.StepLR(model.optimizer, 1)
    assert not model._native_adam()                # weight decay, and a scheduler's own step
    model.learn(x, t)
    scheduler.step()


@pytest.mark.parametrize("count", [1, 63, 1000, 300001])
def test_label_check(count):
    from msd_pytorch_amd import _native
    gen = torch.Generator().manual_seed(count)
    labels = torch.randint(-3, 9, (count,), generator=gen).cuda()
    seen = torch.tensor([2, 4]).cuda()
    out = _native.host().label_check(labels, 6, seen)
    assert torch.equal(out, labels.clamp(0, 5))
    assert seen.tolist() == [min(2, int(labels.min())), max(4, int(labels.max()))]


@pytest.mark.parametrize("count", [(1 << 18) - 1, (1 << 18) + 1, (1 << 20) + 1])
def test_label_check_of_whole_images(count):
    """A grid of labels less and more one, and one more than the grid takes in one round."""
    from msd_pytorch_amd import _native
    labels = torch.randint(0, 5, (count,), generator=torch.Generator().manual_seed(count))
    labels[count - 1], labels[count // 2] = -7, 12
    seen = torch.tensor([2, 4]).cuda()
    out = _native.host().label_check(labels.cuda(), 5, seen)
    assert torch.equal(out.cpu(), labels.clamp(0, 4)) and seen.tolist() == [-7, 12]


@pytest.mark.parametrize("ndim,size", [(2, (30, 70)), (3, (5, 8, 40))])
def test_prediction_without_gradients_equals_the_differentiable_pass(ndim, size):
    (model,) = _models("L2", ndim, 5, 1, 3, 1)
    x = torch.rand(2, 2, *size).cuda()
    with torch.no_grad():
        got = model.net(x)
    want = model.net(x)
    assert want.requires_grad and torch.equal(got, want.detach())


@pytest.mark.parametrize("ndim,size,depth,width", [(2, (512, 512), 9, 1), (2, (256, 1024), 4, 2), (3, (64, 64, 64), 4, 1)])
def test_planes_of_whole_64_kilobytes(ndim, size, depth, width):
    """The native calls keep the channels of such stacks a little apart; the general path does not.
    The launches and their order of summation are the same."""
    native, general = _models("L2", ndim, depth, width, 2, 2)
    general._native_step = lambda: False
    gen = torch.Generator().manual_seed(11)
    x, t = torch.randn(2, 2, *size, generator=gen).cuda(), torch.randn(2, 2, *size, generator=gen).cuda()
    with torch.no_grad():
        got = native.net(x)
    assert torch.equal(got, general.net(x).detach())
    for m in (native, general):
        m.learn(x, t)
    assert native.loss.grad_fn is None and general.loss.grad_fn is not None
    assert rel_err(native.output, general.output) <= 1e-5
    for p, q in zip(native.msd.parameters(), general.msd.parameters()):
        assert rel_err(p.grad, q.grad) <= 1e-4


def _optimised(dtype, capturable, count, seed):
    """A model that is nothing but an Adam over `count` parameters, a thousand steps old."""
    from msd_pytorch_amd.msd_model import MSDModel
    gen = torch.Generator().manual_seed(seed)
    sizes = [1, 3, 63, 64, 65, 257, 1000, 4099]

    def draw(n):
        return torch.randn(n, generator=gen, dtype=dtype).cuda()

    params = [torch.nn.Parameter(0.01 * draw(sizes[i % len(sizes)])) for i in range(count)]
    model = MSDModel.__new__(MSDModel)
    model.optimizer = torch.optim.Adam(params, lr=2e-3, betas=(0.8, 0.99), eps=1e-6, capturable=capturable)
    for p in params:
        step = torch.tensor(1000.0)
        model.optimizer.state[p] = {"step": step.cuda() if capturable else step, "exp_avg": 1e-3 * draw(p.numel()),
                                    "exp_avg_sq": 1e-6 * (0.1 + draw(p.numel()).abs())}
    return model, params, [[1e-3 * draw(p.numel()) for p in params] for _ in range(5)]


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("capturable", [False, True])
@pytest.mark.parametrize("count", [1, 13, 130])    # 130: more than one launch takes
def test_the_optimiser_in_one_launch_is_torchs(dtype, capturable, count):
    """Moments of a thousand steps, so that an update is a value and not a sign; then the state is
    dropped, replaced in part and as a whole.  Both sides do the same arithmetic in some order, so
    that they are a few roundings apart; but torch forms 1 - beta ** step of a step on the device in 32
    bits whatever the type, which is 6e-8 of the 0.01 of a first step, or 6e-6 of the update."""
    tol = 1e-6 if dtype == torch.float32 else 1e-14
    update_tol = max(tol, 1e-5 if capturable else 0.0)
    native, ours, grads = _optimised(dtype, capturable, count, 9)
    torchs, theirs, _ = _optimised(dtype, capturable, count, 9)
    launched = []

    def drop(model, params, which):
        state = model.optimizer.state
        if which == 2:
            state.clear()
        elif which == 3:
            del state[params[0]]
        elif which == 4:
            state[params[-1]] = {k: v.clone() for k, v in state[params[-1]].items()}

    for i, step in enumerate(grads):
        for model, params in ((native, ours), (torchs, theirs)):
            drop(model, params, i)
            before = [p.detach().clone() for p in params]
            for p, g in zip(params, step):
                p.grad = g.clone()
            if model is native:
                launched.append(model._native_adam())
                if not launched[-1]:
                    model.optimizer.step()
            else:
                model.optimizer.step()
        for p, q, old in zip(ours, theirs, before):
            state, want = native.optimizer.state[p], torchs.optimizer.state[q]
            assert float(state["step"]) == float(want["step"])
            assert rel_err(state["exp_avg"], want["exp_avg"]) <= tol
            assert rel_err(state["exp_avg_sq"], want["exp_avg_sq"]) <= tol
            moved = float((q.detach() - old).abs().max())
            assert float((p - q).detach().abs().max()) <= tol * float(q.detach().abs().max()) + update_tol * moved
            assert moved > 0
    # torch makes what is missing
    assert launched == [True, True, False, False, True]


def test_prediction_where_a_weight_is_not_a_parameter_of_its_module():
    """Replicas of nn.DataParallel hold plain tensors, parametrized modules compute theirs."""
    (model,) = _models("L2", 2, 4, 1, 2, 1)
    x, t = torch.rand(2, 2, 24, 40).cuda(), torch.rand(2, 2, 24, 40).cuda()
    with torch.no_grad():
        want = model.net(x)
        replica = torch.nn.parallel.replicate(model.net, [torch.device("cuda", 0)], detach=True)[0]
        copy = replica[1].msd_block
        assert copy is not model.msd.msd_block
        for name in copy.weight_names:             # (a replica on the module's own device keeps its parameters)
            tensor = copy._parameters.pop(name).detach().clone()
            setattr(copy, name, tensor)
        assert torch.equal(replica(x), want)

    class Half(torch.nn.Module):
        def forward(self, w):
            return 0.5 * w

    block = model.msd.msd_block
    original = block.weight1.detach().clone()
    torch.nn.utils.parametrize.register_parametrization(block, "weight1", Half())
    with torch.no_grad():
        block.parametrizations.weight1.original.mul_(2)
        assert torch.equal(model.net(x), want)
    model.learn(x, t)                              # (the parameter behind the weight is the one that is trained)
    assert model.loss.grad_fn is not None
    assert not torch.equal(0.5 * block.parametrizations.weight1.original.detach(), original)


def test_a_trace_does_not_hold_the_example_output():
    """A layer is recorded as a call; a network cannot be traced (sizes are tensors then) and says so."""
    from msd_pytorch_amd.conv2d import conv2d_relu
    (model,) = _models("L2", 2, 3, 1, 1, 1)
    x, other = torch.rand(1, 2, 24, 40).cuda(), torch.rand(1, 2, 24, 40).cuda()
    w, b = torch.randn(1, 2, 3, 3).cuda(), torch.randn(1).cuda()

    def layer(x):
        return conv2d_relu(x, w, b, torch.empty(1, 1, 24, 40, device="cuda"), 1, 2)

    with torch.no_grad():
        traced = torch.jit.trace(layer, (x,), check_trace=False)
        assert torch.equal(traced(other), layer(other))
        with pytest.raises(RuntimeError):
            torch.jit.trace(model.net, (x,), check_trace=False)


def test_a_tangent_is_not_dropped():
    """No forward mode: the autograd functions say so, and so do the calls that stand in for them."""
    import torch.autograd.forward_ad as fwd
    from msd_pytorch_amd.conv2d import conv2d_relu
    (model,) = _models("L2", 2, 3, 1, 1, 1)
    x, w, b = torch.rand(1, 2, 24, 40).cuda(), torch.randn(1, 2, 3, 3).cuda(), torch.randn(1).cuda()
    out = torch.empty(1, 1, 24, 40).cuda()
    with fwd.dual_level(), torch.no_grad():
        for i in range(3):
            args = [x, w, b]
            args[i] = fwd.make_dual(args[i], torch.ones_like(args[i]))
            with pytest.raises(NotImplementedError):
                conv2d_relu(*args, out, 1, 2)
        with pytest.raises(NotImplementedError):
            model.msd(fwd.make_dual(x, torch.ones_like(x)))
        weights = dict(model.msd.named_parameters())
        weights["msd_block.weight1"] = fwd.make_dual(weights["msd_block.weight1"], torch.ones(1, 3, 3, 3).cuda())
        with pytest.raises(NotImplementedError):
            torch.func.functional_call(model.msd, weights, (x,))


def test_an_optimiser_with_a_zero_grad_of_its_own():
    class Accumulating(torch.optim.Adam):
        def zero_grad(self, set_to_none=True):
            pass

    (model,) = _models("L2", 2, 3, 1, 1, 1)
    x, t = torch.rand(1, 2, 24, 40).cuda(), torch.rand(1, 1, 24, 40).cuda()
    model.gradients(x, t)
    once = [p.grad.clone() for p in model.msd.parameters()]
    plain = model.optimizer

    def replaced():
        model.optimizer = torch.optim.Adam(model.msd.parameters())
        model.optimizer.zero_grad = lambda set_to_none=True: None

    def subclass():
        model.optimizer = Accumulating(model.msd.parameters())

    class Wrapper:                                 # zero_grad and step are all that a step needs
        def zero_grad(self):
            plain.zero_grad()

        def step(self):
            plain.step()

    for change in (replaced, subclass):
        plain.zero_grad()
        change()
        for _ in range(2):
            model.gradients(x, t)
        for p, g in zip(model.msd.parameters(), once):
            assert rel_err(p.grad, 2 * g) <= 1e-5
    model.optimizer = Wrapper()
    before = model.msd.msd_block.bias.detach().clone()
    model.learn(x, t)
    assert not torch.equal(before, model.msd.msd_block.bias)
    assert rel_err(model.msd.msd_block.weight1.grad, once[2]) <= 1e-5


def test_a_training_step_under_watch_goes_through_autograd():
    """Saved-tensor hooks and anomaly detection see the autograd graph, so there has to be one."""
    (model,) = _models("L2", 2, 3, 1, 1, 1)
    x, t = torch.rand(1, 2, 24, 40).cuda(), torch.rand(1, 1, 24, 40).cuda()
    packed = []
    with torch.autograd.graph.saved_tensors_hooks(lambda s: packed.append(s.shape) or s, lambda s: s):
        model.learn(x, t)
    assert packed
    with torch.autograd.detect_anomaly(check_nan=True), pytest.raises(RuntimeError, match="nan"):
        model.learn(torch.full_like(x, float("nan")), t)
    seen = []
    handle = torch.nn.modules.module.register_module_forward_hook(lambda m, i, o: seen.append(m))
    try:
        model.learn(x, t)
    finally:
        handle.remove()
    assert model.scale_in in seen


@pytest.mark.parametrize("gradients", [False, True])
def test_a_forward_pass_that_has_no_room_for_the_planes_of_its_groups(gradients):
    """Up to 21 channels of the stack's size for a while; without them the layers run one by one."""
    (model,) = _models("L2", 2, 20, 1, 1, 1)
    x = torch.rand(1, 2, 1024, 1024).cuda()
    with torch.set_grad_enabled(gradients):
        want = model.net(x).detach().clone()
        torch.cuda.synchronize()
        torch.cuda.empty_cache()
        plane = x.numel() // 2 * 4
        # stack, scaled input, output and half the planes, in a pool of their own: what earlier tests left
        # in the allocator's segments does not count
        room = torch.cuda.memory_reserved() + plane * (22 + 2 + 2 + 10)
        total, pool = torch.cuda.get_device_properties(0).total_memory, torch.cuda.MemPool()
        torch.cuda.set_per_process_memory_fraction(room / total)
        try:
            with torch.cuda.use_mem_pool(pool):
                got = model.net(x).detach()
        finally:
            torch.cuda.set_per_process_memory_fraction(1.0)
        got = got.clone()
    assert not torch.equal(got, want)              # (another order of summation)
    assert rel_err(got, want) <= 1e-5


@pytest.mark.parametrize("host", ["native", "python"])
def test_a_forward_pass_with_room_for_groups_of_seven_only(host):
    """Where the 42 planes of groups of fourteen are not to be had, the 21 of groups of seven are asked for."""
    from msd_pytorch_amd import msd_custom_convolutions as cc
    from test_knobs_gpu import tuning
    gen = torch.Generator().manual_seed(7)
    c_in, depth, size = 12, 14, (1024, 1024)
    image = torch.rand(1, c_in, *size, generator=gen).cuda()
    weights = [(torch.randn(1, c_in + i, 3, 3, generator=gen) * 0.1).cuda() for i in range(depth)]
    bias, dilations = torch.zeros(depth).cuda(), [1 + i % 10 for i in range(depth)]
    final_w, final_b = torch.randn(1, c_in + depth, 1, 1, generator=gen).cuda(), torch.zeros(1).cuda()

    def result():
        if host == "native":
            from msd_pytorch_amd import _native
            return _native.host().net_forward(image, bias, weights, dilations, final_w, final_b)
        stack = torch.empty(1, c_in + depth, *size, device="cuda")
        stack[:, :c_in] = image
        cc.block_forward(stack, c_in, dilations, bias, weights)
        return stack

    with tuning({"fwd.group": 12}):
        sevens = result()
    with tuning({"fwd.group": 0}):
        one_by_one = result()
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    plane = size[0] * size[1] * 4
    room = torch.cuda.memory_reserved() + plane * (c_in + depth + 2 + 30)
    total, pool = torch.cuda.get_device_properties(0).total_memory, torch.cuda.MemPool()
    torch.cuda.set_per_process_memory_fraction(room / total)
    try:
        with torch.cuda.use_mem_pool(pool), tuning({"fwd.group": 1024 + 12}):
            got = result()
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    got = got.clone()
    assert not torch.equal(got, one_by_one)
    assert torch.equal(got, sevens)


@pytest.mark.filterwarnings("ignore:Using a target size")
def test_a_target_of_another_shape_is_left_to_the_criterion():
    (model,) = _models("L2", 2, 3, 1, 1, 1)
    model.set_input(torch.rand(2, 2, 24, 40).cuda())
    for target in (torch.tensor(0.5), torch.rand(40), torch.rand(1, 1, 24, 40)):
        model.target = target.cuda()
        loss = model.learn()
        assert abs(loss - float(((model.output - model.target) ** 2).mean())) <= 1e-5 * loss


@pytest.mark.parametrize("path", ["layer", "prediction", "step"])
def test_native_calls_run_on_the_current_stream(path):
    """The input arrives late on a stream of its own: work on any other stream would miss it."""
    from msd_pytorch_amd.conv2d import conv2d_relu
    (model,) = _models("L2", 2, 9, 1, 1, 1)
    value, t = torch.rand(1, 2, 64, 96).cuda(), torch.rand(1, 1, 64, 96).cuda()
    w, b = torch.randn(1, 2, 3, 3).cuda().requires_grad_(), torch.randn(1).cuda().requires_grad_()

    def run(x):
        if path == "layer":
            leaf = x.requires_grad_()
            y = conv2d_relu(leaf, w, b, torch.empty_like(t), 1, 3)
            return [y.detach(), *torch.autograd.grad(y, (leaf, w, b), t)]
        if path == "prediction":
            with torch.no_grad():
                return [model.net(x)]
        model.step_async(x, t, update=False)
        assert model.loss.grad_fn is None
        return [model.loss, model.output, *(p.grad for p in model.msd.parameters())]

    want = [r.clone() for r in run(value.clone())]
    side, late = torch.cuda.Stream(), torch.zeros_like(value)
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        torch.cuda._sleep(50_000_000)              # some 20 ms
        late.copy_(value)
        got = run(late)
        assert not side.query()                    # (nothing has waited)
    side.synchronize()
    for a, c in zip(got, want):
        assert torch.equal(a, c)


def test_a_capturable_optimiser_with_its_counts_on_the_host_is_refused():
    (model,) = _models("L2", 2, 3, 1, 1, 1)
    x, t = torch.rand(1, 2, 24, 40).cuda(), torch.rand(1, 1, 24, 40).cuda()
    model.learn(x, t)
    model.learn(x, t)
    model.optimizer.param_groups[0]["capturable"] = True
    with pytest.raises(AssertionError, match="capturable"):
        model.learn(x, t)


def test_autocast_acts_as_on_the_autograd_path():
    (model,) = _models("L2", 2, 3, 1, 1, 1)
    (labels,) = _models("labels", 2, 3, 1, 4, 1)
    x, t = torch.rand(1, 2, 24, 40).cuda(), torch.rand(1, 1, 24, 40).cuda()
    y = torch.randint(0, 4, (1, 1, 24, 40)).cuda()
    want = labels.gradients(x, y)
    with torch.autocast("cuda", dtype=torch.float16):
        with pytest.raises(RuntimeError, match="same type"):
            model.learn(x, t)
        assert abs(labels.gradients(x, y) - want) <= 1e-5 * want and labels.loss.grad_fn is not None


@pytest.mark.parametrize("task,ndim,size,c_out", [("L2", 2, (20, 33), 3), ("labels", 3, (5, 7, 9), 2)])
def test_a_training_step_in_double_precision(task, ndim, size, c_out):
    native, general = _models(task, ndim, 5, 1, c_out, 2)
    general._native_step = lambda: False
    gen = torch.Generator().manual_seed(6)
    x = torch.randn(2, 2, *size, generator=gen, dtype=torch.float64).cuda()
    t = torch.randint(0, c_out, (2, 1, *size), generator=gen).cuda() if task == "labels" \
        else torch.randn(2, c_out, *size, generator=gen, dtype=torch.float64).cuda()
    for m in (native, general):
        m.net.double()
        m.gradients(x, t)
    assert native.loss.grad_fn is None and general.loss.grad_fn is not None
    assert abs(float(native.loss) - float(general.loss)) <= 1e-13 * float(general.loss)
    assert rel_err(native.output, general.output) <= 1e-13
    for p, q in zip(native.msd.parameters(), general.msd.parameters()):
        assert rel_err(p.grad, q.grad) <= 1e-12
