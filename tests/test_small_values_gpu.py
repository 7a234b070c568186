"""Values near the lower end of the fp32 range keep all their bits in the passes that take fp32 products in bf16 parts.

Each operand in turn is scaled by 2^-122 (values of 2^-116 down to 2^-149, the bits of the latter included), or the left half of
an image whose right half is of the usual size.  The results are as exact as elsewhere: against double precision, with the
tolerance of ordinary values; what is below 2^-149 is at most 2^-22 of them."""
import pytest
import torch

from cases import rel_err
from test_knobs_gpu import tuning

pytestmark = pytest.mark.gpu

SCALE = 2.0 ** -122
HALF, REACH = 48, 24                              # columns of the left half, of it what no value of the right half reaches


def error(got, want):
    return rel_err(got.double() / SCALE, want.double() / SCALE)


def scaled(t, where, operand):
    """t, or what the case makes of the operand of that name."""
    if where == operand:
        return t * SCALE
    if where == operand + ", left half":
        t = t.clone()
        t[..., :HALF] *= SCALE
    return t


@pytest.mark.parametrize("size,depth", [((9, 96), 6), ((9, 96), 14), ((5, 6, 96), 2), ((5, 6, 96), 4)],
                         ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else "depth%d" % v)
@pytest.mark.parametrize("where", ["gradient", "gradient, left half", "stack", "weights"])
def test_backward_groups(where, size, depth):
    from msd_pytorch_amd import msd_custom_convolutions as cc
    gen = torch.Generator().manual_seed(83)
    c_in, dilations = 5, [1 + i % 2 for i in range(depth)]
    stack = scaled(torch.rand(2, c_in + depth, *size, generator=gen) + 0.1, where, "stack")         # every ReLU open
    gradient = torch.randn(2, c_in + depth, *size, generator=gen)
    if where == "weights":
        gradient[:, :-1] = 0                      # (else the results are sums of values of the usual size)
    gradient = scaled(gradient, where, "gradient")
    weights = [scaled(torch.randn(1, c_in + i, *[3] * len(size), generator=gen) * 0.1, where, "weights") for i in range(depth)]
    found = []
    for dtype in (torch.float32, torch.float64):
        s, g = stack.cuda().to(dtype), gradient.cuda().to(dtype)
        w = [k.cuda().to(dtype) for k in weights]
        gk, gb = [torch.zeros_like(k) for k in w], torch.zeros(depth, dtype=dtype).cuda()
        with tuning({"bwd.group": 1}):
            cc.block_backward(s, g, c_in, dilations, w, gk, gb, True)
        found.append((g[:, :c_in], *gk))
    if where.endswith("left half"):
        assert error(found[0][0][..., :REACH], found[1][0][..., :REACH]) <= 1e-5
        return
    # (weights: the gradients of all but the uppermost layer's are of the size of 2^-122, too)
    for got, want in zip(*found):
        assert error(got, want) <= 1e-5


@pytest.mark.parametrize("size", [(5, 6, 37), (13, 259)], ids=str)
@pytest.mark.parametrize("where", ["gradient", "input", "weight"])
def test_layer_gradients_in_one_pass(where, size):
    from test_layer_pass_gpu import gradients, problem, ran_in_one_pass
    x, w, b, g = problem(size, 2, 33, 2, seed=89)
    x, w, g = scaled(x, where, "input"), scaled(w, where, "weight"), scaled(g, where, "gradient")
    got, in_one_pass = ran_in_one_pass(lambda: gradients(x, w, b, g, 2, False))
    assert in_one_pass
    want = gradients(x.double(), w.double(), b.double(), g.double(), 2, False)
    for a, c in zip(got[:2], want[:2]):
        assert error(a, c) <= 1e-5


@pytest.mark.parametrize("c_in", [33, 140], ids="c{}".format)
@pytest.mark.parametrize("where", ["input", "input, left half", "weights"])
def test_forward_groups_of_fourteen(where, c_in):
    from msd_pytorch_amd import msd_custom_convolutions as cc
    gen = torch.Generator().manual_seed(97)
    depth, size = 14, (7, 96)
    image = scaled(torch.randn(1, c_in, *size, generator=gen), where, "input")
    weights = [scaled(torch.randn(1, c_in + i, 3, 3, generator=gen) * 0.05, where, "weights") for i in range(depth)]
    found = []
    for dtype in (torch.float32, torch.float64):
        stack = torch.empty(1, c_in + depth, *size, device="cuda", dtype=dtype)
        stack[:, :c_in] = image.cuda().to(dtype)
        with tuning({"fwd.group": 1024}):
            cc.block_forward(stack, c_in, [1 + i % 2 for i in range(depth)], torch.zeros(depth, device="cuda", dtype=dtype),
                             [w.cuda().to(dtype) for w in weights])
        found.append(stack[:, c_in:])
    columns = REACH if where.endswith("left half") else size[1]
    assert error(found[0][..., :columns], found[1][..., :columns]) <= 1e-5


# The same pass takes a tile that holds a value of 2^36 = 6.9e10 or more whole: at the line, just past it and far past it, with values
# of 2^-122 in the same tile.
LARGE = [6.8e10, 7e10, 1e30]


@pytest.mark.parametrize("size,depth", [((9, 96), 6), ((9, 96), 14), ((5, 6, 96), 4)],
                         ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else "depth%d" % v)
@pytest.mark.parametrize("where", ["gradient", "stack", "weights"])
@pytest.mark.parametrize("value", LARGE)
def test_backward_groups_with_a_large_value(value, where, size, depth):
    from msd_pytorch_amd import msd_custom_convolutions as cc
    gen = torch.Generator().manual_seed(101)
    c_in, dilations, last = 5, [1 + i % 2 for i in range(depth)], 92
    stack = torch.rand(1, c_in + depth, *size, generator=gen) + 0.1
    gradient = scaled(torch.randn(1, c_in + depth, *size, generator=gen), "gradient, left half", "gradient")
    weights = [torch.randn(1, c_in + i, *[3] * len(size), generator=gen) * 0.1 for i in range(depth)]
    if where == "stack":
        stack[0, 3, ..., last] = value
    elif where == "gradient":
        gradient[0, -1, ..., last] = value
    else:
        weights[-1].view(-1)[4] = value
    found = []
    for dtype in (torch.float32, torch.float64):
        s, g = stack.cuda().to(dtype), gradient.cuda().to(dtype)
        w = [k.cuda().to(dtype) for k in weights]
        gk, gb = [torch.zeros_like(k) for k in w], torch.zeros(depth, dtype=dtype).cuda()
        with tuning({"bwd.group": 1}):
            cc.block_backward(s, g, c_in, dilations, w, gk, gb, True)
        found.append((g[:, :c_in], *gk))
    assert error(found[0][0][..., :REACH], found[1][0][..., :REACH]) <= 1e-5
    for got, want in zip(*found):
        assert error(got, want) <= 1e-5


def test_products_of_values_at_the_line_fit():
    from test_layer_pass_gpu import gradients, problem
    x, w, b, g = (6.8e10 * (0.5 + 0.5 * torch.rand_like(t)) for t in problem((13, 259), 2, 33, 2))
    got = gradients(x, w, b, g, 2, False)
    want = gradients(x.double(), w.double(), b.double(), g.double(), 2, False)
    for a, c in zip(got[:2], want[:2]):
        assert error(a, c) <= 1e-5


@pytest.mark.parametrize("where", ["input", "weights"])
@pytest.mark.parametrize("value", LARGE)
def test_forward_groups_with_a_large_value(value, where):
    from msd_pytorch_amd import msd_custom_convolutions as cc
    gen = torch.Generator().manual_seed(103)
    c_in, depth, size = 45, 9, (7, 96)
    image = scaled(torch.rand(1, c_in, *size, generator=gen), "input, left half", "input")
    weights = [torch.rand(1, c_in + i, 3, 3, generator=gen) * 0.05 for i in range(depth)]
    if where == "input":
        image[0, 40, :, 92] = value
    else:
        weights[-1].view(-1)[4] = value
    found = []
    for dtype in (torch.float32, torch.float64):
        stack = torch.empty(1, c_in + depth, *size, device="cuda", dtype=dtype)
        stack[:, :c_in] = image.cuda().to(dtype)
        with tuning({"fwd.group": 1024}):
            cc.block_forward(stack, c_in, [1 + i % 2 for i in range(depth)], torch.zeros(depth, device="cuda", dtype=dtype),
                             [w.cuda().to(dtype) for w in weights])
        found.append(stack[:, c_in:])
    for layer in range(depth):
        for columns in (REACH, size[1]):
            assert error(found[0][:, layer, :, :columns], found[1][:, layer, :, :columns]) <= 1e-5
