"""All gradients of a layer in one pass over its input (up to seven outputs, two in 3D)."""
import pytest
import torch

from parity import captured_kernels, rel_err, same_specials

pytestmark = pytest.mark.gpu


def gradients(x, w, b, g, dilation, relu):
    from msd_pytorch_amd import conv2d, conv3d
    if x.dim() == 4:
        fn = conv2d.conv2d_relu if relu else conv2d.conv2d
    else:
        fn = conv3d.conv3d_relu if relu else conv3d.conv3d
    leaves = [t.detach().clone().requires_grad_() for t in (x, w, b)]
    out = torch.empty_like(g)
    y = fn(*leaves, out, 1, dilation)
    return torch.autograd.grad(y, leaves, g)


def ran_in_one_pass(run):
    """run()'s result, and whether its backward pass was the one that takes all three gradients (its own class of launches)."""
    import ctypes
    from msd_pytorch_amd import _native
    lib = _native.load()
    ms, calls = (ctypes.c_double * 4)(), (ctypes.c_int64 * 4)()
    assert lib.msd_profile_enable(1) == 0
    try:
        result = run()
        assert lib.msd_profile_read(ms, calls) == 0
    finally:
        lib.msd_profile_enable(0)
    return result, calls[3] == 1 and calls[1] == calls[2] == 0


def problem(size, batch, c_in, c_out, seed=11):
    gen = torch.Generator().manual_seed(seed)
    x = torch.randn(batch, c_in, *size, generator=gen).cuda()
    taps = [3] * len(size)
    w = (torch.randn(c_out, c_in, *taps, generator=gen) * (2.0 / (3 ** len(size) * c_in)) ** 0.5).cuda()
    return x, w, (torch.randn(c_out, generator=gen) * 0.1).cuda(), torch.randn(batch, c_out, *size, generator=gen).cuda()


# Blocks of 16 channels that four or two waves share, one and two chunks of the grid, channels at, below and past a
# block; volumes of one segment of 32 voxels, of one more, of fewer than a tile, rows shorter than a segment; a
# dilation of the volume's extent; images that end inside a tile.  Two outputs at any number of channels.  2D: odd rows
# of more than 256 voxels and even ones of more than 512, one to seven outputs, from 64, 40 and 12 channels on, or five
# where the image is of middling size.
CASES = [
    ((2, 4, 4), 1, 16, 1, 1),
    ((3, 1, 11), 2, 16, 1, 1),
    ((5, 7, 9), 3, 33, 1, 5),
    ((4, 6, 32), 1, 16, 1, 4),
    ((6, 5, 45), 2, 64, 1, 2),
    ((3, 4, 33), 1, 80, 1, 3),
    ((9, 11, 13), 2, 1, 2, 9),
    ((4, 5, 70), 1, 17, 2, 1),
    ((7, 6, 40), 2, 40, 2, 3),
    ((3, 5, 37), 1, 130, 2, 2),
    ((40, 33, 35), 1, 20, 2, 10),
    ((3, 257), 2, 1, 1, 3),
    ((9, 259), 1, 17, 2, 1),
    ((5, 514), 2, 33, 1, 5),
    ((7, 1021), 1, 7, 1, 2),
    ((6, 32), 3, 64, 1, 6),
    ((4, 45), 2, 40, 2, 1),
    ((130, 131), 1, 5, 3, 10),
    ((12, 70), 2, 12, 4, 12),
    ((5, 96), 1, 70, 5, 2),
    ((8, 50), 2, 20, 6, 3),
    ((4, 33), 1, 12, 7, 1),
    ((40, 64), 1, 130, 7, 7),
]


@pytest.mark.parametrize("relu", [True, False], ids=["relu", "plain"])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c[0])) + "-B%d-c%d-w%d-d%d" % c[1:])
def test_layer_gradients(case, relu):
    size, batch, c_in, c_out, dilation = case
    tensors = problem(size, batch, c_in, c_out)
    got, in_one_pass = ran_in_one_pass(lambda: gradients(*tensors, dilation, relu))
    assert in_one_pass
    # (double precision goes through the shape-generic kernels; a ReLU that is open in one precision only would show)
    want = gradients(*(t.double() for t in tensors), dilation, relu)
    for a, b in zip(got[:2], want[:2]):
        assert rel_err(a, b) <= 1e-5
    # the bias gradient is a sum of terms of both signs, in chains and trees of fewer than 64 additions here: each
    # rounds to 2^-24 of at most the sum of the terms' sizes
    terms = tensors[3].double().abs().sum(dim=[0, *range(2, tensors[3].dim())])
    assert bool(((got[2] - want[2]).abs() <= 64 * 2.0 ** -24 * terms).all())


# More than the 64 channels of a chunk: side by side in one launch where they make chunks of one size or the image is small, one
# launch after the other where they do not (two blocks, one block and one channel over).
@pytest.mark.parametrize("size, batch, c_in, c_out, launches", [
    ((512, 513), 1, 65, 3, 1), ((512, 513), 1, 130, 2, 1), ((700, 720), 1, 65, 3, 2), ((700, 720), 1, 97, 3, 1), ((900, 1000), 1, 65, 3, 2), ((450, 1001), 2, 97, 7, 2), ((900, 1000), 1, 96, 3, 1),
    ((902, 999), 1, 193, 4, 4), ((98, 97, 97), 1, 65, 2, 2), ((48, 100, 97), 2, 160, 1, 3), ((97, 97, 98), 1, 90, 2, 1)],
    ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else str(v))
def test_layer_gradients_over_several_chunks(size, batch, c_in, c_out, launches):
    tensors = problem(size, batch, c_in, c_out, seed=17)
    torch.cuda.synchronize()
    kernels = captured_kernels(lambda: gradients(*tensors, 3, True))
    assert sum("pull_rows" in name for name, _ in kernels) == launches
    got, in_one_pass = ran_in_one_pass(lambda: gradients(*tensors, 3, True))
    assert in_one_pass
    # (the ReLU as the forward pass in single precision found it: one that is open in one precision only would show)
    from msd_pytorch_amd import conv2d, conv3d
    x, w, b, g = tensors
    open_relu = (conv2d.conv2d_relu if len(size) == 2 else conv3d.conv3d_relu)(x, w, b, torch.empty_like(g), 1, 3) > 0
    want = gradients(x.double(), w.double(), b.double(), (g * open_relu).double(), 3, False)
    for a, b in zip(got[:2], want[:2]):
        assert rel_err(a, b) <= 1e-5
    # the sums over voxels: chains of 1/256 of the tiles, then trees, as terms of both signs; each addition rounds to 2^-24 of at
    # most the sum of the terms' sizes
    terms = g.double().abs().sum(dim=[0, *range(2, g.dim())])
    assert bool(((got[2] - want[2]).abs() <= 64 * 2.0 ** -24 * terms).all())


@pytest.mark.parametrize("where", ["input", "gradient", "weight"])
@pytest.mark.parametrize("value", [float("inf"), float("-inf"), float("nan"), 3.4e38])
@pytest.mark.parametrize("size", [(5, 6, 37), (13, 259)], ids=str)
def test_values_without_bf16_parts(size, where, value):
    from msd_pytorch_amd import _native
    lib = _native.load()
    x, w, b, g = problem(size, 2, 33, 2, seed=13)
    x, w, g = x.abs() * 1e-3 + 1e-3, w.abs() * 1e-3 + 1e-4, g.abs() * 1e-3 + 1e-4      # (every ReLU open, sums of one sign)
    {"input": x, "gradient": g, "weight": w}[where].view(-1)[777 % (w.numel() if where == "weight" else g.numel())] = value
    found = []
    for path in (1, 0):
        assert lib.msd_set_kernel_path(path) == 0
        try:
            result, in_one_pass = ran_in_one_pass(lambda: gradients(x, w, b + 1, g, 2, True))
            found.append(result)
            assert in_one_pass == (path == 0)
        finally:
            lib.msd_set_kernel_path(0)
    for want, got in zip(*found):
        assert same_specials(got, want)
        finite = torch.isfinite(want)
        assert not bool(finite.any()) or rel_err(got[finite], want[finite]) <= 1e-4
