"""Groups of layers of a 2D block on the matrix cores, forced on small images, against the oracle."""
import pytest
import torch

from parity import block_problem, captured_kernels, check_block, rel_err, same_specials
from test_knobs_gpu import tuning

pytestmark = pytest.mark.gpu

# Edges: rows of less than a wave, of whole waves, of every tail length, of 16 waves, cut into
# segments (also short last ones), several teams in a workgroup; a last group of one to seven
# layers; channels in front that are a multiple of four, one more, one less, more than the 128
# whose weights fit the table at once; dilations up to the image, folds on both sides; two
# channels per layer; several images.
BLOCKS = [
    # (size, c_in, width, depth, batch, dilations)
    ((33, 64), 1, 1, 15, 1, None),
    ((10, 40), 4, 1, 9, 2, [1, 10, 3]),
    ((12, 129), 2, 1, 8, 1, [7, 1, 12, 2]),
    ((9, 131), 3, 1, 14, 2, [9, 3, 1]),
    ((7, 1021), 1, 1, 9, 1, [7, 1, 2]),
    ((11, 1024), 5, 1, 16, 1, [11, 10, 1, 5]),
    ((6, 1500), 1, 1, 8, 1, [6, 1, 3]),
    ((130, 1100), 2, 1, 3, 1, [128, 1, 100]),
    ((5, 2048), 2, 2, 6, 1, [5, 1, 2, 3]),
    ((13, 333), 2, 2, 8, 2, [1, 10, 4]),
    ((8, 70), 127, 1, 9, 1, [1, 2, 8]),
    ((8, 64), 140, 2, 4, 1, [1, 2]),
]


@pytest.mark.parametrize("case", BLOCKS, ids=lambda c: "x".join(map(str, c[0])) + "-c%d-w%d-d%d-B%d" % c[1:5])
def test_block_in_layer_groups(case):
    size, c_in, width, depth, batch, dilations = case
    dilations = [(dilations or range(1, 11))[i % len(dilations or range(1, 11))] for i in range(depth)]
    with tuning({"fwd.group": 1}):
        check_block(2, size, c_in, width, depth, batch, dilations=dilations, seed=41)


# The backward pass works in tiles of 32 voxels (the last one of a row moved left), blocks of 16
# channels and chunks of at most 112: rows of one tile, of one voxel more, of every remainder modulo
# four; channels below, at and past a block and a chunk; three groups and a rest; dilations up to
# the image (both mirrors at once); more tiles than waves.
BACKWARD = [
    ((33, 32), 1, 1, 15, 1, None),
    ((5, 33), 4, 1, 9, 2, [1, 5, 3]),
    ((12, 66), 9, 1, 8, 1, [7, 1, 12, 2]),
    ((9, 95), 3, 1, 24, 2, [9, 3, 1]),
    ((40, 132), 16, 1, 7, 1, [40, 33, 1, 16]),
    ((32, 35), 2, 1, 8, 1, [32, 31, 30]),
    ((7, 1021), 105, 1, 14, 1, [7, 1, 2]),
    ((6, 64), 226, 1, 8, 1, [6, 1, 3]),
    ((13, 333), 2, 2, 8, 2, [1, 10, 4]),
    ((5, 40), 122, 2, 4, 1, [1, 2]),
    ((300, 320), 1, 1, 9, 1, None),
]


@pytest.mark.parametrize("case", BACKWARD, ids=lambda c: "x".join(map(str, c[0])) + "-c%d-w%d-d%d-B%d" % c[1:5])
@pytest.mark.parametrize("input_grad", [True, False])
def test_block_backward_in_layer_groups(case, input_grad):
    size, c_in, width, depth, batch, dilations = case
    dilations = [(dilations or range(1, 11))[i % len(dilations or range(1, 11))] for i in range(depth)]
    with tuning({"bwd.group": 1}):
        check_block(2, size, c_in, width, depth, batch, dilations=dilations, seed=43, input_grad=input_grad)


# More channels than a chunk holds (128 of them for more than seven outputs, 64 for fewer): a rest
# of one channel and of several blocks, with and without gradients of the channels that the rest holds, several images, a volume.
@pytest.mark.parametrize("input_grad", [True, False])
@pytest.mark.parametrize("size, c_in, width, depth, batch", [
    ((512, 513), 122, 1, 8, 1), ((260, 512), 128, 1, 10, 2), ((515, 512), 140, 2, 7, 1), ((512, 520), 250, 1, 8, 1),
    ((512, 515), 70, 1, 6, 1), ((64, 66, 65), 130, 1, 4, 1), ((65, 64, 66), 64, 1, 2, 1)],
    ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else str(v))
def test_backward_groups_over_several_chunks(size, c_in, width, depth, batch, input_grad):
    check_block(len(size), size, c_in, width, depth, batch, dilations=[1 + 3 * i % 10 for i in range(depth)], seed=47,
                input_grad=input_grad)


# The same where the chunks have launches of their own: nine and ten blocks from 8192 segments of 32 voxels on, from 14000 with
# a rest of at most five blocks, from 65536 on with any; up to seven outputs (3D: two) over five blocks from 28000 on, else in
# one launch.  Just below and just above.
@pytest.mark.parametrize("size, c_in, depth, batch, launches", [
    ((510, 512), 136, 8, 1, 1), ((512, 512), 153, 8, 1, 2), ((600, 720), 154, 8, 1, 1), ((320, 701), 180, 8, 2, 2),
    ((640, 704), 201, 8, 1, 2), ((640, 704), 202, 8, 1, 1), ((32760, 33), 205, 8, 1, 1), ((32770, 33), 205, 8, 1, 2),
    ((900, 1000), 70, 2, 1, 2), ((870, 1000), 70, 2, 1, 1), ((900, 1000), 100, 2, 1, 1),
    ((63, 64, 65), 130, 4, 1, 1), ((65, 64, 65), 130, 4, 1, 2), ((76, 76, 77), 158, 4, 1, 1), ((77, 77, 77), 158, 4, 1, 2)],
    ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else str(v))
def test_backward_chunks_in_launches_of_their_own(size, c_in, depth, batch, launches):
    from msd_pytorch_amd.msd_block import msd_block
    dilations = [1 + 3 * i % 10 for i in range(depth)]
    x, dil, bias, ws, g = block_problem(len(size), size, c_in, 1, depth, batch, dilations, 47)
    leaves = [t.cuda().requires_grad_() for t in (bias, *ws)]
    xd, up = x.cuda().requires_grad_(), g.cuda()
    torch.cuda.synchronize()
    kernels = captured_kernels(lambda: torch.autograd.grad(msd_block(xd, dil, *leaves), leaves, up))
    assert sum("pull_rows" in name for name, _ in kernels) == launches
    assert sum("sum_group" in name for name, _ in kernels) == launches
    del leaves, xd, up
    check_block(len(size), size, c_in, 1, depth, batch, dilations=dilations, seed=47)


# Groups of eight to fourteen outputs: two slabs of 64 matrix rows, the upper outputs' share of the lower
# channels in one launch.  Blocks of 16 channels shared by four, two or one waves (1, 2 | 3, 4 | 5 to 8 blocks),
# two chunks; tiles of four segments that end inside an image, also between two images; halves of 7 + 7, 7 + 1,
# 6 + 8 and 6 + 2 outputs.
FOURTEEN = [
    ((5, 33), 1, 1, 8, 2, [1, 5, 3]),
    ((7, 95), 3, 1, 14, 2, [7, 2]),
    ((9, 66), 4, 1, 13, 1, None),
    ((6, 130), 19, 1, 14, 1, [6, 1, 4]),
    ((11, 64), 20, 1, 14, 3, [3, 11]),
    ((5, 127), 52, 1, 14, 1, [5, 1]),
    ((4, 97), 115, 1, 14, 1, [1, 4]),
    ((4, 40), 116, 1, 14, 2, [2, 3]),
    ((6, 70), 5, 2, 7, 1, [1, 6, 2]),
    ((13, 35), 3, 2, 4, 2, [13, 1]),
    ((40, 160), 2, 1, 28, 1, None),
]


@pytest.mark.parametrize("case", FOURTEEN, ids=lambda c: "x".join(map(str, c[0])) + "-c%d-w%d-d%d-B%d" % c[1:5])
def test_block_backward_in_groups_of_up_to_fourteen(case):
    size, c_in, width, depth, batch, dilations = case
    dilations = [min(size[0], (dilations or range(1, 11))[i % len(dilations or range(1, 11))]) for i in range(depth)]
    with tuning({"bwd.group": 1}):
        check_block(2, size, c_in, width, depth, batch, dilations=dilations, seed=59)


# Passes over one to four blocks of 16 channels, where a tile is gathered while the one before goes through the products: one, two or
# three tiles for a workgroup, not the same number for all of them, workers without a block, rows that end inside a
# tile; one slab of outputs and two.
@pytest.mark.parametrize("size, batch", [((7, 64), 1), ((90, 200), 1), ((64, 257), 2), ((9, 17, 35), 1), ((12, 40, 72), 2)], ids=str)
@pytest.mark.parametrize("c_in", [3, 20, 40, 60])
@pytest.mark.parametrize("slabs", [1, 2])
def test_backward_passes_over_few_blocks(size, batch, c_in, slabs):
    depth = (5 if slabs == 1 else 9) if len(size) == 2 else 2 * slabs
    with tuning({"bwd.group": 1}):
        check_block(len(size), size, c_in, 1, depth, batch, dilations=[1 + 2 * i % 5 for i in range(depth)], seed=107)


def exact_weight_gradients(x, g, dilations):
    """[output, channel, tap] in 64 bits: sum over v of x[c][reflected(v + dilation (tap - 1))] g[o][v]."""
    size = x.shape[2:]
    found = []
    for o, d in enumerate(dilations):
        source = []
        for n in size:
            at = torch.arange(n, device=x.device) + d * torch.arange(-1, 2, device=x.device)[:, None]
            at = torch.where(at < 0, -1 - at, at)
            source.append(torch.where(at >= n, 2 * n - 1 - at, at))
        taps = []
        for tap in range(3 ** len(size)):
            h = g[:, o].double()                   # what each voxel of x meets
            for axis in range(len(size)):
                k = tap // 3 ** (len(size) - 1 - axis) % 3
                h = torch.zeros_like(h).index_add_(axis + 1, source[axis][k], h)
            taps.append(torch.stack([(x[:, c].double() * h).sum() for c in range(x.shape[1])]))
        found.append(torch.stack(taps, 1))
    return torch.stack(found)


# Sums over millions of voxels: chains of 16 additions, of a sixteenth of the units of 32 voxels that a worker of one of 256 workgroups has
# (two workers share a block where there are one or two), and some 32 levels below and above them.  An addition of terms of mixed sign rounds to 0.6
# 2^-24 of its sum (the rms of half a unit in the last place), of which n in a chain come to sqrt(n / 2).  1.3: x is of one sign, so that
# some partial sums are larger.
@pytest.mark.parametrize("size, c_in, outputs, workers", [
    ((2048, 2048), 25, 14, 2), ((2048, 2048), 40, 14, 1), ((3000, 4096), 25, 7, 2), ((192, 192, 192), 30, 4, 2), ((192, 192, 192), 46, 4, 1)],
    ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else str(v))
def test_weight_gradients_over_many_voxels(size, c_in, outputs, workers):
    from msd_pytorch_amd import msd_custom_convolutions as cc
    gen = torch.Generator(device="cuda").manual_seed(83)
    stack = torch.rand(1, c_in + outputs, *size, device="cuda", generator=gen)
    stack[:, c_in:] = 1                            # every ReLU open
    gradient = torch.randn(1, c_in + outputs, *size, device="cuda", generator=gen)
    dilations = [1 + i % 10 for i in range(outputs)]
    weights = [torch.randn(1, c_in + i, *[3] * len(size), device="cuda", generator=gen) * 0.1 for i in range(outputs)]
    for w in weights:
        w[:, c_in:] = 0                            # (the outputs' gradients are what they are given as)
    want = exact_weight_gradients(stack[:, :c_in], gradient[:, c_in:], dilations)
    gk, gb = [torch.zeros_like(w) for w in weights], torch.zeros(outputs, device="cuda")
    with tuning({"bwd.group": 1}):
        cc.block_backward(stack, gradient, c_in, dilations, weights, gk, gb, True)
    got = torch.stack([k[0, :c_in].reshape(c_in, -1) for k in gk])
    units = torch.Size(size).numel() / 32 / 256 / workers
    bound = 1.3 * 0.6 * 2.0 ** -24 * (16 / 2 + units / 16 / 2 + 32 / 2) ** 0.5
    assert float((got - want).norm() / want.norm()) <= bound


# One slab of outputs over three and four blocks: images from 20000 segments of 32 voxels on for each 256 workgroups of a chunk, volumes from 30 x 2^20 values of
# the channels and the outputs on, take the eight waves that gather and multiply in turn.  Just below and just above, rows that end inside a segment, rows with gaps, two images, a block without its
# last channels and a chunk of two blocks beside one of three; against the layers on their own.
@pytest.mark.parametrize("size, batch, c_in, gap, wide", [
    ((799, 800), 1, 40, 0, False), ((801, 799), 1, 40, 0, True), ((400, 830), 2, 62, 3, True), ((801, 800), 1, 75, 0, True),
    ((595, 640), 1, 75, 0, False), ((605, 640), 1, 75, 0, True), ((400, 520), 1, 130, 0, True),
    ((70, 76, 80), 1, 70, 0, False), ((72, 76, 80), 1, 70, 0, True), ((80, 100, 60), 1, 65, 1, True),
    ((801, 798), 1, 31, 0, False), ((63, 100, 99), 1, 47, 0, False), ((64, 100, 99), 1, 47, 0, True), ((70, 125, 99), 1, 33, 1, False), ((100, 125, 99), 1, 33, 1, True),
    ((35, 124, 100), 2, 33, 1, False), ((36, 124, 100), 2, 33, 1, True)], ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else str(v))
def test_one_slab_over_three_and_four_blocks(size, batch, c_in, gap, wide):
    from msd_pytorch_amd import msd_custom_convolutions as cc
    gen = torch.Generator(device="cuda").manual_seed(89)
    both = torch.randn(2, batch, c_in + 2, *size[:-1], size[-1] + gap, device="cuda", generator=gen)
    stack, gradient = both[0][..., :size[-1]], both[1][..., :size[-1]]
    weights = [torch.randn(1, c_in + i, *[3] * len(size), device="cuda", generator=gen) * 0.1 for i in range(2)]

    def run(setting):
        g = torch.empty_strided(gradient.shape, gradient.stride(), device="cuda").copy_(gradient)
        gk, gb = [torch.zeros_like(w) for w in weights], torch.zeros(2, device="cuda")
        with tuning({"bwd.group": setting}):
            cc.block_backward(stack, g, c_in, [3, 7], weights, gk, gb, True)
        return g[:, :c_in], gb, *gk

    torch.cuda.synchronize()
    passes = [name for name, _ in captured_kernels(lambda: run(1)) if "pull_rows" in name]
    assert len(passes) == 1 and ("pull_rows_wide" in passes[0]) == wide
    found = [run(setting) for setting in (0, 1)]
    for a, b in zip(*found):
        assert rel_err(b, a) <= 1e-5


# The same of a layer of its own, whose gradients are written: by the values in images too.
@pytest.mark.parametrize("size, batch, c_in, outputs, wide", [
    ((660, 801), 1, 56, 3, False), ((672, 801), 1, 56, 3, True), ((300, 396), 4, 63, 3, False), ((300, 398), 4, 63, 3, True),
    ((77, 100, 99), 1, 40, 1, False), ((78, 100, 99), 1, 40, 1, True), ((58, 101, 80), 1, 64, 2, False), ((61, 101, 80), 1, 64, 2, True), ((25, 99, 181), 2, 33, 2, False),
    ((25, 99, 182), 2, 33, 2, True)],
    ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else str(v))
def test_a_layer_over_three_and_four_blocks(size, batch, c_in, outputs, wide):
    from msd_pytorch_amd import conv2d, conv3d
    gen = torch.Generator(device="cuda").manual_seed(101)
    fn = conv2d.conv2d_relu if len(size) == 2 else conv3d.conv3d_relu
    x = torch.randn(batch, c_in, *size, device="cuda", generator=gen).requires_grad_()
    w = (torch.randn(outputs, c_in, *[3] * len(size), device="cuda", generator=gen) * 0.1).requires_grad_()
    b = torch.zeros(outputs, device="cuda").requires_grad_()
    g = torch.randn(batch, outputs, *size, device="cuda", generator=gen)

    def run(x, w, b, *leaves):
        y = fn(x, w, b, torch.empty(batch, outputs, *size, device="cuda"), 1, 3)
        return torch.autograd.grad(y, leaves, g)

    found = run(x, w, b, x, w, b)
    torch.cuda.synchronize()
    passes = [name for name, _ in captured_kernels(lambda: run(x, w, b, x, w, b)) if "pull_rows" in name]
    assert len(passes) == 1 and ("pull_rows_wide" in passes[0]) == wide
    for a, b in zip(run(x, w.detach(), b.detach(), x) + run(x.detach(), w, b, w, b), found):       # (one gradient at a time: the operators of their own)
        assert rel_err(b, a) <= 1e-5


# Volumes: groups of up to four outputs, the same tiles over the rows of all slices.  Slices and rows
# whose outer taps lie outside on both sides, dilations up to the volume, tiles that end inside a volume and between
# two, every remainder modulo four, groups of 2, 3 and 4 outputs and a layer left over, two channels per layer, blocks
# shared by four, two and one waves, two chunks.
VOLUMES = [
    ((5, 6, 33), 1, 1, 5, 2, [1, 5, 3]),
    ((9, 5, 32), 2, 1, 4, 1, [5, 2, 1]),
    ((3, 11, 67), 9, 1, 7, 2, [3, 1, 2]),
    ((12, 13, 38), 14, 1, 6, 1, [1, 12, 7]),
    ((4, 4, 101), 30, 1, 4, 3, [4, 1]),
    ((6, 3, 64), 52, 1, 9, 1, [3, 2, 1]),
    ((2, 5, 45), 100, 1, 4, 1, [2, 1]),
    ((3, 2, 35), 125, 1, 3, 2, [1, 2]),
    ((24, 30, 75), 1, 1, 9, 1, None),
    ((5, 7, 33), 1, 2, 2, 2, [5, 1]),
    ((4, 6, 130), 15, 2, 5, 1, [3, 1, 4]),
    ((25, 23, 65), 2, 2, 4, 1, [10, 9, 1]),
    ((4, 3, 5), 2, 1, 4, 2, [3, 1]),
    ((2, 4, 4), 17, 1, 3, 1, [2, 1]),
    ((19, 9, 7), 3, 2, 3, 3, [7, 2]),
]


@pytest.mark.parametrize("case", VOLUMES, ids=lambda c: "x".join(map(str, c[0])) + "-c%d-w%d-d%d-B%d" % c[1:5])
@pytest.mark.parametrize("input_grad", [True, False])
def test_block_backward_of_volumes_in_groups(case, input_grad):
    size, c_in, width, depth, batch, dilations = case
    dilations = [(dilations or range(1, 11))[i % len(dilations or range(1, 11))] for i in range(depth)]
    with tuning({"bwd.group": 1}):
        check_block(3, size, c_in, width, depth, batch, dilations=dilations, seed=67, input_grad=input_grad)


# Layers of one and two channels in one group: seven outputs above a layer of one, one output above a layer of two (3D: in a
# volume with and without gaps), against the layers on their own.
@pytest.mark.parametrize("size,widths,gap", [((9, 37), [1, 1, 2, 2, 2, 2, 2, 2], 0), ((4, 5, 37), [2, 1], 0), ((4, 5, 37), [2, 1], 3),
                                             ((5, 4, 33), [1, 2, 1], 0)], ids=str)
def test_backward_groups_of_mixed_widths(size, widths, gap):
    from msd_pytorch_amd import msd_custom_convolutions as cc
    gen = torch.Generator().manual_seed(73)
    c_in, channels = 3, 3 + sum(widths)
    big = torch.randn(2, 2, channels, *size[:-1], size[-1] + gap, generator=gen).cuda()
    stack, gradient = big[0][..., :size[-1]], big[1][..., :size[-1]]
    reads = [c_in + sum(widths[:i]) for i in range(len(widths))]
    weights = [torch.randn(w, c, *([3] * len(size)), generator=gen).cuda() * 0.1 for w, c in zip(widths, reads)]
    found = []
    for setting in (0, 1):
        g = torch.empty_strided(gradient.shape, gradient.stride(), device="cuda").copy_(gradient)
        gk, gb = [torch.zeros_like(w) for w in weights], torch.zeros(channels - c_in).cuda()
        with tuning({"bwd.group": setting}):
            cc.block_backward(stack, g, c_in, [1 + i % 4 for i in range(len(widths))], weights, gk, gb, True)
        found.append((g[:, :c_in], gb, *gk))
    for a, b in zip(*found):
        assert rel_err(b, a) <= 1e-5


# A volume without gaps is taken as one row, any other by its rows (of 32 voxels at least): the same gradients from
# rows with gaps, from slices with gaps and from slices and rows in the other order.
@pytest.mark.parametrize("layout", ["rows", "slices", "transposed"])
@pytest.mark.parametrize("c_in,width,depth", [(3, 1, 4), (33, 1, 3), (66, 1, 4), (5, 1, 2), (40, 1, 2), (2, 2, 2), (1, 2, 5), (3, 1, 5)])
def test_volumes_in_other_layouts(c_in, width, depth, layout):
    from msd_pytorch_amd import msd_custom_convolutions as cc
    gen = torch.Generator().manual_seed(71)
    size, channels = (4, 5, 45), c_in + depth * width
    stack, gradient = (torch.randn(2, channels, *size, generator=gen).cuda() for _ in range(2))
    weights = [torch.randn(width, c_in + i * width, 3, 3, 3, generator=gen).cuda() * 0.1 for i in range(depth)]

    def view(t):
        d, h, w = size
        big = {"rows": (d, h, w + 3), "slices": (d, h + 2, w), "transposed": (h, d, w)}[layout]
        big = torch.full((2, channels, *big), float("nan"), device="cuda")
        big = big.transpose(2, 3) if layout == "transposed" else big[..., :h, :w]
        return big.copy_(t)

    found = []
    for s, g in ((stack, gradient.clone()), (view(stack), view(gradient))):
        gk, gb = [torch.zeros_like(w) for w in weights], torch.zeros(depth * width).cuda()
        cc.block_backward(s, g, c_in, [1 + i % 4 for i in range(depth)], weights, gk, gb, True)
        found.append((g[:, :c_in], gb, *gk))
    for a, b in zip(*found):
        assert rel_err(b, a) <= 1e-5


# What is no sum of three bf16 values takes the fp32 instruction: the same infinities and NaNs as from the
# layers' own kernels, and the largest finite values (which round to an infinity in bf16) stay finite.
@pytest.mark.parametrize("where", ["stack", "gradient", "weight"])
@pytest.mark.parametrize("value", [float("inf"), float("-inf"), float("nan"), 3.4e38, -3.4028234e38])
@pytest.mark.parametrize("depth", [6, 14])
def test_values_without_bf16_parts(where, value, depth):
    from msd_pytorch_amd import msd_custom_convolutions as cc
    gen = torch.Generator().manual_seed(29)
    c_in, size = 4, (9, 71)
    stack = torch.rand(1, c_in + depth, *size, generator=gen).cuda() + 0.1     # every ReLU open
    gradient = torch.rand(1, c_in + depth, *size, generator=gen).cuda() * 1e-3
    weights = [(torch.rand(1, c_in + i, 3, 3, generator=gen) * 1e-3 + 1e-4).cuda() for i in range(depth)]
    if where == "stack":
        stack[0, 2, 4, 65] = value
    elif where == "gradient":
        gradient[0, c_in + 1, 4, 66] = value
    else:
        weights[depth - 2][0, 1, 1, 2] = value
    found = []
    for setting in (0, 1):
        gk, gb, grads = [torch.zeros_like(w) for w in weights], torch.zeros(depth).cuda(), gradient.clone()
        with tuning({"bwd.group": setting}):
            cc.block_backward(stack, grads, c_in, [1 + i % 4 for i in range(depth)], weights, gk, gb, True)
        found.append(torch.cat([grads[:, :c_in].flatten(), gb, *(k.flatten() for k in gk)]))
    assert same_specials(found[1], found[0])
    finite = torch.isfinite(found[0])
    assert bool(finite.any())
    # (sums of up to 639 terms of one sign in another order, relative to the largest)
    a, b = found[0][finite].double(), found[1][finite].double()
    assert float(((a - b).abs() / a.abs().clamp_min(1e-30)).max()) <= 1e-4


# The same where a workgroup walks several tiles and only one or two of them, not the first (in either buffer) holds such a value, so that some of its units are
# left to the second run and some are not: passes over one to four blocks of channels of two slabs and of one, over five and six (all waves alike), one slab in a
# large image, volumes with and without gaps.  The rest of all gradients is compared as well: grad_input is added to in place, by one run or the other.
@pytest.mark.parametrize("where", ["stack", "gradient", "weight"])
@pytest.mark.parametrize("value", [float("inf"), float("nan"), 3.4e38])
@pytest.mark.parametrize("size, gap, c_in, depth, at", [
    ((160, 320), 0, 4, 14, 0.4), ((160, 321), 0, 20, 14, 0.9), ((160, 320), 0, 40, 14, 0.7), ((320, 330), 3, 60, 14, 0.35), ((400, 320), 0, 80, 14, 0.3),
    ((400, 320), 0, 90, 9, 0.9), ((320, 320), 0, 10, 6, 0.4), ((320, 320), 0, 30, 6, 0.7), ((320, 333), 0, 50, 6, 0.6), ((650, 1000), 0, 40, 2, 0.5),
    ((16, 40, 65), 0, 10, 4, 0.4), ((16, 40, 65), 0, 30, 4, 0.7), ((16, 40, 65), 0, 50, 4, 0.8), ((16, 50, 65), 3, 50, 4, 0.4), ((32, 60, 65), 0, 70, 4, 0.6),
    ((32, 60, 65), 2, 70, 3, 0.3), ((20, 60, 65), 0, 20, 2, 0.6), ((30, 60, 65), 1, 40, 2, 0.5),
    ((30, 60, 65), 1, 20, 2, 0.7)],
    ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else str(v))
def test_values_without_bf16_parts_in_some_tiles(size, gap, c_in, depth, at, value, where):
    from msd_pytorch_amd import msd_custom_convolutions as cc
    gen = torch.Generator(device="cuda").manual_seed(31)
    taps = [3] * len(size)

    def some(scale, least):
        big = torch.rand(1, c_in + depth, *size[:-1], size[-1] + gap, device="cuda", generator=gen)
        return (big * scale + least)[..., :size[-1]]

    stack, gradient = some(1, 0.1), some(1e-3, 0)              # every ReLU open
    weights = [torch.rand(1, c_in + i, *taps, device="cuda", generator=gen) * 1e-3 + 1e-4 for i in range(depth)]
    voxel = [int(at * n) for n in size[:-1]] + [size[-1] // 2]
    if where == "stack":
        stack[(0, c_in // 2, *voxel)] = value
    elif where == "gradient":
        gradient[(0, c_in, *voxel)] = value          # (the lowest layer: it stays where it is)
    else:
        weights[depth - 1][(0, c_in - 1, *[1] * len(size))] = value
    found = []
    for setting in (0, 1):
        grads = torch.empty_strided(gradient.shape, gradient.stride(), device="cuda").copy_(gradient)
        gk, gb = [torch.zeros_like(w) for w in weights], torch.zeros(depth, device="cuda")
        with tuning({"bwd.group": setting}):
            cc.block_backward(stack, grads, c_in, [1 + i % 4 for i in range(depth)], weights, gk, gb, True)
        found.append(torch.cat([grads[:, :c_in].flatten(), gb, *(k.flatten() for k in gk)]))
    assert same_specials(found[1], found[0])
    finite = torch.isfinite(found[0])
    assert bool(finite.any())
    # (sums of terms of one sign: chains of at most some thousand additions, relative to the largest)
    a, b = found[0][finite].double(), found[1][finite].double()
    assert float(((a - b).abs() / a.abs().clamp_min(1e-30)).max()) <= 1e-4


def test_an_infinity_meets_its_own_voxels_only():
    """The last tile of a row repeats voxels of the one before (here 8 to 31): what they hold counts once."""
    from msd_pytorch_amd import msd_custom_convolutions as cc
    gen = torch.Generator().manual_seed(3)
    c_in, depth, size = 4, 8, (6, 40)
    stack = torch.rand(1, c_in + depth, *size, generator=gen).cuda() + 0.1     # every ReLU open
    stack[0, 1, 3, 20] = float("inf")
    gradient = torch.randn(1, c_in + depth, *size, generator=gen).cuda()
    weights = [torch.randn(1, c_in + i, 3, 3, generator=gen).cuda() for i in range(depth)]
    found = []
    for setting in (0, 1):
        gk, gb = [torch.zeros_like(w) for w in weights], torch.zeros(depth).cuda()
        with tuning({"bwd.group": setting}):
            cc.block_backward(stack, gradient.clone(), c_in, [1, 2, 3, 1, 2, 3, 1, 2], weights, gk, gb, True)
        found.append(torch.cat([k.flatten() for k in gk]))
    assert torch.isinf(found[0]).any()
    assert same_specials(found[1], found[0])


@pytest.mark.parametrize("c_in", [4, 5, 6, 7, 129])
def test_an_infinity_in_front_of_a_forward_group_stays_one(c_in):
    """A step of the pass takes four channels; the last one's repetitions must not meet it."""
    from msd_pytorch_amd import msd_custom_convolutions as cc
    gen = torch.Generator().manual_seed(5)
    depth, size = 9, (6, 40)
    image = torch.rand(1, c_in, *size, generator=gen).cuda()
    image[0, c_in - 1, 2, 17] = float("inf")
    weights = [(torch.rand(1, c_in + i, 3, 3, generator=gen) * 0.1 + 0.01).cuda() for i in range(depth)]
    found = []
    for setting in (0, 1):
        stack = torch.empty(1, c_in + depth, *size, device="cuda")
        stack[:, :c_in] = image
        with tuning({"fwd.group": setting}):
            cc.block_forward(stack, c_in, [1, 2, 3, 1, 2, 3, 1, 2, 3], torch.zeros(depth, device="cuda"), weights)
        found.append(stack)
    assert torch.isinf(found[0][:, c_in:]).any() and not torch.isnan(found[0]).any()
    finite = torch.isfinite(found[0])
    assert same_specials(found[1], found[0])
    assert rel_err(found[1][finite], found[0][finite]) <= 1e-5


# Forward groups of eight to fourteen outputs (forced; dilations up to 16): one segment of 64 voxels, several, a last
# one of a single voxel or of less than a halo, of odd lengths; rows in parts; one step of 32 channels, whole
# steps, one channel more, more than the table of weights holds at once; two channels per layer; dilations
# above 16, which go in sevens; rows that the finishing launches take one voxel at a time.
FORWARD_FOURTEEN = [
    ((40, 64), 2, 1, 14, 1, [1, 16, 5]),
    ((33, 65), 3, 1, 9, 2, [16, 3]),
    ((20, 520), 32, 1, 14, 1, None),
    ((17, 111), 33, 1, 14, 3, [12, 7, 1]),
    ((9, 1021), 12, 1, 16, 1, [9, 2]),
    ((1100, 35), 130, 1, 14, 1, [1, 2, 4, 8]),
    ((12, 1024), 7, 2, 7, 1, None),
    ((27, 499), 6, 2, 7, 1, [3, 12]),
    ((30, 32), 65, 1, 14, 1, [16, 15]),
    ((20, 96), 5, 1, 15, 1, [17, 1]),
    ((5, 2048), 30, 2, 5, 1, [5, 1]),
]


@pytest.mark.parametrize("case", FORWARD_FOURTEEN, ids=lambda c: "x".join(map(str, c[0])) + "-c%d-w%d-d%d-B%d" % c[1:5])
def test_block_in_forward_groups_of_up_to_fourteen(case):
    size, c_in, width, depth, batch, dilations = case
    dilations = [(dilations or range(1, 11))[i % len(dilations or range(1, 11))] for i in range(depth)]
    with tuning({"fwd.group": 1024}):
        check_block(2, size, c_in, width, depth, batch, dilations=dilations, seed=61)


# As many channels as the table of weights holds at once, one step more and three parts of it; fewer rows than the workgroups of one XCD have
# waves, one row, more rows than there are waves; rows in parts, of several segments, a last one of less than four voxels.
@pytest.mark.parametrize("case", [
    ((16, 70), 255, 1, 9, 1, [3, 16]),
    ((17, 131), 257, 1, 14, 1, [1, 16, 7]),
    ((1, 33), 300, 1, 10, 1, [1, 1]),
    ((9, 1022), 520, 1, 8, 1, [9, 4]),
    ((1030, 34), 260, 2, 5, 1, [2, 11]),
    ((66, 67), 12, 2, 7, 2, [5, 16, 1]),
], ids=lambda c: "x".join(map(str, c[0])) + "-c%d-w%d-d%d-B%d" % c[1:5])
def test_forward_groups_of_fourteen_over_many_channels(case):
    size, c_in, width, depth, batch, dilations = case
    dilations = [dilations[i % len(dilations)] for i in range(depth)]
    with tuning({"fwd.group": 1024}):
        check_block(2, size, c_in, width, depth, batch, dilations=dilations, seed=67)


# Where the weights of a pass are loaded in parts, the order of the additions changes from segment to segment of a row, but the same rows
# give the same bits at every place of a batch: more rows than there are waves, of an odd and an even number of segments.
@pytest.mark.parametrize("width", [100, 150])
@pytest.mark.parametrize("c_in", [200, 260])
def test_the_place_in_a_batch_does_not_change_a_forward_group(c_in, width):
    from msd_pytorch_amd import msd_custom_convolutions as cc
    gen = torch.Generator().manual_seed(97)
    depth = 9
    stack = torch.empty(5, c_in + depth, 300, width, device="cuda")
    stack[:, :c_in] = torch.randn(c_in, 300, width, generator=gen).cuda()
    weights = [(torch.randn(1, c_in + i, 3, 3, generator=gen) * 0.05).cuda() for i in range(depth)]
    with tuning({"fwd.group": 1024}):
        cc.block_forward(stack, c_in, [1 + i % 4 for i in range(depth)], torch.zeros(depth, device="cuda"), weights)
    assert all(torch.equal(image, stack[0]) for image in stack[1:])


@pytest.mark.parametrize("where", ["input", "weight"])
@pytest.mark.parametrize("value", [float("inf"), float("nan"), 3.4e38])
def test_values_without_bf16_parts_in_front_of_a_forward_group(where, value):
    from msd_pytorch_amd import msd_custom_convolutions as cc
    gen = torch.Generator().manual_seed(37)
    c_in, depth, size = 45, 9, (22, 513)
    image = torch.rand(1, c_in, *size, generator=gen).cuda()
    # (small weights of one sign: what a layer makes of the largest finite value is finite)
    weights = [(torch.rand(1, c_in + i, 3, 3, generator=gen) * 1e-3 + 1e-4).cuda() for i in range(depth)]
    if where == "input":
        image[0, c_in - 1, 17, 511] = value
    else:
        weights[2][0, 40, 1, 2] = value
        image[0, 40] = image[0, 40] * 1e-3 + 1e-4
    found = []
    for setting in (0, 1024):
        stack = torch.empty(1, c_in + depth, *size, device="cuda")
        stack[:, :c_in] = image
        with tuning({"fwd.group": setting}):
            cc.block_forward(stack, c_in, [1, 12, 3, 1, 2, 3, 1, 2, 3], torch.zeros(depth, device="cuda"), weights)
        found.append(stack[:, c_in:])
    assert same_specials(found[1], found[0])
    finite = torch.isfinite(found[0])
    assert bool(finite.any()) and rel_err(found[1][finite], found[0][finite]) <= 1e-5


# Rows that the finishing launch does not take (more than 1024 voxels that are not whole groups of
# four, more than 2048): fwd_lattice adds the planes, with no channel of the group's own and with some.
@pytest.mark.parametrize("case", [
    ((7, 1030), 12, 1, 9, 2, [7, 1, 2]),
    ((6, 2046), 12, 1, 8, 1, [1, 6, 3]),
    ((5, 2052), 13, 1, 9, 1, [5, 1, 2]),
    ((5, 1026), 6, 2, 4, 1, [1, 2, 5]),
    ((4, 4096), 8, 2, 5, 1, [1, 2, 4]),
], ids=lambda c: "x".join(map(str, c[0])) + "-c%d-w%d-d%d-B%d" % c[1:5])
def test_forward_groups_of_long_rows(case):
    size, c_in, width, depth, batch, dilations = case
    dilations = [dilations[i % len(dilations)] for i in range(depth)]
    check_block(2, size, c_in, width, depth, batch, dilations=dilations, seed=47)


@pytest.mark.parametrize("size", [(256, 256), (9, 20, 64)], ids=str)
def test_blocks_with_less_workspace_than_the_groups_ask_for(size):
    """Callers of the C interface choose the workspace: down to what the layers ask for one by one."""
    import ctypes
    import oracle
    from msd_pytorch_amd import _native, msd_custom_convolutions as cc
    from parity import block_problem
    lib = _native.load()
    ndim, c_in, depth = len(size), 17, 15
    x, dil, bias, ws, g = block_problem(ndim, size, c_in, 1, depth, 1, seed=3)
    want = oracle.block_forward(x.double(), dil, bias.double(), [w.double() for w in ws])
    weights, bias_d = [w.cuda() for w in ws], bias.cuda()
    stack = torch.empty(1, c_in + depth, *size, device="cuda")
    stack[:, :c_in] = x.cuda()
    head = cc._block_head(stack, c_in, dil, weights)
    query = (head[0], head[1], head[2], c_in, depth, head[5], head[6])
    pointers, stream = cc._ptr_array(weights), cc._stream(stack)

    def scratch(need):
        # what lies behind the workspace has to stay as it is
        buffer = torch.full((need + 1024,), 0x5a, dtype=torch.uint8, device="cuda")
        return buffer, ctypes.c_void_p(buffer.data_ptr())

    need = lib.msd_block_forward_workspace_bytes(*query)
    assert need == (3 * 7 * size[0] * size[1] * 4 if ndim == 2 else 0)
    if need:
        need -= 4                                  # (the second group, of the last layer alone, is none)
        buffer, at = scratch(need)
        assert lib.msd_block_forward_ws(*head, *cc._view(stack), pointers, ctypes.c_void_p(bias_d.data_ptr()), at, need,
                                        stream) == 0, _native.last_error()
        assert rel_err(stack, want) <= 1e-5
        assert bool((buffer[need:] == 0x5a).all())
    else:
        stack.copy_(want)

    layers = [lib.msd_workspace_bytes(head[0], ndim, 1, c_in + i, 1, head[6]) for i in range(depth)]
    pairs = [lib.msd_workspace_bytes(head[0], ndim, 1, c_in + i, 2, head[6]) for i in range(depth - 1)]
    need = max(layers)
    # (a 2D group over 17 to 32 channels asks for 4.2 MB here)
    assert need < max(pairs) and (ndim == 3 or need < 4_200_000) and need < lib.msd_block_workspace_bytes(*query)
    buffer, at = scratch(need)
    grads = g.cuda()
    gk, gb = [torch.zeros_like(w) for w in weights], torch.zeros_like(bias_d)
    assert lib.msd_block_backward(*head, *cc._view(stack), *cc._view(grads), pointers, cc._ptr_array(gk),
                                  ctypes.c_void_p(gb.data_ptr()), 1, at, need, stream) == 0, _native.last_error()
    want_gx, want_gb, want_gw = oracle.block_backward(stack.double().cpu(), g.double(), dil, bias.double(),
                                                      [w.double() for w in ws])
    assert rel_err(grads[:, :c_in], want_gx) <= 1e-4 and rel_err(gb, want_gb) <= 1e-4
    for a, c in zip(gk, want_gw):
        assert rel_err(a, c) <= 1e-4
    assert bool((buffer[need:] == 0x5a).all())


# Layers of one and of two channels in one block: groups of five to seven outputs whose layers start
# at odd outputs, with an odd number of channels in front and above.
@pytest.mark.parametrize("widths", [
    [1, 2, 1, 2, 1, 2, 2, 1, 2, 1],
    [2, 2, 2, 1, 2, 2, 2, 1],
    [2, 1, 2, 2, 2, 2, 1, 1, 2],
    [2, 2, 1, 1, 1, 2, 1, 1, 1, 1, 2],
], ids=lambda w: "".join(map(str, w)))
@pytest.mark.parametrize("size,c_in", [((18, 64), 4), ((9, 77), 13)])
def test_groups_of_layers_of_one_and_two_channels(widths, size, c_in):
    import oracle
    from msd_pytorch_amd.msd_block import msd_block
    gen = torch.Generator().manual_seed(19)
    weights, channels = [], c_in
    for w in widths:
        weights.append(torch.randn(w, channels, 3, 3, generator=gen) * (2.0 / (9 * channels)) ** 0.5)
        channels += w
    dilations = [1 + i % 4 for i in range(len(widths))]
    x, bias = torch.rand(2, c_in, *size, generator=gen), torch.randn(channels - c_in, generator=gen) * 0.05
    g = torch.randn(2, channels, *size, generator=gen)
    leaves = [t.cuda().requires_grad_() for t in (x, bias, *weights)]
    with tuning({"fwd.group": 1, "bwd.group": 1}):
        got = msd_block(leaves[0], dilations, leaves[1], *leaves[2:])
        grads = torch.autograd.grad(got, leaves, g.cuda())
    w64 = [w.double() for w in weights]
    assert rel_err(got, oracle.block_forward(x.double(), dilations, bias.double(), w64)) <= 1e-5
    want_gx, want_gb, want_gw = oracle.block_backward(got.detach().double().cpu(), g.double(), dilations, bias.double(), w64)
    for a, b in zip(grads, (want_gx, want_gb, *want_gw)):
        assert rel_err(a, b) <= 1e-4


# What passes of two layers run where the groups do not apply, at sizes that a block takes in groups by default.
@pytest.mark.parametrize("case", [
    ((40, 67), 20, 1, 6, 1, None),                 # odd rows, 17 to 32 channels
    ((64, 128), 50, 1, 4, 1, None),                # whole rows, 33 to 64
], ids=lambda c: "x".join(map(str, c[0])) + "-c%d-w%d-d%d-B%d" % c[1:5])
def test_pairs_of_layers_where_groups_would_run(case):
    size, c_in, width, depth, batch, dilations = case
    with tuning({"block.pair": 1, "block.triple": 0}):
        check_block(2, size, c_in, width, depth, batch, dilations=dilations, seed=53)


@pytest.mark.parametrize("pitch,gap,offset", [(80, 0, 0), (83, 5, 3), (96, 64, 1)])
def test_groups_on_views_with_gaps(pitch, gap, offset):
    """Rows and planes apart, and not on 16 bytes: a view of a larger buffer, what lies between is left alone."""
    import oracle
    from msd_pytorch_amd import msd_custom_convolutions as cc
    from parity import block_problem
    size, c_in, depth, batch = (11, 77), 13, 9, 2
    x, dil, bias, ws, g = block_problem(2, size, c_in, 1, depth, batch, seed=23)
    channels, plane = c_in + depth, size[0] * pitch + gap

    def view():
        buffer = torch.full((offset + batch * channels * plane,), 7.0, device="cuda")
        strides = (channels * plane, plane, pitch, 1)
        return buffer, buffer.as_strided((batch, channels, *size), strides, offset)

    (sbuf, stack), (gbuf, grads) = view(), view()
    stack[:, :c_in] = x.cuda()
    grads.copy_(g)
    weights, gk, gb = [w.cuda() for w in ws], [torch.zeros_like(w).cuda() for w in ws], torch.zeros(depth).cuda()
    with tuning({"fwd.group": 1, "bwd.group": 1}):
        cc.block_forward(stack, c_in, dil, bias.cuda(), weights)
        cc.block_backward(stack, grads, c_in, dil, weights, gk, gb, True)
    w64 = [w.double() for w in ws]
    assert rel_err(stack, oracle.block_forward(x.double(), dil, bias.double(), w64)) <= 1e-5
    want_gx, want_gb, want_gw = oracle.block_backward(stack.double().cpu().contiguous(), g.double(), dil, bias.double(), w64)
    assert rel_err(grads[:, :c_in], want_gx) <= 1e-4 and rel_err(gb, want_gb) <= 1e-4
    for a, b in zip(gk, want_gw):
        assert rel_err(a, b) <= 1e-4
    for buffer, inner in ((sbuf, stack), (gbuf, grads)):
        inner.fill_(7.0)
        assert bool((buffer == 7.0).all())
