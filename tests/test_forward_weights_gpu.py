"""What the forward kernel is launched with.  How it takes its weights: from vector registers, where it forms all rows of a tile, also those past the
image edge, or from scalar registers, where it skips such rows.  And in how many groups it takes the channels."""
import re

import pytest
import torch

from cases import make_problem, problem_on
from parity import captured_kernels, check_operator_problem
from test_knobs_gpu import tuning

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def cc():
    from msd_pytorch_amd import msd_custom_convolutions
    return msd_custom_convolutions


def forward_instances(cc, shape):
    """Each launch of fwd_lattice that a layer's forward pass makes: its template arguments as numbers and the lanes of a workgroup."""
    p = problem_on(make_problem(shape, torch.float32), "cuda")
    kernels = captured_kernels(lambda: cc.conv_relu_forward(p["x"], p["k"], p["bias"], p["y"], p["d"]))
    found = [(re.search(r"fwd_latticeI((?:L[ib]\d+E)+)E", name), lanes) for name, lanes in kernels]
    return [([int(v) for v in re.findall(r"L[ib](\d+)E", m.group(1))], lanes) for m, lanes in found if m]


# (settings, (B, C_in, C_out, spatial, dilation), copies): volumes and images with fewer slices or rows per residue class than a tile of
# the instance has, and with exactly as many, for each tile and number of outputs; one channel group and several.
THIN = [({}, s, c) for s, c in (
    ((1, 5, 1, (2, 23, 70), 2), 0), ((1, 14, 1, (3, 20, 64), 2), 1), ((2, 9, 1, (23, 3, 40), 3), 0), ((1, 4, 1, (23, 6, 40), 2), 0),
    ((1, 4, 1, (23, 7, 40), 2), 1), ((1, 30, 1, (8, 9, 130), 8), 0), ((1, 5, 2, (4, 33, 66), 4), 0), ((1, 5, 2, (5, 25, 66), 4), 1))]
THIN += [({"fwd.lattice3d": m}, s, c) for m, s, c in (
    (24, (1, 7, 1, (9, 3, 40), 3), 0), (33, (1, 7, 1, (6, 9, 40), 3), 0), (33, (1, 7, 1, (7, 9, 40), 3), 1), (44, (1, 7, 1, (6, 16, 40), 2), 0),
    (44, (1, 20, 1, (16, 3, 65), 2), 0), (44, (1, 7, 1, (7, 16, 40), 2), 1))]
THIN += [({"fwd.split": 1, "fwd.lattice3d": 0}, s, c) for s, c in (
    ((1, 7, 1, (1, 12, 40), 1), 0), ((1, 7, 1, (27, 6, 40), 3), 0), ((1, 7, 1, (27, 7, 40), 3), 1))]
THIN += [({"fwd.rows2d": r, "fwd.vec2d": v}, (2, 6, 1, (3 * r - 3, 256 if v == 4 else 128 if v == 2 else 70), 3), 0)
         for r in (2, 3, 4, 5, 6) for v in (1, 2, 4)]
THIN += [({"fwd.vec2d": v}, (1, 6, 2, (4, 256 if v == 4 else 128 if v == 2 else 71), 2), 0) for v in (1, 2, 4)]


def _id(case):
    settings, s, _ = case
    return ",".join("%s=%d" % kv for kv in settings.items()) + "-B%d-C%d-w%d-%s-d%d" % (*s[:3], "x".join(map(str, s[3])), s[4])


@pytest.mark.parametrize("case", THIN, ids=_id)
def test_rows_past_the_edge_are_skipped_where_no_tile_is_whole(cc, case):
    settings, shape, copies = case
    with tuning(settings):
        (found, _), = forward_instances(cc, shape)
        assert found[-1] == copies
        tile = found[4:6]
        rows = [1] * (3 - len(shape[3])) + [-(-n // shape[4]) for n in shape[3][:-1]]
        assert copies == all(n >= t for n, t in zip(rows, tile))
        check_operator_problem(cc, shape, seed=19)


# 2D: copies where waves share a SIMD.  Rows of the longest workgroups (16 waves) at each number of rows and voxels per lane;
# rows of one wave in few and in many workgroups, of four waves (two channel groups) once and twice to a compute unit.
IMAGES = [({"fwd.rows2d": r, "fwd.vec2d": v}, (1, 6, 1, (2 * r, {1: 1000, 2: 1022, 4: 2044}[v]), 2), int(r * v >= 3))
          for r in (2, 3, 4, 5, 6) for v in (1, 2, 4)]
IMAGES += [({}, s, c) for s, c in (
    ((1, 5, 1, (64, 64), 1), 0), ((1, 5, 1, (256, 256), 3), 0), ((1, 5, 1, (512, 512), 1), 0), ((1, 2, 1, (1024, 40), 1), 0),
    ((1, 12, 1, (1024, 256), 1), 0), ((1, 12, 1, (1024, 512), 1), 1), ((1, 3, 1, (900, 900), 4), 1), ((1, 13, 1, (900, 837), 1), 1),
    ((1, 10, 1, (700, 1000), 8), 1), ((1, 11, 1, (700, 1000), 8), 0), ((1, 4, 1, (500, 1000), 1), 0), ((8, 3, 1, (260, 256), 3), 1), ((1, 6, 2, (9, 64), 2), 0),
    ((1, 6, 2, (12, 128), 3), 0), ((1, 6, 2, (256, 256), 8), 0), ((1, 4, 2, (16, 512), 1), 0), ((3, 4, 2, (512, 512), 1), 1),
    ((1, 4, 2, (9, 333), 1), 1), ((1, 6, 2, (12, 1022), 3), 1), ((1, 6, 2, (9, 2044), 2), 1))]


@pytest.mark.parametrize("case", IMAGES, ids=_id)
def test_images_copy_weights_where_waves_share_a_simd(cc, case):
    settings, shape, copies = case
    with tuning(settings):
        (found, _), = forward_instances(cc, shape)
        assert found[-1] == copies
        check_operator_problem(cc, shape, seed=23)


# 3D: channel groups by the waves of all tiles (in brackets) and the channels, on both sides of each line; a tile of 3 x 3 rows, several volumes.
GROUPS = [((1, 3, 1, (16, 16, 32), 1), 2), ((1, 4, 1, (16, 16, 32), 1), 4), ((1, 8, 1, (16, 16, 32), 2), 4), ((1, 9, 1, (16, 16, 32), 1), 8),
          ((1, 15, 1, (40, 45, 47), 5), 8),                                                     # (225 of 3 x 3 rows)
          ((1, 9, 1, (34, 64, 40), 1), 4), ((1, 31, 1, (34, 64, 40), 1), 4), ((1, 32, 1, (34, 64, 40), 1), 8), ((2, 9, 1, (32, 32, 32), 2), 8),
          ((1, 33, 1, (60, 60, 33), 1), 4),
          ((3, 9, 1, (32, 32, 32), 2), 4),                                                      # (272, 256, 450, 384)
          ((1, 7, 1, (66, 66, 33), 1), 2), ((1, 8, 1, (66, 66, 33), 1), 4), ((1, 11, 1, (80, 80, 34), 1), 2), ((1, 12, 1, (80, 80, 34), 1), 4),
          ((1, 14, 1, (96, 96, 33), 1), 2),                                                     # (561, 800, 1152)
          ((1, 4, 1, (30, 60, 70), 1), 4), ((1, 33, 1, (30, 60, 70), 1), 4), ((1, 15, 1, (36, 60, 65), 1), 2), ((1, 16, 1, (36, 60, 65), 1), 4),
          ((1, 20, 1, (60, 93, 75), 1), 2)]                                                     # (rows of two waves: 450, 540, 1440)


@pytest.mark.parametrize("case", GROUPS, ids=lambda c: _id(({}, c[0], 0)))
def test_channel_groups_by_the_size_of_a_volume(cc, case):
    shape, groups = case
    (_, lanes), = forward_instances(cc, shape)
    assert lanes == groups * -(-shape[3][-1] // 64) * 64
    check_operator_problem(cc, shape, seed=29)
