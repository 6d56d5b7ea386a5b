"""lutgemm_mx_kernel making its rows itself (tf-approximate_amd/csrc/lutgemm_mx_expand_kernel.hip), at the sizes where it
can go wrong: every tile height, the shortest tiles (two fills) and K splits, one and several tiles per workgroup, ragged
rows and columns, odd numbers of channel quads, the flat layout with one load and with four per group, dilation, a last K
split that is shorter.  Whole int32 sums and whole float outputs must equal, bit for bit, those of the kernel that expands
inside its tiles on the vector ALUs; the smaller cases are compared with the oracle too."""
import numpy as np
import pytest
import torch

import bench
import refimpl

pytestmark = pytest.mark.gpu

MM = (-1.0, 1.0, -0.5, 0.5)

# input, filter (rows, columns, columns out), stride, dilation, padding
CASES = [
    ((1, 7, 7, 64), (1, 1, 8), 1, 1, "SAME"),
    ((1, 7, 7, 512), (3, 3, 512), 1, 1, "SAME"),
    ((1, 9, 5, 17), (1, 1, 9), 1, 1, "SAME"),            # two fills, the second with one channel
    ((1, 28, 28, 40), (5, 5, 8), 1, 1, "SAME"),
    ((16, 57, 55, 24), (3, 3, 30), 2, 1, "VALID"),       # four loads a group, single stores
    ((8, 57, 55, 40), (3, 3, 12), 1, 1, "SAME"),
    ((64, 7, 7, 64), (3, 3, 256), 1, 1, "SAME"),
    ((8, 64, 64, 64), (3, 3, 20), 1, 1, "SAME"),
    ((48, 8, 8, 64), (1, 1, 2048), 1, 1, "SAME"),        # 12, 13, 14 and 18 units
    ((52, 8, 8, 64), (1, 1, 2048), 1, 1, "SAME"),
    ((56, 8, 8, 64), (1, 1, 2048), 1, 1, "SAME"),
    ((72, 8, 8, 64), (1, 1, 2048), 1, 1, "SAME"),
    ((61, 57, 59, 32), (3, 3, 72), 1, 1, "SAME"),        # several tiles per workgroup, ragged everything
    ((40, 64, 64, 16), (3, 3, 64), 1, 1, "SAME"),
    ((32, 56, 56, 32), (1, 1, 512), 1, 1, "SAME"),       # tiles of two fills, one after the other
    ((7, 61, 45, 20), (3, 3, 75), 2, 1, "VALID"),        # odd numbers of quads: five, three
    ((4, 40, 31, 12), (5, 5, 40), 1, 2, "SAME"),
    ((8, 57, 61, 3), (5, 5, 40), 1, 1, "SAME"),          # flat layout: a load per pixel, one load for four
    ((16, 112, 112, 2), (5, 5, 64), 2, 1, "VALID"),
]


def _id(case):
    xs, fs, stride, dil, padding = case
    return "%dx%dx%dx%d-%dx%d-to%d-s%d-d%d-%s" % (xs + fs + (stride, dil, padding))


@pytest.fixture()
def own_rows(pkg):
    pkg.ops.set_matrix_rows(2)
    try:
        yield pkg.ops
    finally:
        pkg.ops.set_matrix_rows(0)


def _plan(ops, case):
    xs, fs, stride, dil, padding = case
    return ops.conv2d_matrix_plan(xs, (fs[0], fs[1], xs[3], fs[2]), (1, stride, stride, 1), padding, (1, dil, dil, 1))


@pytest.mark.parametrize("case", CASES, ids=_id)
def test_sums_and_outputs_equal_the_expanding_kernel(pkg, oracle, own_rows, case):
    print("case", _id(case), flush=True)
    xs, fs, stride, dil, padding = case
    plan = _plan(own_rows, case)
    assert plan is not None and plan["own_rows"] == 1, plan
    table = pkg.synth.table_random(sum(xs) + fs[2])
    xd, fd = bench.device_tensors(pkg, xs, (fs[0], fs[1], xs[3], fs[2]), "uniform", seed=sum(xs) + 3 * sum(fs))
    bias = torch.linspace(-1.0, 1.0, fs[2], device=xd.device)
    op = pkg.ApproxConv2DWithMinMaxVars([1, stride, stride, 1], 8, table, padding, dilations=[1, dil, dil, 1])

    def run():
        return op.accumulators(xd, fd, *MM), op(xd, fd, *MM), op(xd, fd, *MM, bias=bias, activation="relu")
    got = run()
    own_rows.set_preexpand(-1)
    try:
        want = run()
    finally:
        own_rows.set_preexpand(0)
    for g, w in zip(got, want):
        bad = g.view(torch.int32) != w.view(torch.int32)
        assert not bool(bad.any()), "%d of %d differ, first at %s" % (
            int(bad.sum()), bad.numel(), tuple(int(v) for v in bad.nonzero()[0]))
    if np.prod(xs) * fs[0] * fs[1] * fs[2] < 3e8:
        rc, y_ref, acc_ref = oracle.conv2d_fast(table, xd.cpu().numpy(), fd.cpu().numpy(), *MM, strides=(stride, stride),
                                                padding=padding, dilations=(dil, dil), threads=8)
        assert rc == 0
        assert np.array_equal(got[0].cpu().numpy(), acc_ref)
        assert refimpl.linf_rel(got[1].cpu().numpy(), y_ref) <= 1e-5


def test_every_tile_height_is_covered(own_rows):
    assert {_plan(own_rows, c)["units_per_wavefront"] for c in CASES} >= {2, 3, 4, 6, 8, 10, 12, 13, 14, 16, 18, 20}


def test_codes_entry_point_and_integer_op(pkg, oracle, own_rows):
    xs, fs = (3, 14, 14, 48), (3, 3, 48, 40)
    rng = np.random.RandomState(5)
    x, f = rng.randint(0, 256, xs).astype(np.uint8), rng.randint(0, 256, fs).astype(np.uint8)
    table = pkg.ops.TruthTable(pkg.synth.table_random(9))
    xd, fd = torch.from_numpy(x).to("cuda:0"), torch.from_numpy(f).to("cuda:0")
    got = own_rows.ax_conv2d(xd, fd, *MM, [1, 1, 1, 1], "SAME", table)
    own_rows.set_matrix_rows(0)
    own_rows.set_preexpand(-1)
    try:
        want = own_rows.ax_conv2d(xd, fd, *MM, [1, 1, 1, 1], "SAME", table)
    finally:
        own_rows.set_preexpand(0)
    assert torch.equal(got[0], want[0])


def test_two_layers_in_turn(pkg, own_rows):
    table = pkg.synth.table_noisy(3)
    layers = []
    for seed, (xs, fs) in enumerate([((2, 14, 14, 64), (3, 3, 64, 64)), ((1, 7, 7, 256), (1, 1, 256, 512))]):
        xd, fd = bench.device_tensors(pkg, xs, fs, "uniform", seed=seed)
        op = pkg.ApproxConv2DWithMinMaxVars([1, 1, 1, 1], 8, table, "SAME")
        layers.append((op, xd, fd, op(xd, fd, *MM).clone()))
    for _ in range(3):
        for op, xd, fd, want in layers:
            assert torch.equal(op(xd, fd, *MM), want)
