"""lutgemm_mx_kernel making its rows itself (tf-approximate_amd/csrc/lutgemm_mx_expand_kernel.hip), at the sizes where it
can go wrong: every tile height, the shortest tiles (three fills) and K splits, one and several tiles per workgroup, ragged
rows and columns, odd numbers of channel quads, the flat layout with one load and with four per group, dilation, a last K
split that is shorter.  Whole int32 sums and whole float outputs must equal, bit for bit, those of the kernel that expands
inside its tiles on the vector ALUs; the smaller cases are compared with the oracle too."""
import numpy as np
import pytest
import torch

import bench
import refimpl
import test_gpu_matrix_sums

pytestmark = pytest.mark.gpu

MM = (-1.0, 1.0, -0.5, 0.5)

# input, filter (rows, columns, columns out), stride, dilation, padding
CASES = [
    ((1, 7, 7, 64), (1, 1, 8), 1, 1, "SAME"),
    ((1, 7, 7, 512), (3, 3, 512), 1, 1, "SAME"),
    ((1, 9, 5, 33), (1, 1, 9), 1, 1, "SAME"),            # three fills, the last with one channel
    ((1, 28, 28, 40), (5, 5, 8), 1, 1, "SAME"),
    ((1, 56, 56, 256), (1, 1, 128), 1, 1, "SAME"),
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
    ((32, 56, 56, 48), (1, 1, 512), 1, 1, "SAME"),       # tiles of three fills, one after the other
    ((7, 61, 45, 20), (3, 3, 75), 2, 1, "VALID"),        # odd numbers of quads: five, three
    ((4, 40, 31, 12), (5, 5, 40), 1, 2, "SAME"),
    ((8, 57, 61, 3), (5, 5, 40), 1, 1, "SAME"),          # flat layout: a load per pixel, one load for four
    ((16, 112, 112, 2), (5, 5, 64), 2, 1, "VALID"),
]


# ... and with the operands exchanged: few pixels, none of them or of the columns in eights or fours, channel counts that are
# no multiple of four, filters whose patches leave the image, a strided 1x1 layer (gathered first), wide and tall tiles
SWAPPED = [
    ((1, 7, 7, 512), (3, 3, 512), 1, 1, "SAME"),
    ((1, 7, 7, 64), (1, 1, 1030), 1, 1, "SAME"),
    ((1, 1, 1, 300), (1, 1, 77), 1, 1, "SAME"),          # one pixel
    ((2, 5, 3, 7), (3, 3, 9), 1, 1, "SAME"),             # 63 filter elements, few columns
    ((1, 9, 5, 17), (5, 4, 260), 1, 1, "SAME"),
    ((2, 9, 11, 65), (3, 3, 50), 2, 1, "VALID"),
    ((1, 14, 14, 256), (1, 1, 1024), 1, 1, "SAME"),
    ((1, 14, 14, 128), (1, 1, 512), 2, 1, "SAME"),
    ((3, 6, 7, 20), (3, 3, 2050), 1, 2, "SAME"),
    ((1, 12, 12, 96), (3, 3, 5000), 1, 1, "SAME"),       # several tiles per workgroup
    ((1, 40, 1, 32), (7, 1, 333), 1, 1, "SAME"),
    ((1, 1, 1100, 36), (1, 3, 40), 1, 1, "SAME"),        # rows too wide for bands: patch sums of another kernel
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


@pytest.fixture()
def swapped(pkg):
    pkg.ops.set_matrix_rows(3)
    try:
        yield pkg.ops
    finally:
        pkg.ops.set_matrix_rows(0)


def _plan(ops, case):
    xs, fs, stride, dil, padding = case
    return ops.conv2d_matrix_plan(xs, (fs[0], fs[1], xs[3], fs[2]), (1, stride, stride, 1), padding, (1, dil, dil, 1))


def _compare(pkg, oracle, ops, case):
    print("case", _id(case), flush=True)
    xs, fs, stride, dil, padding = case
    table = pkg.synth.table_random(sum(xs) + fs[2])
    xd, fd = bench.device_tensors(pkg, xs, (fs[0], fs[1], xs[3], fs[2]), "uniform", seed=sum(xs) + 3 * sum(fs))
    bias = torch.linspace(-1.0, 1.0, fs[2], device=xd.device)
    op = pkg.ApproxConv2DWithMinMaxVars([1, stride, stride, 1], 8, table, padding, dilations=[1, dil, dil, 1])

    def run():
        return op.accumulators(xd, fd, *MM), op(xd, fd, *MM), op(xd, fd, *MM, bias=bias, activation="relu")
    got = run()
    ops.set_preexpand(-1)
    try:
        want = run()
    finally:
        ops.set_preexpand(0)
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


@pytest.mark.parametrize("case", CASES, ids=_id)
def test_sums_and_outputs_equal_the_expanding_kernel(pkg, oracle, own_rows, case):
    plan = _plan(own_rows, case)
    assert plan is not None and plan["own_rows"] == 1, plan
    _compare(pkg, oracle, own_rows, case)


@pytest.mark.usefixtures("launches")
@pytest.mark.parametrize("case", [c[:5] for c in test_gpu_matrix_sums.CASES], ids=_id)
def test_the_cases_of_pre_expanded_rows_as_planned(pkg, oracle, case):
    """The cases chosen for the heights of the kernel that reads pre-expanded rows, in the form that the planner picks."""
    plan = _plan(pkg.ops, case)
    assert plan is not None
    pkg.ops.profile_enable(True)
    pkg.ops.profile_reset()
    try:
        xs, fs, stride, dil, padding = case
        xd, fd = bench.device_tensors(pkg, xs, (fs[0], fs[1], xs[3], fs[2]), "uniform", seed=1)
        pkg.ApproxConv2DWithMinMaxVars([1, stride, stride, 1], 8, pkg.synth.table_exact(), padding,
                                       dilations=[1, dil, dil, 1])(xd, fd, *MM)
        names = {k for k in pkg.ops.profile_read() if k.startswith("lutgemm")}
    finally:
        pkg.ops.profile_enable(False)
    assert names == ({"lutgemm_mx"} if plan["own_rows"] else {"lutgemm_mx", "lutgemm_px"}), (plan, names)
    _compare(pkg, oracle, pkg.ops, case)


@pytest.mark.parametrize("case", SWAPPED, ids=_id)
def test_operands_exchanged(pkg, oracle, swapped, case):
    plan = _plan(swapped, case)
    assert plan is not None and plan["own_rows"] == 2, plan
    _compare(pkg, oracle, swapped, case)


# 1x1 layers whose images count as one row of pixels (in fours, in twos, each for itself), and those just outside that rule
FOLDED = [
    ((4, 7, 7, 128), (1, 1, 40), 1, 1, "SAME"),
    ((8, 15, 17, 132), (1, 1, 30), 1, 1, "VALID"),       # 1020 pixels a row
    ((6, 10, 21, 256), (1, 1, 64), 1, 1, "SAME"),        # two images
    ((3, 14, 14, 600), (1, 1, 36), 1, 1, "SAME"),        # one
    ((12, 14, 13, 256), (1, 1, 64), 2, 1, "SAME"),       # gathered 7x7 first
    ((6, 7, 7, 128), (1, 1, 40), 1, 1, "SAME"),          # six images of 7x7 are no fours
    ((4, 16, 17, 128), (1, 1, 40), 1, 1, "SAME"),        # 272 pixels in rows of 17
    ((4, 15, 19, 128), (1, 1, 40), 1, 1, "SAME"),        # 1140 pixels: too many
]


@pytest.mark.usefixtures("launches")
@pytest.mark.parametrize("mode", [0, 1, 2])
@pytest.mark.parametrize("case", FOLDED, ids=_id)
def test_rows_of_whole_images(pkg, oracle, own_rows, case, mode):
    assert np.prod(case[0]) * case[1][2] < 3e8   # so that the oracle has them
    own_rows.set_matrix_rows(mode)
    _compare(pkg, oracle, own_rows, case)


@pytest.mark.parametrize("case", [SWAPPED[0], SWAPPED[3], SWAPPED[5], SWAPPED[7]], ids=_id)
def test_layer_call_with_operands_exchanged(pkg, swapped, case):
    xs, fs, stride, _, padding = case
    table = pkg.ops.TruthTable(pkg.synth.table_noisy(5))
    gen = torch.Generator(device="cuda:0")
    gen.manual_seed(11)
    x = torch.randn(xs, device="cuda:0", generator=gen)
    f = torch.randn((fs[0], fs[1], xs[3], fs[2]), device="cuda:0", generator=gen)
    bias = torch.linspace(-1.0, 1.0, fs[2], device="cuda:0")
    layer = pkg.ops.FakeApproxConv2D((stride, stride), table, padding, activation="relu")
    got = layer(x, f, bias)
    swapped.set_preexpand(-1)
    try:
        want = layer(x, f, bias)
    finally:
        swapped.set_preexpand(0)
    assert torch.equal(got, want)


def test_every_tile_height_is_covered(own_rows):
    assert {_plan(own_rows, c)["units_per_wavefront"] for c in CASES} >= {2, 3, 4, 6, 8, 10, 12, 13, 14, 16, 18}


@pytest.mark.parametrize("mode", [2, 3])
def test_codes_entry_point_and_integer_op(pkg, own_rows, mode):
    own_rows.set_matrix_rows(mode)
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


# strided layers whose rows of codes, with their padding, would be a multiple of 128 bytes: one column more in front
WIDER = [
    ((4, 31, 31, 16), (3, 3, 24), 2, 1, "SAME"),         # 32 -> 33
    ((3, 9, 32, 20), (3, 3, 12), 2, 1, "VALID"),         # no padding of its own
    ((2, 10, 95, 24), (3, 3, 30), 3, 1, "SAME"),         # 96
    ((2, 63, 63, 12), (5, 5, 16), 4, 1, "SAME"),
    ((1, 40, 124, 8), (3, 3, 20), 2, 2, "SAME"),         # dilation
    ((3, 31, 31, 48), (3, 3, 70), 2, 1, "SAME"),
]


@pytest.mark.parametrize("mode,case", [(2, c) for c in WIDER] + [(1, ((64, 63, 63, 64), (3, 3, 64), 2, 1, "SAME")),
                                                                 (1, ((32, 32, 32, 64), (3, 3, 128), 2, 1, "VALID"))],
                         ids=lambda v: _id(v) if isinstance(v, tuple) else str(v))
def test_strided_rows_of_128_bytes(pkg, oracle, own_rows, mode, case):
    own_rows.set_matrix_rows(mode)
    plan = _plan(own_rows, case)
    assert plan is not None and plan["own_rows"] == mode - 1, plan
    _compare(pkg, oracle, own_rows, case)


# sizes that the planner would not give this form to: many pixels, up to the bounds of compute_swap_plan (65536 pixels, packed
# codes of 1 GiB on either side)
SWAPPED_FAR = [
    ((3, 57, 61, 24), (3, 3, 44), 1, 1, "SAME"),         # 10431 pixels
    ((16, 64, 64, 4), (3, 3, 12), 1, 1, "SAME"),         # 65536
    ((16, 64, 64, 908), (3, 3, 8), 1, 1, "SAME"),        # ... of 8172 elements: 1.07 GB of packed codes
    ((1, 2, 2, 1820), (3, 3, 65536), 1, 1, "SAME"),      # and as much on the filter's side
]


@pytest.mark.parametrize("case", SWAPPED_FAR, ids=_id)
def test_operands_exchanged_up_to_the_bounds(pkg, oracle, swapped, case):
    plan = _plan(swapped, case)
    assert plan is not None and plan["own_rows"] == 2, plan
    _compare(pkg, oracle, swapped, case)


# input, filter, stride, the launch behind the lookups in the exchanged form
CODES = [
    ((3, 14, 14, 48), (3, 3, 48, 40), 1, "SAME"),
    ((2, 15, 13, 64), (3, 3, 64, 24), 2, "VALID"),
    ((2, 14, 14, 130), (1, 1, 130, 36), 2, "SAME"),      # strided 1x1: codes gathered first
    ((4, 7, 7, 256), (1, 1, 256, 64), 1, "SAME"),        # images that count as one row
    ((2, 31, 31, 24), (3, 3, 24, 16), 2, "SAME"),        # one column more in front of rows of 128 bytes
]


@pytest.mark.parametrize("mode", [2, 3])
@pytest.mark.parametrize("xs,fs,stride,padding", CODES, ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else str(v))
def test_codes_as_given(pkg, oracle, own_rows, xs, fs, stride, padding, mode):
    """conv2d_codes_acc_i32 in both forms: the same sums as the kernel that expands inside its tiles, and as the oracle's."""
    print("case", xs, fs, stride, padding, mode, flush=True)
    ops = own_rows
    ops.set_matrix_rows(mode)
    plan = ops.conv2d_matrix_plan(xs, fs, (1, stride, stride, 1), padding)
    assert plan is not None and plan["own_rows"] == mode - 1, plan
    rng = np.random.RandomState(sum(xs))
    x, f = rng.randint(0, 256, xs).astype(np.uint8), rng.randint(0, 256, fs).astype(np.uint8)
    host_table = pkg.synth.table_random(9)
    table = ops.TruthTable(host_table)
    xd, fd = torch.from_numpy(x).to("cuda:0"), torch.from_numpy(f).to("cuda:0")

    def run():
        return ops.conv2d_codes_acc_i32(table, xd, fd, 77, (1, stride, stride, 1), padding)
    ops.profile_enable(True)
    ops.profile_reset()
    try:
        got = run()
        names = set(ops.profile_read())
    finally:
        ops.profile_enable(False)
    assert {k for k in names if k.startswith("lutgemm")} == {"lutgemm_mx"} and ("swap_pack" in names) == (mode == 3), names
    ops.set_preexpand(-1)
    try:
        want = run()
    finally:
        ops.set_preexpand(0)
    assert torch.equal(got, want)
    patches = refimpl.gather_patches(x, 77, fs[0], fs[1], (stride, stride), padding, (1, 1))
    assert np.array_equal(got.cpu().numpy().reshape(-1, fs[3]),
                          oracle.lut_gemm_codes(host_table, patches.reshape(-1, fs[0] * fs[1] * fs[2]), f.reshape(-1, fs[3])))


@pytest.mark.parametrize("mode", [2, 3])
@pytest.mark.parametrize("xs,fs,stride", [((2, 14, 14, 64), (1, 1, 64, 8), 5), ((1, 13, 11, 40), (3, 3, 40, 12), 4)],
                         ids=["1x1", "3x3"])
def test_integer_op_with_a_padding_origin_of_its_own(pkg, oracle, own_rows, xs, fs, stride, mode):
    """The tf1 op in both forms; its windows begin behind the image's first pixel (1x1: a padding of -1)."""
    print("case", xs, fs, stride, mode, flush=True)
    ops = own_rows
    ops.set_matrix_rows(mode)
    rng = np.random.RandomState(sum(xs) + mode)
    x, f = rng.randint(0, 256, xs).astype(np.uint8), rng.randint(0, 256, fs).astype(np.uint8)
    table = pkg.synth.table_random(4)
    ops.profile_enable(True)
    ops.profile_reset()
    try:
        out, _, _ = ops.ax_conv2d(torch.from_numpy(x).to("cuda:0"), torch.from_numpy(f).to("cuda:0"), *MM,
                                  [1, stride, stride, 1], "SAME", ops.TruthTable(table))
        names = set(ops.profile_read())
    finally:
        ops.profile_enable(False)
    assert {k for k in names if k.startswith("lutgemm")} == {"lutgemm_mx"}, names
    off_in = ops.float_to_quantized_unclamped_quint8(0.0, MM[0], MM[1])
    off_f = ops.float_to_quantized_unclamped_quint8(0.0, MM[2], MM[3])
    assert np.array_equal(out.cpu().numpy(), oracle.axconv2d_tf1(table, x, f, off_in, off_f, stride, "SAME"))


@pytest.mark.parametrize("mode", [2, 3])
def test_a_wait_that_runs_out_is_reported_by_the_next_call(pkg, own_rows, mode):
    """With a wait limit of zero polls every wavefront leaves the kernel (tests/test_lookup_mx_expand.py follows them), the
    launch returns as usual, the next call on the device reports it, once, and with the limit restored the layer is right."""
    ops = own_rows
    ops.set_matrix_rows(mode)
    xs, fs = (8, 32, 32, 64), (3, 3, 64, 64)
    plan = ops.conv2d_matrix_plan(xs, fs)
    assert plan is not None and plan["own_rows"] == mode - 1, plan
    xd, fd = bench.device_tensors(pkg, xs, fs, "uniform", seed=1)
    op = pkg.ApproxConv2DWithMinMaxVars([1, 1, 1, 1], 8, pkg.synth.table_random(2), "SAME")
    good = op.accumulators(xd, fd, *MM).clone()
    torch.cuda.synchronize()
    ops.set_wait_limit(0)
    try:
        print("launch with a wait limit of 0 polls", flush=True)
        op.accumulators(xd, fd, *MM)
        torch.cuda.synchronize()
    finally:
        ops.set_wait_limit(1 << 20)
    with pytest.raises(RuntimeError, match="gave up a wait"):
        op.accumulators(xd, fd, *MM)
    again = op.accumulators(xd, fd, *MM)
    torch.cuda.synchronize()
    assert torch.equal(again, good)
