"""direct_kernel (tf-approximate_amd/csrc/direct_kernel.hip), a whole layer in one launch, at the sizes where it can go wrong:
pixels, columns and filter elements that are no whole tiles, chunks or fours, one chunk and many, several tiles per workgroup,
strides, dilation, patches that leave the image.  Whole int32 sums and whole outputs must equal, bit for bit, those of the kernel
that expands its rows on the vector ALUs; the oracle has them too."""
import numpy as np
import pytest
import torch

import bench
import refimpl

pytestmark = pytest.mark.gpu

MM = (-1.0, 1.0, -0.5, 0.5)

# input, filter (rows, columns, columns out), stride, dilation, padding
CASES = [
    ((1, 1, 1, 1), (1, 1, 1), 1, 1, "SAME"),
    ((1, 32, 32, 16), (3, 3, 32), 1, 1, "SAME"),
    ((1, 1, 1, 2048), (1, 1, 3), 1, 1, "SAME"),          # one pixel, many chunks
    ((2, 5, 3, 7), (3, 3, 9), 1, 1, "SAME"),             # channels not in fours
    ((3, 9, 11, 5), (3, 3, 7), 1, 1, "SAME"),
    ((2, 17, 13, 3), (5, 3, 9), 2, 1, "VALID"),
    ((1, 7, 7, 130), (3, 3, 70), 1, 1, "SAME"),          # a last chunk of two elements more than eights
    ((7, 61, 45, 20), (3, 3, 75), 2, 1, "VALID"),
    ((4, 20, 31, 12), (5, 5, 40), 1, 2, "SAME"),         # dilated
    ((5, 33, 2, 33), (7, 1, 65), 1, 1, "SAME"),
    ((1, 14, 14, 256), (1, 1, 1024), 1, 1, "SAME"),
    ((3, 14, 14, 64), (1, 1, 100), 2, 1, "SAME"),        # strided 1x1
    ((16, 28, 28, 8), (1, 1, 200), 1, 1, "SAME"),        # several tiles per workgroup, wide ones
    ((33, 30, 29, 3), (3, 3, 24), 1, 1, "SAME"),         # ... tall ones
    ((1, 7, 7, 512), (3, 3, 64), 1, 1, "SAME"),          # 4 608 filter elements
]


def _id(case):
    xs, fs, stride, dil, padding = case
    return "%dx%dx%dx%d-%dx%d-to%d-s%d-d%d-%s" % (xs + fs + (stride, dil, padding))


@pytest.fixture()
def direct(pkg):
    """with direct(): the call runs the kernel; outside, the one that expands its rows on the vector ALUs."""
    class Pinned:
        def __enter__(self):
            pkg.ops.set_preexpand(0)
            pkg.ops.set_matrix_rows(4)

        def __exit__(self, *exc):
            pkg.ops.set_matrix_rows(0)
            pkg.ops.set_preexpand(-1)
    pkg.ops.set_preexpand(-1)
    try:
        yield Pinned
    finally:
        pkg.ops.set_matrix_rows(0)
        pkg.ops.set_preexpand(0)


def _same(got, want):
    bad = got.contiguous().view(torch.int32) != want.contiguous().view(torch.int32)
    if got.is_floating_point():
        bad &= ~(got.isnan() & want.isnan())
    assert not bool(bad.any()), "%d of %d differ, first at %s" % (
        int(bad.sum()), bad.numel(), tuple(int(v) for v in bad.nonzero()[0]))


@pytest.mark.parametrize("case", CASES, ids=_id)
def test_sums_and_outputs(pkg, oracle, direct, case):
    print("case", _id(case), flush=True)
    xs, fs, stride, dil, padding = case
    table = pkg.synth.table_random(sum(xs) + fs[2])
    xd, fd = bench.device_tensors(pkg, xs, (fs[0], fs[1], xs[3], fs[2]), "uniform", seed=sum(xs) + 3 * sum(fs))
    bias = torch.linspace(-1.0, 1.0, fs[2], device=xd.device)
    op = pkg.ApproxConv2DWithMinMaxVars([1, stride, stride, 1], 8, table, padding, dilations=[1, dil, dil, 1])

    def run():
        return op.accumulators(xd, fd, *MM), op(xd, fd, *MM), op(xd, fd, *MM, bias=bias, activation="relu")
    with direct():
        got = run()
    for g, w in zip(got, run()):
        _same(g, w)
    rc, y_ref, acc_ref = oracle.conv2d_fast(table, xd.cpu().numpy(), fd.cpu().numpy(), *MM, strides=(stride, stride),
                                            padding=padding, dilations=(dil, dil), threads=8)
    assert rc == 0
    assert np.array_equal(got[0].cpu().numpy(), acc_ref)
    assert refimpl.linf_rel(got[1].cpu().numpy(), y_ref) <= 1e-5


@pytest.mark.parametrize("case", [CASES[1], CASES[5], CASES[8], CASES[11], CASES[13]], ids=_id)
def test_layer_call(pkg, direct, case):
    """Ranges found on the device, fake quantization of both tensors but not of what lies outside the image."""
    xs, fs, stride, dil, padding = case
    table = pkg.ops.TruthTable(pkg.synth.table_noisy(5))
    gen = torch.Generator(device="cuda:0")
    gen.manual_seed(11)
    x = torch.randn(xs, device="cuda:0", generator=gen) + 0.3
    f = torch.randn((fs[0], fs[1], xs[3], fs[2]), device="cuda:0", generator=gen)
    bias = torch.linspace(-1.0, 1.0, fs[2], device="cuda:0")
    layer = pkg.ops.FakeApproxConv2D((stride, stride), table, padding, dilation_rate=(dil, dil), activation="relu")
    with direct():
        got = layer(x, f, bias), layer(x, f)
    for g, w in zip(got, (layer(x, f, bias), layer(x, f))):
        _same(g, w)


def test_values_off_the_grid(pkg, direct):
    """Out of range, infinite, NaN, minus zero: codes clamp, sums take them as they are."""
    table = pkg.synth.table_random(1)
    gen = torch.Generator(device="cuda:0")
    gen.manual_seed(3)
    x = torch.randn((2, 13, 11, 8), device="cuda:0", generator=gen) * 2.0
    f = torch.randn((3, 3, 8, 24), device="cuda:0", generator=gen)
    x.view(-1)[::97] = float("inf")
    x.view(-1)[50::193] = float("nan")
    x.view(-1)[7::31] = -0.0
    f.view(-1)[5::211] = float("-inf")
    op = pkg.ApproxConv2DWithMinMaxVars([1, 1, 1, 1], 8, table, "SAME")
    with direct():
        got = op.accumulators(x, f, *MM), op(x, f, *MM), op(x, f, *MM, activation="relu")
    for g, w in zip(got, (op.accumulators(x, f, *MM), op(x, f, *MM), op(x, f, *MM, activation="relu"))):
        _same(g, w)


def test_tensors_that_begin_at_any_float(pkg, direct):
    table = pkg.synth.table_noisy(2)
    xs, fs = (2, 9, 9, 16), (3, 3, 16, 20)
    xb, fb = torch.rand(1 + int(np.prod(xs)), device="cuda:0"), torch.rand(3 + int(np.prod(fs)), device="cuda:0") - 0.5
    x, f = xb[1:].view(xs), fb[3:].view(fs)
    op = pkg.ApproxConv2DWithMinMaxVars([1, 1, 1, 1], 8, table, "SAME")
    with direct():
        got = op(x, f, *MM)
    _same(got, op(x, f, *MM))


@pytest.mark.parametrize("mode,launched", [(0, False), (1, True), (-1, False)])
def test_what_the_timers_time(pkg, mode, launched):
    """A small layer, and one given as codes, as a call without timers runs them (1) or part by part."""
    ops = pkg.ops
    table = ops.TruthTable(pkg.synth.table_noisy(2))
    x, f = torch.rand((1, 16, 16, 16), device="cuda:0"), torch.rand((3, 3, 16, 20), device="cuda:0") - 0.5
    codes, weights = (torch.randint(0, 256, s, dtype=torch.uint8, device="cuda:0") for s in ((7, 8, 8, 64), (1, 1, 64, 100)))
    op = pkg.ApproxConv2DWithMinMaxVars([1, 1, 1, 1], 8, table, "SAME")

    def run():
        return op(x, f, *MM), ops.conv2d_codes_acc_i32(table, codes, weights, 3)
    want = run()
    ops.set_merged_launches(mode)
    ops.profile_enable(True)
    ops.profile_reset()
    try:
        got = run()
        names = set(ops.profile_read())
    finally:
        ops.profile_enable(False)
        ops.set_merged_launches(0)
    for g, w in zip(got, want):
        _same(g, w)
    assert ("direct" in names) == launched and ("patch_sums" in names or "patch_sums_flat" in names) != launched, names
    assert ("codes_prep" in names) == launched and ("codes_relayout" in names) != launched, names
