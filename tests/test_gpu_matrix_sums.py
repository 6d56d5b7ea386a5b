"""The LUT-GEMM kernel whose sums the matrix cores make (tf-approximate_amd/csrc/lutgemm_mx_kernel.hip), at the sizes
where it can go wrong: every tile height, tiles whose last unit is partial or missing, output rows that are no whole
groups of four, column counts that are no multiple of 8 or 4, filter positions that end inside a fill, K splits, strides,
dilation, padding on every side, the flat layout, several tiles per workgroup, and the entry points.  Whole int32 sums
and whole float outputs must equal, bit for bit, those of the kernel that expands inside its tiles (itself pinned
against the oracle by the per-layer tests); the smaller cases are compared with the oracle too."""
import numpy as np
import pytest
import torch

import bench
import gpu_util
import refimpl

pytestmark = pytest.mark.gpu

MM = (-1.0, 1.0, -0.5, 0.5)

# input, filter (rows, columns, columns out), stride, dilation, padding -> tile height, K split
CASES = [
    ((1, 7, 7, 64), (1, 1, 8), 1, 1, "SAME", 2, False),
    ((1, 7, 7, 40), (5, 5, 8), 1, 1, "SAME", 2, True),
    ((1, 7, 7, 8), (3, 3, 8), 2, 1, "VALID", 2, False),          # 18 quads: half a fill at the end
    ((16, 57, 55, 40), (3, 3, 8), 2, 1, "VALID", 2, True),
    ((3, 14, 14, 64), (1, 1, 8), 1, 1, "SAME", 3, False),
    ((3, 14, 14, 40), (5, 5, 8), 1, 1, "SAME", 3, True),
    ((16, 57, 55, 24), (1, 1, 40), 1, 1, "SAME", 4, False),      # rows of 55: three pixels in the last group
    ((1, 28, 28, 40), (5, 5, 8), 1, 1, "SAME", 4, True),
    ((16, 57, 55, 24), (3, 3, 30), 2, 1, "VALID", 4, True),      # 30 columns: single stores
    ((16, 64, 64, 24), (1, 1, 40), 1, 1, "SAME", 6, False),
    ((8, 57, 55, 40), (3, 3, 12), 1, 1, "SAME", 6, True),
    ((4, 57, 55, 40), (5, 5, 12), 1, 1, "SAME", 8, True),
    ((8, 64, 64, 64), (3, 3, 20), 1, 1, "SAME", 10, True),
    ((7, 57, 55, 64), (5, 5, 64), 1, 1, "SAME", 13, True),
    ((16, 64, 64, 40), (5, 5, 40), 1, 1, "SAME", 16, True),
    ((40, 64, 64, 16), (3, 3, 64), 1, 1, "SAME", 20, False),
    ((16, 64, 64, 16), (3, 3, 64), 1, 2, "SAME", None, None),    # dilation
    ((64, 56, 56, 64), (3, 3, 64), 1, 1, "SAME", 25, False),
    ((61, 57, 59, 32), (3, 3, 72), 1, 1, "SAME", None, None),    # ragged everything, nine column tiles
    ((32, 56, 56, 256), (1, 1, 512), 1, 1, "SAME", None, None),  # several tiles per workgroup
    # odd numbers of channel quads, whose other kernel expands the rows inside its tiles
    ((8, 57, 55, 4), (5, 5, 40), 1, 1, "SAME", 2, False),        # one quad: four taps to a step of the filter position
    ((4, 40, 31, 12), (5, 5, 40), 1, 1, "SAME", 2, True),        # three
    ((7, 61, 45, 20), (3, 3, 75), 2, 1, "VALID", 3, True),       # five
    ((5, 57, 29, 36), (3, 3, 40), 1, 1, "VALID", 4, True),       # nine
    # flat layout: the codes under a filter row are one run of bytes
    ((9, 40, 31, 9), (5, 3, 50), 1, 1, "SAME", 2, False),        # 27 bytes in seven quads, fifty columns
    ((8, 57, 61, 3), (5, 5, 40), 1, 1, "SAME", 3, False),        # three bytes between pixels: a load per pixel
    # ... and with four bytes between neighbouring outputs' pixels: one load for a group of four
    ((16, 113, 111, 2), (3, 3, 40), 2, 1, "SAME", 4, False),     # two channels, stride 2
    ((16, 112, 112, 2), (5, 5, 64), 2, 1, "VALID", 6, False),
    ((8, 225, 223, 1), (5, 8, 33), 4, 1, "SAME", 2, False),      # one channel, stride 4, ragged
    ((64, 31, 30, 1), (9, 9, 72), 4, 1, "VALID", 2, False),
]


def _id(case):
    xs, fs, stride, dil, padding = case[:5]
    return "%dx%dx%dx%d-%dx%d-to%d-s%d-d%d-%s" % (xs + fs + (stride, dil, padding))


def _plan(pkg, case):
    xs, fs, stride, dil, padding = case[:5]
    return pkg.ops.conv2d_matrix_plan(xs, (fs[0], fs[1], xs[3], fs[2]), (1, stride, stride, 1), padding, (1, dil, dil, 1))


@pytest.fixture()
def pre_expanded_rows(pkg):
    """The heights and K splits of CASES are those of the kernel that reads pre-expanded rows; where the planner would have
    it make its rows itself instead, test_gpu_matrix_rows.py runs the same cases as planned."""
    pkg.ops.set_matrix_rows(1)
    try:
        yield
    finally:
        pkg.ops.set_matrix_rows(0)


@pytest.mark.usefixtures("pre_expanded_rows")
@pytest.mark.parametrize("case", CASES, ids=_id)
def test_sums_and_outputs_equal_the_expanding_kernel(pkg, oracle, case):
    print("case", _id(case), flush=True)
    xs, fs, stride, dil, padding, height, split = case
    ops, fs4 = pkg.ops, (fs[0], fs[1], xs[3], fs[2])
    plan = _plan(pkg, case)
    assert plan is not None
    if height is not None:
        assert plan["units_per_wavefront"] == height and (plan["k_splits"] > 1) == split, plan
    table = pkg.synth.table_random(sum(xs) + fs[2])
    xd, fd = bench.device_tensors(pkg, xs, fs4, "uniform", seed=sum(xs) + 3 * sum(fs))
    bias = torch.linspace(-1.0, 1.0, fs[2], device=xd.device)
    op = pkg.ApproxConv2DWithMinMaxVars([1, stride, stride, 1], 8, table, padding, dilations=[1, dil, dil, 1])

    def run():
        return (op.accumulators(xd, fd, *MM), op(xd, fd, *MM), op(xd, fd, *MM, bias=bias, activation="relu"),
                op(xd, fd, *MM, bias=bias), op(xd, fd, *MM, activation="relu"))
    ops.profile_enable(True)
    ops.profile_reset()
    try:
        got = run()
        torch.cuda.synchronize()
        assert {k for k in ops.profile_read() if k.startswith("lutgemm")} == {"lutgemm_px", "lutgemm_mx"}
        ops.set_preexpand(-1)
        want = run()
    finally:
        ops.set_preexpand(0)
        ops.profile_enable(False)
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


@pytest.mark.usefixtures("pre_expanded_rows")
def test_every_tile_height_is_covered(pkg):
    assert {_plan(pkg, c)["units_per_wavefront"] for c in CASES} >= {2, 3, 4, 6, 8, 10, 13, 16, 20, 25}


@pytest.mark.usefixtures("launches")
def test_layer_entry_and_integer_op(pkg, oracle):
    """Ranges found on the device (zero point and constants read from memory) and the tf1 op with its own padding
    origin, which may be negative, against the oracle."""
    rng = np.random.default_rng(5)
    ops, dev = pkg.ops, gpu_util.dev()
    xs, fs = (3, 14, 14, 64), (1, 1, 64, 8)
    assert ops.conv2d_matrix_plan(xs, fs) is not None
    x = rng.uniform(-2.0, 1.0, size=xs).astype(np.float32)
    w = (rng.standard_normal(fs) * 0.3).astype(np.float32)
    bias = rng.uniform(-1, 1, size=fs[3]).astype(np.float32)
    table = pkg.synth.table_noisy(5)
    layer = pkg.FakeApproxConv2D((1, 1), table, "SAME", activation="relu")
    y = layer(torch.from_numpy(x).to(dev), torch.from_numpy(w).to(dev), torch.from_numpy(bias).to(dev)).cpu().numpy()
    r = (float(x.min()), float(x.max()), float(w.min()), float(w.max()))
    fq = pkg.fake_quant.fake_quant_with_min_max_vars
    rc, y_ref, _ = oracle.conv2d_fast(table, fq(x, r[0], r[1]), fq(w, r[2], r[3]), *r, strides=(1, 1), padding="SAME")
    assert rc == 0
    assert refimpl.linf_rel(y, np.maximum((y_ref + bias).astype(np.float32), 0.0)) <= 1e-5
    for xs, fs, stride, padding in (((1, 7, 7, 40), (5, 5, 40, 8), 1, "SAME"), ((2, 13, 13, 64), (1, 1, 64, 8), 3, "SAME"),
                                    ((1, 7, 7, 8), (3, 3, 8, 8), 2, "VALID")):
        xc = rng.integers(0, 256, size=xs).astype(np.uint8)
        fc = rng.integers(0, 256, size=fs).astype(np.uint8)
        out, _, _ = ops.ax_conv2d(torch.from_numpy(xc).to(dev), torch.from_numpy(fc).to(dev), *MM, [1, stride, stride, 1],
                                  padding, pkg.TruthTable(table))
        off_in = ops.float_to_quantized_unclamped_quint8(0.0, MM[0], MM[1])
        off_f = ops.float_to_quantized_unclamped_quint8(0.0, MM[2], MM[3])
        assert np.array_equal(out.cpu().numpy(), oracle.axconv2d_tf1(table, xc, fc, off_in, off_f, stride, padding)), xs


@pytest.mark.parametrize("xs,fs", [((1, 1, 30001, 32), (1, 3, 32, 20000)), ((2, 1, 20001, 32), (1, 1, 32, 32774))])
def test_output_rows_beyond_2_gib(pkg, xs, fs):
    """One output row takes more bytes than a store's 31-bit offset counts, and tiles begin anywhere in it."""
    print("case", xs, fs, flush=True)
    ops = pkg.ops
    assert ops.conv2d_matrix_plan(xs, fs) is not None and xs[2] % 4 != 0 and xs[2] * fs[3] * 4 > 1 << 31
    table = pkg.synth.table_random(3)
    xd, fd = bench.device_tensors(pkg, xs, fs, "uniform", seed=3)
    op = pkg.ApproxConv2DWithMinMaxVars([1, 1, 1, 1], 8, table, "SAME")
    for run in (lambda: op.accumulators(xd, fd, *MM), lambda: op(xd, fd, *MM, activation="relu").view(torch.int32)):
        got = run()
        try:
            ops.set_preexpand(-1)
            want = run()
        finally:
            ops.set_preexpand(0)
        assert torch.equal(got, want), "%d of %d differ" % (int((got != want).sum()), got.numel())


def test_a_wait_that_runs_out_is_reported_by_the_next_call(pkg):
    """With a wait limit of zero polls the first wavefront to look at a counter before its time gives up, the others
    follow when they next wait, and every wavefront leaves the kernel.  The launch itself returns as usual; the next call
    on the device reports it, once; with the limit restored the layer is right again."""
    xs, fs = (16, 64, 64, 24), (3, 3, 24, 64)
    ops = pkg.ops
    assert ops.conv2d_matrix_plan(xs, fs) is not None
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
    again = op.accumulators(xd, fd, *MM)      # reported once
    torch.cuda.synchronize()
    assert torch.equal(again, good)
