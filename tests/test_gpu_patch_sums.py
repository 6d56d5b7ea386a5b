"""Patch sums by bands of rows (tf-approximate_amd/csrc/prepass_kernels.hip, patch_sums_rows_body) for channel counts that
are no multiple of four, that fill no whole number of reads, that do not divide the workgroup, and for inputs at any
alignment: inputs off the quantization grid, so that every patch sum's rounding shows, and float outputs bit-equal to the
oracle's."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

# input, filter rows, columns, columns out, stride, padding, floats by which the input is off a 16-byte boundary
CASES = [
    ((2, 9, 11, 65), 3, 3, 8, 1, "SAME", 0),
    ((2, 9, 11, 66), 1, 1, 8, 1, "SAME", 0),           # 1x1: no flat list for these
    ((1, 10, 7, 127), 5, 5, 12, 2, "VALID", 0),
    ((3, 8, 8, 67), 3, 1, 9, 1, "SAME", 1),
    ((1, 6, 90, 131), 3, 3, 8, 1, "SAME", 0),          # wide rows: column segments
    ((1, 6, 90, 530), 3, 3, 8, 2, "SAME", 0),
    ((2, 7, 9, 68), 3, 3, 8, 1, "SAME", 1),            # whole quads, misaligned
    ((1, 7, 30, 256), 3, 3, 8, 1, "SAME", 3),
    ((2, 7, 9, 36), 3, 3, 8, 1, "SAME", 0),            # 9 quads, padded to 10
    ((2, 7, 9, 52), 3, 3, 8, 1, "SAME", 0),            # 13 to 15
    ((2, 13, 9, 92), 3, 3, 8, 2, "SAME", 0),           # 23 to 24
    ((2, 7, 9, 24), 5, 5, 8, 1, "SAME", 0),            # batches of 6, 5, 4
    ((2, 7, 9, 20), 3, 3, 8, 1, "VALID", 0),
    ((2, 7, 9, 16), 3, 3, 8, 1, "VALID", 0),
    ((2, 7, 9, 12), 3, 3, 8, 1, "VALID", 0),           # below four quads: no batches
    ((1, 5, 6, 1100), 3, 3, 8, 1, "SAME", 0),          # 275 quads: 275 of 512 threads copy
    ((128, 47, 47, 28), 1, 1, 8, 1, "SAME", 0),        # bands of one row: one item a thread
    ((1200, 1, 30, 67), 1, 1, 8, 1, "SAME", 0),
    ((20, 30, 214, 12), 1, 1, 8, 1, "SAME", 0),        # three
    ((30, 30, 94, 12), 3, 3, 8, 1, "SAME", 0),         # six
]


def _id(c):
    return "%dx%dx%dx%d-%dx%d-to%d-s%d-%s-off%d" % (c[0] + tuple(c[1:]))


def _tensors(case, seed):
    xs, kh, kw, co, stride, padding, off = case
    rng = np.random.RandomState(seed)
    x = (rng.standard_normal(xs) * 0.4 + 0.3).astype(np.float32)
    f = (rng.standard_normal((kh, kw, xs[3], co)) * 0.2).astype(np.float32)
    store = torch.zeros(x.size + 4, dtype=torch.float32, device="cuda:0")
    xd = store[off:off + x.size].view(xs)
    xd.copy_(torch.from_numpy(x))
    assert xd.data_ptr() % 16 == 4 * off and xd.is_contiguous()
    return x, f, xd, torch.from_numpy(f).to("cuda:0")


def _assert_patch_sums_run(pkg, call):
    """The timers name what a call without merged launches runs (conftest.launches)."""
    pkg.ops.profile_enable(True)
    pkg.ops.profile_reset()
    try:
        call()
        names = set(pkg.ops.profile_read())
    finally:
        pkg.ops.profile_enable(False)
    assert names & {"patch_sums", "patch_sums_flat"} and "direct" not in names, names


@pytest.mark.parametrize("case", CASES, ids=_id)
def test_float_outputs_bit_equal(pkg, oracle, case, launches):
    print("case", _id(case), flush=True)
    stride, padding = case[4], case[5]
    x, f, xd, fd = _tensors(case, sum(case[0]))
    table, mm = pkg.synth.table_random(3), (-0.8, 1.4, -0.5, 0.5)
    op = pkg.ApproxConv2DWithMinMaxVars([1, stride, stride, 1], 8, table, padding)
    rc, y, acc = oracle.conv2d_fast(table, x, f, *mm, strides=(stride, stride), padding=padding, dilations=(1, 1), threads=8)
    assert rc == 0
    assert np.array_equal(op.accumulators(xd, fd, *mm).cpu().numpy(), acc)
    assert np.array_equal(op(xd, fd, *mm).cpu().numpy(), y)     # the same sums in the same order: no tolerance needed
    if launches == "part_by_part":
        _assert_patch_sums_run(pkg, lambda: op(xd, fd, *mm))


@pytest.mark.parametrize("case", [CASES[0], CASES[3], CASES[4], CASES[8]], ids=_id)
def test_layer_call_equals_the_op_on_fake_quantized_tensors(pkg, case, launches):
    """The padding quads must not be fake-quantized: zero is not on the grid."""
    _, _, xd, fd = _tensors(case, 7)
    stride, padding = case[4], case[5]
    table = pkg.ops.TruthTable(pkg.synth.table_noisy(5))
    layer = pkg.ops.FakeApproxConv2D((stride, stride), table, padding)
    y = layer(xd, fd)
    if launches == "part_by_part":
        _assert_patch_sums_run(pkg, lambda: layer(xd, fd))
    lo, hi, flo, fhi = (float(v) for v in (xd.min(), xd.max(), fd.min(), fd.max()))
    fq = pkg.fake_quant.fake_quant_with_min_max_vars
    op = pkg.ApproxConv2DWithMinMaxVars([1, stride, stride, 1], 8, table, padding)
    xq = torch.from_numpy(fq(xd.cpu().numpy(), lo, hi)).to("cuda:0")
    fqd = torch.from_numpy(fq(fd.cpu().numpy(), flo, fhi)).to("cuda:0")
    assert torch.equal(y, op(xq, fqd, lo, hi, flo, fhi))
