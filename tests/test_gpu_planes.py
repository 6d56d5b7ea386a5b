"""Strided layers whose input is split by tap columns first (split_columns_kernel in tf-approximate_amd/csrc/prepass_kernels.hip):
same bits as the vector-ALU kernels', which read the input as it is, and as the same kernel's without the room for the columns."""
import ctypes

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

MM = (-1.0, 1.0, -0.5, 0.5)

CASES = [
    # input, filter, strides, padding, dilations
    ((33, 61, 63, 64), (3, 3, 64, 72), (2, 2), "SAME", (1, 1)),       # rows of 32 pixels, padding on the right
    ((99, 31, 27, 160), (3, 3, 160, 136), (2, 2), "VALID", (1, 1)),   # 13: the last group reads the next row's first ones
    ((60, 29, 28, 131), (3, 2, 131, 160), (1, 2), "SAME", (1, 1)),    # a remainder of channels; padding on one side only
    ((33, 64, 37, 36), (5, 5, 36, 64), (3, 3), "SAME", (1, 1)),       # a wider stride
    ((20, 40, 64, 32), (7, 7, 32, 40), (2, 3), "SAME", (1, 1)),       # strides that differ
    ((17, 45, 45, 48), (3, 3, 48, 80), (1, 2), "SAME", (2, 4)),       # taps four columns apart
    ((400, 29, 5, 96), (1, 3, 96, 264), (1, 2), "SAME", (1, 1)),      # rows of three pixels; no padding above or below
]


def _ids(v):
    return "x".join(map(str, v)) if isinstance(v, tuple) else str(v)


@pytest.mark.parametrize("mode", [1, 2])
@pytest.mark.parametrize("xs,fs,strides,padding,dilations", CASES, ids=_ids)
def test_by_tap_columns(pkg, xs, fs, strides, padding, dilations, mode):
    print("case", xs, fs, strides, padding, dilations, mode, flush=True)
    ops = pkg.ops
    rng = np.random.RandomState(sum(xs))
    x = torch.from_numpy((rng.rand(*xs) * 2 - 1).astype(np.float32)).to("cuda:0")
    f = torch.from_numpy((rng.rand(*fs) - 0.5).astype(np.float32)).to("cuda:0")
    xc = torch.from_numpy(rng.randint(0, 256, xs).astype(np.uint8)).to("cuda:0")
    fc = torch.from_numpy(rng.randint(0, 256, fs).astype(np.uint8)).to("cuda:0")
    table = ops.TruthTable(pkg.synth.table_random(4))
    st, dl = [1, *strides, 1], [1, *dilations, 1]
    op = ops.ApproxConv2DWithMinMaxVars(st, 8, table, padding, dilations=dl)

    def run():
        y = [op(x, f, *MM), op.accumulators(x, f, *MM)]
        if dilations == (1, 1):
            y.append(ops.conv2d_codes_acc_i32(table, xc, fc, 77, st, padding))
        return y
    ops.set_preexpand(-1)
    try:
        want = run()
    finally:
        ops.set_preexpand(0)
    ops.set_matrix_rows(mode)
    ops.profile_enable(True)
    try:
        ops.profile_reset()
        timed = run()
        assert "split_columns" in ops.profile_read()
        ops.profile_enable(False)
        got = run()
    finally:
        ops.profile_enable(False)
        ops.set_matrix_rows(0)
    for g, t, w in zip(got, timed, want):
        assert torch.equal(t, w) and torch.equal(g, w)


def test_without_the_room(pkg):
    """256 bytes less than the layer asks for: the same kernel, its input as it is."""
    from tf_approximate_amd import _lib
    ops, lib = pkg.ops, _lib.load()
    rng = np.random.RandomState(2)
    x = torch.from_numpy((rng.rand(16, 57, 57, 64) * 2 - 1).astype(np.float32)).to("cuda:0")
    f = torch.from_numpy((rng.rand(3, 3, 64, 128) - 0.5).astype(np.float32)).to("cuda:0")
    table = ops.TruthTable(pkg.synth.table_random(4))
    desc = ops.make_desc(tuple(x.shape), tuple(f.shape), [1, 2, 2, 1], "SAME")
    n = ctypes.c_size_t()
    assert lib.axc_conv2d_workspace_bytes(ctypes.byref(desc), ctypes.byref(n)) == 0
    ws = torch.empty(n.value, dtype=torch.uint8, device=x.device)
    outs, names = [], []
    for less in (0, 256):
        out = torch.full((16, 29, 29, 128), float("nan"), device=x.device)
        ops.profile_enable(True)
        ops.profile_reset()
        try:
            rc = lib.axc_conv2d_minmax(table.handle, ctypes.byref(desc), x.data_ptr(), f.data_ptr(), *MM, out.data_ptr(),
                                       ws.data_ptr(), n.value - less, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
            torch.cuda.synchronize()
            names.append(set(ops.profile_read()))
        finally:
            ops.profile_enable(False)
        assert rc == 0, lib.axc_last_error()
        outs.append(out)
    assert "split_columns" in names[0] and "split_columns" not in names[1]
    assert "lutgemm_mx" in names[0] and "lutgemm_mx" in names[1]
    assert not bool(outs[0].isnan().any()) and torch.equal(outs[0], outs[1])
