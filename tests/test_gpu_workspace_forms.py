"""Layers in a workspace without the room for the form that the planner prefers (prepare_dense_for in
tf-approximate_amd/csrc/axconv_api.hip): same bits, from the allocation-free entry point and from a caller's smaller
workspace."""
import ctypes

import pytest
import torch

import bench

pytestmark = pytest.mark.gpu

MM = (-1.0, 1.0, -0.5, 0.5)


class _Layer:
    def __init__(self, pkg, xs, fs, seed):
        from tf_approximate_amd import _lib, ops
        print("case", xs, fs, flush=True)
        self.lib, self.ops, self.table = _lib.load(), ops, ops.TruthTable(pkg.synth.table_random(seed))
        self.xd, self.fd = bench.device_tensors(pkg, xs, fs, "uniform", seed=seed)
        self.desc = ops.make_desc(xs, fs, [1, 1, 1, 1], "SAME")
        n = ctypes.c_size_t()
        assert self.lib.axc_conv2d_workspace_bytes(ctypes.byref(self.desc), ctypes.byref(n)) == 0
        self.ws_bytes, self.shape = n.value, (xs[0], xs[1], xs[2], fs[3])

    def _call(self, fn, *tail):
        out = torch.full(self.shape, float("nan"), dtype=torch.float32, device=self.xd.device)
        stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
        self.ops.profile_enable(True)
        self.ops.profile_reset()
        try:
            rc = fn(self.table.handle, ctypes.byref(self.desc), self.xd.data_ptr(), self.fd.data_ptr(), *MM,
                    out.data_ptr(), *tail, stream)
            torch.cuda.synchronize()
            self.kernels = {k for k in self.ops.profile_read() if k.startswith("lutgemm")}
        finally:
            self.ops.profile_enable(False)
        return rc, out

    def in_workspace(self, nbytes):
        ws = torch.empty(max(nbytes, 256), dtype=torch.uint8, device=self.xd.device)
        return self._call(self.lib.axc_conv2d_minmax, ws.data_ptr(), nbytes)

    def static(self):
        return self._call(self.lib.axc_conv2d_minmax_static)


def test_images_that_count_as_one_row_in_the_static_workspace(pkg):
    """With six images as six rows of 1020 pixels, and as long a row of zero points behind them, the layer asks for 35.5 MB at
    least; as they are it fits into the 33.6 of the static workspace."""
    layer = _Layer(pkg, (6, 30, 34, 4500), (1, 1, 4500, 8), 3)
    rc, want = layer.in_workspace(layer.ws_bytes)
    assert rc == 0 and not bool(want.isnan().any())
    rc, got = layer.static()
    assert rc == 0, layer.lib.axc_last_error()
    assert torch.equal(got, want)
    rc, got = layer.in_workspace(32 << 20)
    assert rc == 0 and torch.equal(got, want)


@pytest.mark.parametrize("xs,fs,static_form", [
    ((32, 56, 56, 64), (3, 3, 64, 128), {"lutgemm_mx"}),                  # planned with rows (38 MB): makes them itself
    ((256, 5, 44, 128), (3, 3, 128, 16), {"lutgemm_px", "lutgemm_mx"}),   # planned with K splits (sums of 22 MB): rows, no split
], ids=["own_rows", "rows"])
def test_another_form_of_the_matrix_core_kernel(pkg, xs, fs, static_form):
    """The static workspace lacks the room for what the planner prefers, but not for another form of the same kernel."""
    layer = _Layer(pkg, xs, fs, 5)
    assert layer.ws_bytes > 32 << 20
    plan = pkg.ops.conv2d_matrix_plan(xs, fs)
    assert plan is not None and (plan["own_rows"] == 0) == ("lutgemm_px" not in static_form), plan
    rc, want = layer.in_workspace(layer.ws_bytes)
    assert rc == 0 and not bool(want.isnan().any())
    planned = layer.kernels
    assert ("lutgemm_px" in planned) == (plan["own_rows"] == 0)
    rc, got = layer.static()
    assert rc == 0, layer.lib.axc_last_error()
    assert layer.kernels == static_form
    assert torch.equal(got, want)
    # down to where none of its forms fits any more
    pkg.ops.set_preexpand(-1)
    try:
        n = ctypes.c_size_t()
        assert layer.lib.axc_conv2d_workspace_bytes(ctypes.byref(layer.desc), ctypes.byref(n)) == 0
    finally:
        pkg.ops.set_preexpand(0)
    rc, got = layer.in_workspace(n.value)
    assert rc == 0, layer.lib.axc_last_error()
    assert torch.equal(got, want)
    rc, _ = layer.in_workspace(1 << 20)
    assert rc != 0 and b"workspace too small" in layer.lib.axc_last_error()
