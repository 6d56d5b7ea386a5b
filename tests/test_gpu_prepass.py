"""Branches of the pre-pass dispatch (launch_patch_sums in tf-approximate_amd/csrc/prepass_kernels.hip) against the
oracle: who packs the filter codes of a layer whose patch sums run in bands of rows."""
import numpy as np
import pytest

import gpu_util
import refimpl

pytestmark = pytest.mark.gpu

MM = (-1.0, 1.0, -0.5, 0.5)


@pytest.mark.parametrize("xs,fs,stride", [
    ((1, 7, 7, 128), (3, 3, 128, 96), 1),    # few bands: workgroups of their own pack
    ((1, 9, 9, 132), (3, 3, 132, 40), 2),
    ((40, 9, 9, 16), (3, 3, 16, 20), 1),     # many bands: their idle wavefronts pack
    ((12, 9, 9, 16), (3, 3, 16, 36), 1),
])
def test_filter_codes_packed_under_few_and_many_bands(pkg, oracle, xs, fs, stride):
    print("case", xs, fs, flush=True)
    table = pkg.synth.table_random(sum(xs))
    x, f, _, _ = refimpl.grid_case(pkg, xs, fs, MM, seed=sum(xs) + fs[3])
    pkg.ops.set_preexpand(-1)
    try:
        y, acc = gpu_util.run_op(pkg, table, x, f, MM, (stride, stride))
    finally:
        pkg.ops.set_preexpand(0)
    rc, y_ref, acc_ref = oracle.conv2d_fast(table, x, f, *MM, strides=(stride, stride), padding="SAME", threads=8)
    assert rc == 0
    assert np.array_equal(acc, acc_ref)
    assert refimpl.linf_rel(y, y_ref) <= 1e-5
