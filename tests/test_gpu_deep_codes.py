"""1x1 layers of many channels and few pixels (patch_sums_deep_body in tf-approximate_amd/csrc/prepass_kernels.hip): the codes that
go out of LDS beside the chains, in every layout a kernel reads them in.  Floats bit-equal to the oracle's."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

CASES = [
    ((1, 7, 7, 512), 24),        # 8 pixels a workgroup, the last one with one
    ((5, 5, 9, 516), 16),        # a pass of one quad behind two whole ones
    ((70, 13, 11, 772), 8),      # 16 pixels a workgroup, ten in the last one
    ((64, 14, 14, 1024), 9),     # images that count as one row
    ((65, 14, 14, 640), 12),     # ... and that do not
]


@pytest.mark.parametrize("route", ["rows", "own_rows", "vector_alus"])
@pytest.mark.parametrize("xs,co", CASES, ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else str(v))
def test_floats_bit_equal(pkg, oracle, xs, co, route):
    print("case", xs, co, route, flush=True)
    rng = np.random.RandomState(sum(xs))
    x = (rng.standard_normal(xs) * 0.4 + 0.3).astype(np.float32)
    f = (rng.standard_normal((1, 1, xs[3], co)) * 0.2).astype(np.float32)
    table, mm = pkg.synth.table_random(3), (-0.8, 1.4, -0.5, 0.5)
    op = pkg.ApproxConv2DWithMinMaxVars([1, 1, 1, 1], 8, table, "SAME")
    pkg.ops.set_preexpand(-1 if route == "vector_alus" else 0)
    pkg.ops.set_matrix_rows({"rows": 1, "own_rows": 2}.get(route, 0))
    try:
        got = op(torch.from_numpy(x).to("cuda:0"), torch.from_numpy(f).to("cuda:0"), *mm).cpu().numpy()
    finally:
        pkg.ops.set_matrix_rows(0)
        pkg.ops.set_preexpand(0)
    rc, want, _ = oracle.conv2d_fast(table, x, f, *mm, strides=(1, 1), padding="SAME", dilations=(1, 1), threads=8)
    assert rc == 0 and np.array_equal(got, want)
