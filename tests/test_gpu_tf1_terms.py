"""The zero-point terms of the integer op (axconv_terms_kernel in tf-approximate_amd/csrc/prepass_kernels.hip) against
the oracle: every load width, tensors that begin between two words, images too wide for the LDS, windows that begin
outside, slices of K that do not fill a workgroup; added by the store of the matrix-core kernel, with and without K
splits, and by the pass behind the other kernels.  All integers: equality."""
import numpy as np
import pytest
import torch

import gpu_util

pytestmark = pytest.mark.gpu


@pytest.mark.usefixtures("launches")
@pytest.mark.parametrize("xs,fs,stride,padding,shift", [
    ((2, 9, 11, 16), (3, 3, 20), 1, "SAME", 0),       # 16-byte loads
    ((2, 9, 11, 16), (3, 3, 20), 1, "SAME", 4),       # ... which this tensor does not begin on
    ((2, 9, 11, 16), (3, 3, 20), 2, "VALID", 1),
    ((1, 7, 7, 12), (1, 1, 17), 3, "SAME", 0),
    ((3, 8, 5, 3), (5, 3, 33), 2, "SAME", 0),
    ((1, 2, 6000, 1), (3, 1, 8), 1, "SAME", 0),       # three rows of 6 000 sums do not fit
    ((1, 7, 7, 40), (5, 5, 8), 1, "SAME", 0),         # matrix-core kernel, K split
    ((16, 32, 32, 16), (3, 3, 24), 1, "SAME", 0),     # matrix-core kernel, several output rows per workgroup
])
def test_zero_point_terms(pkg, oracle, xs, fs, stride, padding, shift):
    print("case", xs, fs, stride, padding, shift, flush=True)
    ops, dev = pkg.ops, gpu_util.dev()
    rng = np.random.default_rng(sum(xs) + fs[2] + shift)
    mm = (-1.0, 0.7, -0.5, 0.9)
    x = rng.integers(0, 256, size=xs).astype(np.uint8)
    f = rng.integers(0, 256, size=(fs[0], fs[1], xs[3], fs[2])).astype(np.uint8)
    xd = torch.empty(x.size + shift, dtype=torch.uint8, device=dev)[shift:].view(xs).copy_(torch.from_numpy(x))
    table = pkg.synth.table_random(sum(xs))
    out, _, _ = ops.ax_conv2d(xd, torch.from_numpy(f).to(dev), *mm, [1, stride, stride, 1], padding, pkg.TruthTable(table))
    off_in = ops.float_to_quantized_unclamped_quint8(0.0, mm[0], mm[1])
    off_f = ops.float_to_quantized_unclamped_quint8(0.0, mm[2], mm[3])
    assert np.array_equal(out.cpu().numpy(), oracle.axconv2d_tf1(table, x, f, off_in, off_f, stride, padding))
