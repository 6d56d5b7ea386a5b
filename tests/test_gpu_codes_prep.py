"""codes_prep_kernel (tf-approximate_amd/csrc/prepass_kernels.hip): the three parts of the pre-pass of layers given as codes in
one launch.  While the library's timers run the parts are launched one by one: sums must be the same."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

MM = (-1.0, 1.0, -0.5, 0.5)

CASES = [
    # input, filter, stride, padding
    ((3, 14, 14, 16), (3, 3, 16, 40), 1, "SAME"),        # four quads, loads of 16 bytes
    ((2, 15, 9, 20), (3, 3, 20, 24), 1, "SAME"),         # five, of 4; an odd number of blocks of pixels
    ((5, 13, 7, 33), (3, 3, 33, 9), 2, "VALID"),         # nine, byte by byte
    ((1, 40, 31, 70), (1, 5, 70, 17), 1, "SAME"),        # two rows of blocks
    ((7, 8, 8, 64), (1, 1, 64, 100), 1, "SAME"),
]


@pytest.mark.parametrize("mode", [1, 2])
@pytest.mark.parametrize("xs,fs,stride,padding", CASES, ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else str(v))
def test_one_launch_and_three(pkg, xs, fs, stride, padding, mode):
    print("case", xs, fs, stride, padding, mode, flush=True)
    ops = pkg.ops
    rng = np.random.RandomState(sum(xs))
    x = torch.from_numpy(rng.randint(0, 256, xs).astype(np.uint8)).to("cuda:0")
    f = torch.from_numpy(rng.randint(0, 256, fs).astype(np.uint8)).to("cuda:0")
    table = ops.TruthTable(pkg.synth.table_random(4))

    def run():
        return (ops.ax_conv2d(x, f, *MM, [1, stride, stride, 1], padding, table)[0],
                ops.conv2d_codes_acc_i32(table, x, f, 77, (1, stride, stride, 1), padding))
    ops.set_matrix_rows(mode)
    try:
        got = run()
        ops.profile_enable(True)
        ops.profile_reset()
        want = run()
    finally:
        ops.profile_enable(False)
        ops.set_matrix_rows(0)
    for g, w in zip(got, want):
        assert torch.equal(g, w)
