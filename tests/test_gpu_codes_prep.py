"""codes_prep_kernel (tf-approximate_amd/csrc/prepass_kernels.hip): the three parts of the pre-pass of layers given as codes in
one launch, against the oracle; and the parts one by one."""
import numpy as np
import pytest
import torch

import refimpl

pytestmark = pytest.mark.gpu

MM = (-1.0, 1.0, -0.5, 0.5)

CASES = [
    # input, filter, stride, padding, with pre-expanded rows (1) and / or rows of the kernel's own (2)
    ((3, 14, 14, 16), (3, 3, 16, 40), 1, "SAME", (1, 2)),        # four quads, loads of 16 bytes
    ((2, 15, 9, 20), (3, 3, 20, 24), 1, "SAME", (2,)),           # five, of 4; an odd number of blocks of pixels
    ((9, 27, 17, 20), (3, 3, 20, 40), 1, "SAME", (1, 2)),
    ((5, 13, 7, 33), (3, 3, 33, 9), 2, "VALID", (2,)),           # nine, byte by byte
    ((17, 27, 37, 35), (3, 3, 35, 40), 2, "VALID", (1, 2)),
    ((1, 40, 31, 70), (1, 5, 70, 17), 1, "SAME", (2,)),          # two rows of blocks
    ((24, 40, 31, 70), (1, 5, 70, 40), 1, "SAME", (1, 2)),
    ((7, 8, 8, 64), (1, 1, 64, 100), 1, "SAME", (1, 2)),
]


@pytest.mark.parametrize("xs,fs,stride,padding,mode", [c[:4] + (mode,) for c in CASES for mode in c[4]],
                         ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else str(v))
def test_one_launch_and_three(pkg, oracle, xs, fs, stride, padding, mode):
    print("case", xs, fs, stride, padding, mode, flush=True)
    ops = pkg.ops
    rng = np.random.RandomState(sum(xs))
    x = rng.randint(0, 256, xs).astype(np.uint8)
    f = rng.randint(0, 256, fs).astype(np.uint8)
    xd, fd = torch.from_numpy(x).to("cuda:0"), torch.from_numpy(f).to("cuda:0")
    table_np = pkg.synth.table_random(4)
    table = ops.TruthTable(table_np)
    off_in, off_f = (ops.float_to_quantized_unclamped_quint8(0.0, *MM[i:i + 2]) for i in (0, 2))
    patches = refimpl.gather_patches(x, 77, fs[0], fs[1], (stride, stride), padding, (1, 1))
    want = (oracle.axconv2d_tf1(table_np, x, f, off_in, off_f, stride, padding),
            oracle.lut_gemm_codes(table_np, patches.reshape(-1, np.prod(fs[:3])), f.reshape(-1, fs[3])).reshape(
                patches.shape[:3] + (fs[3],)))

    def check(merged):
        """Both ops against the oracle; which launches the timers saw of each."""
        ops.set_merged_launches(merged)
        names = []
        for call, w in zip((lambda: ops.ax_conv2d(xd, fd, *MM, [1, stride, stride, 1], padding, table)[0],
                            lambda: ops.conv2d_codes_acc_i32(table, xd, fd, 77, (1, stride, stride, 1), padding)), want):
            ops.profile_reset()
            assert np.array_equal(call().cpu().numpy(), w)
            names.append({k for k, v in ops.profile_read().items() if v[1]})
        return names
    ops.set_matrix_rows(mode)
    try:
        plan = ops.conv2d_matrix_plan(xs, fs, (1, stride, stride, 1), padding)
        assert plan is not None and plan["own_rows"] == mode - 1
        check(0)
        ops.profile_enable(True)
        parts = {"codes_relayout", "axconv_terms", "filter_pack"}
        tf1, codes = check(1)
        assert "codes_prep" in tf1 and not tf1 & parts, tf1
        if "quantize_flat_rows" in codes:         # (channels that do not come in fours may stay side by side)
            assert xs[3] & 3
        else:
            assert "codes_prep" in codes and not codes & parts, codes
        tf1, codes = check(-1)
        assert parts <= tf1 | {"filter_pack"} and "codes_prep" not in tf1 | codes, (tf1, codes)
    finally:
        ops.profile_enable(False)
        ops.set_merged_launches(0)
        ops.set_matrix_rows(0)
