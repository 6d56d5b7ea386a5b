"""depthwise_lut_window_kernel (tf-approximate_amd/csrc/depthwise_kernel.hip): 5x5, 5x1 and 3x1 filters at strides 1 and 2
(and the 3x3 kernel's column segments), against the depthwise oracle, int32 sums and floats bit for bit: images smaller than
a band or a window, last bands, segments and channel groups that are incomplete, both paddings, inputs off the quantization
grid, bias and ReLU, the layer call."""
import numpy as np
import pytest
import torch

import gpu_util

pytestmark = pytest.mark.gpu

MM = (-0.9, 1.3, -0.5, 0.5)
CASES = [(xs, k, s, padding) for k in ((5, 5), (5, 1), (3, 1)) for xs, s, padding in [
    ((2, 7, 9, 13), 1, "SAME"), ((1, 5, 5, 8), 1, "VALID"), ((3, 17, 30, 40), 1, "SAME"), ((1, 12, 70, 33), 2, "SAME"),
    ((2, 13, 11, 9), 2, "VALID"), ((1, 3, 2, 70), 1, "SAME"), ((9, 6, 50, 24), 2, "SAME")] if padding == "SAME" or xs[1] >= k[0]]
# the column filters, and 5x5 at stride 2, take the window kernel from 2^18 (2^17) outputs on: the same images, more of them
CASES += [((-(-(1 << 18) // (-(-xs[1] // s) * -(-xs[2] // s) * xs[3])) * 2,) + xs[1:], k, s, padding)
          for xs, k, s, padding in CASES if k[1] == 1 or s == 2]
# 3x3: column segments down to one pixel while every task has a wavefront, of 8 to 24 pixels beyond
CASES += [((1, 9, 30, 40), (3, 3), 1, "SAME"), ((2, 9, 30, 2080), (3, 3), 1, "VALID"), ((11, 9, 30, 2080), (3, 3), 1, "SAME"),
          ((1, 13, 59, 40), (3, 3), 2, "SAME"), ((2, 13, 59, 2080), (3, 3), 2, "SAME"), ((11, 13, 59, 2080), (3, 3), 2, "VALID")]


def _id(c):
    return "%dx%dx%dx%d-%dx%d-s%d-%s" % (c[0] + c[1] + c[2:])


def _tensors(case):
    xs, k, stride, padding = case
    rng = np.random.RandomState(sum(xs) + k[0] + stride)
    return ((rng.standard_normal(xs) * 0.5 + 0.2).astype(np.float32),
            (rng.standard_normal(k + (xs[3], 1)) * 0.2).astype(np.float32))


@pytest.mark.parametrize("case", CASES, ids=_id)
def test_against_the_oracle(pkg, oracle, case):
    print("case", _id(case), flush=True)
    x, f = _tensors(case)
    table = pkg.synth.table_random(7)
    y, acc = gpu_util.run_op(pkg, table, x, f, MM, (case[2], case[2]), case[3], depthwise=True)
    rc, y_ref, acc_ref = oracle.depthwise_conv2d(table, x, f, *MM, strides=(case[2], case[2]), padding=case[3], dilations=(1, 1))
    assert rc == 0
    assert np.array_equal(acc, acc_ref) and np.array_equal(y, y_ref)


@pytest.mark.parametrize("case", [CASES[0], CASES[3], CASES[9], CASES[17], CASES[-7], CASES[-14], CASES[-6], CASES[-1]], ids=_id)
def test_layer_call_and_tail(pkg, oracle, case):
    x, f = _tensors(case)
    strides = (case[2], case[2])
    table = pkg.synth.table_noisy(3)
    bias = np.linspace(-1.0, 1.0, x.shape[3]).astype(np.float32)
    xd, fd, bd = (torch.from_numpy(v).to("cuda:0") for v in (x, f, bias))
    got = pkg.FakeApproxConv2D(strides, table, case[3].lower(), activation="relu", depthwise=True)(xd, fd, bd).cpu().numpy()
    fq = pkg.fake_quant.fake_quant_with_min_max_vars
    mm = (float(x.min()), float(x.max()), float(f.min()), float(f.max()))
    rc, y, _ = oracle.depthwise_conv2d(table, fq(x, mm[0], mm[1]), fq(f, mm[2], mm[3]), *mm, strides=strides, padding=case[3],
                                       dilations=(1, 1))
    assert rc == 0
    want = np.maximum((y + bias).astype(np.float32), 0.0)
    assert np.max(np.abs(got - want)) <= 1e-5 * np.max(np.abs(want))
