"""axc_conv2d_minmax_bias_add_act: a tensor added where a layer's outputs are made, in every kernel that makes outputs and behind
those that do not take it along.  Same bits as the op and an elementwise pass, NaN and infinities included."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

MM = (-1.0, 1.0, -0.5, 0.5)

CASES = [
    # input, filter, stride, kind of route: matrix rows pinned, preexpand pinned, timers that must have run
    ((2, 8, 8, 16), (3, 3, 16, 24), 1, 4, 0, {"direct"}),
    ((1, 9, 7, 20), (3, 3, 20, 7), 1, 4, 0, {"direct"}),
    ((1, 7, 7, 512), (1, 1, 512, 260), 1, 3, 0, {"splitk_epilogue", "lutgemm_mx"}),     # operands exchanged
    ((1, 7, 7, 130), (3, 3, 130, 33), 1, 3, 0, {"splitk_epilogue", "lutgemm_mx"}),
    ((8, 14, 12, 512), (3, 3, 512, 64), 1, 2, 0, {"splitk_epilogue", "lutgemm_mx"}),    # K splits
    ((4, 16, 16, 512), (3, 3, 512, 18), 1, 2, 0, {"splitk_epilogue", "lutgemm_mx"}),    # ... columns not in fours
    ((9, 32, 32, 16), (3, 3, 16, 16), 1, 2, 0, {"lutgemm_mx"}),                         # low tiles
    ((61, 24, 28, 64), (1, 1, 64, 52), 1, 2, 0, {"lutgemm_mx"}),                        # tall ones; the last ones not full
    ((33, 56, 56, 64), (1, 1, 64, 256), 1, 1, 0, {"lutgemm_mx"}),
    ((64, 56, 56, 64), (1, 1, 64, 24), 2, 2, 0, {"lutgemm_mx"}),                        # every second pixel, gathered first
    ((65, 33, 35, 64), (3, 3, 64, 40), 1, 2, 0, {"lutgemm_mx", "add"}),                  # rows of no whole groups
    ((65, 32, 32, 64), (1, 1, 64, 42), 1, 2, 0, {"lutgemm_mx", "add"}),                  # columns not in fours
    ((140, 16, 18, 24), (1, 1, 24, 21), 1, 0, -1, {"lutgemm_expand", "add"}),
    ((160, 32, 32, 32), (1, 1, 32, 16), 1, 0, 1, {"lutgemm_px", "add"}),
    ((3, 6, 6, 640), (3, 3, 640, 32), 1, 0, -1, {"lutgemm_expand", "splitk_epilogue"}),
]


@pytest.mark.parametrize("activation", ["relu", None])
@pytest.mark.parametrize("xs,fs,stride,rows,px,names", CASES, ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else None)
def test_sum_where_the_outputs_are(pkg, xs, fs, stride, rows, px, names, activation):
    print("case", xs, fs, stride, rows, px, activation, flush=True)
    ops = pkg.ops
    rng = np.random.RandomState(sum(xs))
    x = torch.from_numpy((rng.rand(*xs) * 2 - 1).astype(np.float32)).to("cuda:0")
    f = torch.from_numpy((rng.rand(*fs) - 0.5).astype(np.float32)).to("cuda:0")
    table = ops.TruthTable(pkg.synth.table_random(4))
    op = ops.ApproxConv2DWithMinMaxVars([1, stride, stride, 1], 8, table, "SAME")
    ops.set_preexpand(px)
    ops.set_matrix_rows(rows)
    ops.profile_enable(True)
    try:
        ops.profile_reset()
        y = op(x, f, *MM)
        addend = torch.randn(y.shape, device=y.device) * y.abs().mean() - y.mean()
        flat = addend.view(-1)
        flat[::101], flat[1::103], flat[2::107] = float("nan"), float("inf"), -float("inf")
        flat[3::109] = -y.view(-1)[3::109]          # sums of +0 and -0
        ops.profile_reset()
        got = op.call_and_add(x, f, *MM, addend, activation)
        assert names <= set(ops.profile_read()), ops.profile_read()
        assert ("add" in names) == ("add" in ops.profile_read())
    finally:
        ops.profile_enable(False)
        ops.set_matrix_rows(0)
        ops.set_preexpand(0)
    want = y + addend
    if activation == "relu":
        want = torch.where(want <= 0, torch.zeros_like(want), want)
    nan = want.isnan()
    assert torch.equal(got.isnan(), nan)
    assert torch.equal(got[~nan].view(torch.int32), want[~nan].view(torch.int32))
    assert torch.equal(addend.view(-1)[3::109], -y.view(-1)[3::109])


@pytest.mark.usefixtures("launches")
def test_networks_sum_in_the_layers(pkg):
    """A network's forward pass with its sums in the layers' calls, and with a pass of its own for each."""
    from tf_approximate_amd import networks
    table = pkg.ops.TruthTable(pkg.synth.table_noisy(3))
    for program, shape in ((networks.cifar_resnet_program(2), (5, 32, 32, 3)), (networks.resnet50_program()[:26], (2, 64, 64, 3))):
        net = networks.ApproxNetwork(program, shape, table, seed=1)
        x = torch.rand(shape, device="cuda:0")
        net.forward(x, calibrate=True)
        assert len(net.adds) == sum(step[0] == "add_relu" for step in program)
        got = net.forward(x)
        adds, net.adds = net.adds, {}
        want = net.forward(x)
        assert got[1] == want[1] and torch.equal(got[0].view(torch.int32), want[0].view(torch.int32))


@pytest.mark.parametrize("xs,fs,stride,rows,px,names", [CASES[i] for i in (0, 2, 4, 5, 7, 10, 12)],
                         ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else None)
def test_an_addend_that_begins_at_any_float(pkg, xs, fs, stride, rows, px, names):
    print("case", xs, fs, stride, rows, px, flush=True)
    ops = pkg.ops
    gen = torch.Generator(device="cuda:0")
    gen.manual_seed(sum(xs))
    x = torch.rand(xs, device="cuda:0", generator=gen) * 2 - 1
    f = torch.rand(fs, device="cuda:0", generator=gen) - 0.5
    op = ops.ApproxConv2DWithMinMaxVars([1, stride, stride, 1], 8, ops.TruthTable(pkg.synth.table_random(4)), "SAME")
    ops.set_preexpand(px)
    ops.set_matrix_rows(rows)
    try:
        y = op(x, f, *MM)
        for off in (1, 2, 3):
            addend = torch.randn(y.numel() + off, device="cuda:0", generator=gen)[off:].view(y.shape)
            assert addend.is_contiguous() and addend.data_ptr() % 16 == 4 * off
            got = op.call_and_add(x, f, *MM, addend)
            assert torch.equal(got.view(torch.int32), (y + addend).view(torch.int32))
    finally:
        ops.set_matrix_rows(0)
        ops.set_preexpand(0)
