"""Layer calls in turn (axc_fake_approx_conv2d_ranged): what a call reports of its outputs' range is their smallest and largest
value, and the next call gets from it what it would find itself."""
import pytest
import torch

pytestmark = pytest.mark.gpu

# input, filter, stride, matrix rows mode, depthwise
CASES = [
    ((16, 56, 56, 32), (1, 1, 32, 100), 1, 1, False),    # pre-expanded rows; columns that end inside a tile
    ((33, 57, 60, 16), (3, 3, 16, 44), 1, 1, False),     # pixels that end inside a unit
    ((70, 40, 44, 32), (1, 1, 32, 72), 1, 1, False),     # 20 units a wavefront
    ((64, 56, 56, 32), (1, 1, 32, 192), 1, 1, False),    # 25, several tiles a workgroup
    ((64, 57, 60, 16), (3, 3, 16, 20), 1, 2, False),     # rows of its own
    ((60, 112, 112, 16), (3, 3, 16, 40), 2, 1, False),
    ((3, 31, 29, 70), (3, 3, 70, 1), 1, 0, True),        # channels that end inside a group, rows inside a band
    ((5, 30, 33, 64), (3, 3, 64, 1), 2, 0, True),
]


@pytest.mark.parametrize("relu", [False, True])
@pytest.mark.parametrize("case", CASES, ids=str)
def test_what_a_call_reports(pkg, case, relu):
    print("case", case, relu, flush=True)
    xs, fs, stride, mode, depthwise = case
    gen = torch.Generator(device="cuda:0")
    gen.manual_seed(sum(xs))
    x = torch.randn(xs, device="cuda:0", generator=gen)
    f = torch.randn(fs, device="cuda:0", generator=gen)
    bias = torch.linspace(-3.0, 2.0, fs[2] if depthwise else fs[3], device="cuda:0")
    layer = pkg.ops.FakeApproxConv2D((stride, stride), pkg.ops.TruthTable(pkg.synth.table_noisy(2)), "SAME",
                                     activation="relu" if relu else None, depthwise=depthwise)
    pkg.ops.set_matrix_rows(mode)
    try:
        want = layer(x, f, bias)
        got, seen = layer.call_in_turn(x, f, bias)
    finally:
        pkg.ops.set_matrix_rows(0)
    assert torch.equal(got, want)
    assert seen is not None
    pairs = seen.view(-1, 2)
    lo, hi = torch.aminmax(want)
    assert float(pairs[:, 0].min()) == float(lo) and float(pairs[:, 1].max()) == float(hi)


@pytest.mark.parametrize("taps,cols", [(1, 12), (3, 300)])     # the filter's range with the input's, and in a launch of its own
def test_the_next_call(pkg, taps, cols):
    gen = torch.Generator(device="cuda:0")
    gen.manual_seed(5)
    table = pkg.ops.TruthTable(pkg.synth.table_noisy(2))
    x = torch.randn((16, 56, 56, 32), device="cuda:0", generator=gen)
    f1 = torch.randn((1, 1, 32, 100), device="cuda:0", generator=gen)
    f2 = torch.randn((taps, taps, 100, cols), device="cuda:0", generator=gen)
    f3 = torch.randn((3, 3, 100, 1), device="cuda:0", generator=gen)
    first = pkg.ops.FakeApproxConv2D((1, 1), table, "SAME", activation="relu")
    second, third = (pkg.ops.FakeApproxConv2D((2, 2), table, "SAME", depthwise=d) for d in (False, True))
    pkg.ops.set_matrix_rows(1)
    try:
        y, seen = first.call_in_turn(x, f1)
    finally:
        pkg.ops.set_matrix_rows(0)
    assert seen is not None
    assert torch.equal(second.call_in_turn(y, f2, None, seen, False)[0], second(y, f2))
    assert torch.equal(third.call_in_turn(y, f3, None, seen, False)[0], third(y, f3))


def test_kernels_that_do_not_report(pkg):
    layer = pkg.ops.FakeApproxConv2D((1, 1), pkg.ops.TruthTable(pkg.synth.table_noisy(2)), "SAME")
    x, f = torch.randn((1, 9, 9, 16), device="cuda:0"), torch.randn((3, 3, 16, 8), device="cuda:0")
    y, seen = layer.call_in_turn(x, f)
    assert seen is None and torch.equal(y, layer(x, f))


def _reported(pkg):
    """(layer, its output, the range reported with it)"""
    gen = torch.Generator(device="cuda:0")
    gen.manual_seed(9)
    x = torch.randn((16, 56, 56, 32), device="cuda:0", generator=gen)
    f = torch.randn((1, 1, 32, 100), device="cuda:0", generator=gen)
    layer = pkg.ops.FakeApproxConv2D((1, 1), pkg.ops.TruthTable(pkg.synth.table_noisy(2)), "SAME")
    pkg.ops.set_matrix_rows(1)
    try:
        y, seen = layer.call_in_turn(x, f)
    finally:
        pkg.ops.set_matrix_rows(0)
    assert seen is not None
    return layer, y, seen


def test_a_range_is_that_of_one_tensor_as_it_was(pkg):
    """Inputs that the range is not of, or no longer of, are read; the one that it is of is not."""
    layer, y, seen = _reported(pkg)
    f = torch.randn((1, 1, 100, 24), device="cuda:0")
    other = y * 3.0
    assert torch.equal(layer.call_in_turn(other, f, None, seen, False)[0], layer(other, f))
    assert torch.equal(layer.call_in_turn(y.clone(), f, None, seen.clone(), False)[0], layer(y, f))
    seen.view(-1, 2)[:, 1] *= 2.0        # a range that the tensor does not have: what shows that it is taken
    taken = layer.call_in_turn(y, f, None, seen, False)[0]
    assert not torch.equal(taken, layer(y, f))
    for change in (lambda: y.relu_(), lambda: y.view(-1).mul_(0.25), lambda: y[3].add_(100.0)):
        change()
        assert torch.equal(layer.call_in_turn(y, f, None, seen, False)[0], layer(y, f))


def test_ranges_in_inference_mode(pkg):
    with torch.inference_mode():
        layer, y, seen = _reported(pkg)
        f = torch.randn((1, 1, 100, 24), device="cuda:0")
        y.mul_(0.5)
        assert torch.equal(layer.call_in_turn(y, f, None, seen, False)[0], layer(y, f))


def test_what_no_range_can_be_is_refused(pkg):
    layer, y, seen = _reported(pkg)
    f = torch.randn((1, 1, 100, 24), device="cuda:0")
    for bad in (seen.cpu(), seen.double(), seen[:-2], seen.view(2, -1).t(), seen.data_ptr(), [0.0, 1.0]):
        with pytest.raises(pkg.InvalidArgumentError):
            layer.call_in_turn(y, f, None, bad, False)
