"""Which layers run as one launch (axc_conv2d_direct_plan), and that their tiles fit the kernel: chunks, columns and LDS."""
import random

import pytest

LDS_BESIDE_THE_TABLE = 163840 - 131072 - 5 * 64 * 4


@pytest.fixture()
def ops(pkg):
    try:
        yield pkg.ops
    finally:
        pkg.ops.set_matrix_rows(0)
        pkg.ops.set_preexpand(0)
        pkg.ops.set_tile_columns(0)
        pkg.ops.set_merged_launches(0)
        pkg.ops.profile_enable(False)


def test_small_layers_take_it_and_large_ones_do_not(ops):
    assert ops.conv2d_direct_plan((1, 32, 32, 16), (3, 3, 16, 32)) is not None
    assert ops.conv2d_direct_plan((1, 32, 32, 16), (3, 3, 16, 32), layer=True) is not None
    assert ops.conv2d_direct_plan((1, 1, 1, 1), (1, 1, 1, 1)) is not None
    assert ops.conv2d_direct_plan((64, 56, 56, 64), (3, 3, 64, 64)) is None
    assert ops.conv2d_direct_plan((128, 32, 32, 16), (3, 3, 16, 16)) is None
    assert ops.conv2d_direct_plan((0, 8, 8, 4), (3, 3, 4, 4)) is None


def test_pinned_forms_do_without(ops):
    xs, fs = (1, 32, 32, 16), (3, 3, 16, 32)
    for mode in (1, 2, 3):
        ops.set_matrix_rows(mode)
        assert ops.conv2d_direct_plan(xs, fs) is None
    ops.set_matrix_rows(0)
    ops.set_preexpand(-1)
    assert ops.conv2d_direct_plan(xs, fs) is None
    ops.set_preexpand(0)
    ops.set_tile_columns(32)
    assert ops.conv2d_direct_plan(xs, fs) is None


def test_merged_launches(ops):
    """Pinned off, layers run as they would without; with the timers on only where that is asked for."""
    xs, fs = (1, 32, 32, 16), (3, 3, 16, 32)
    plan, without = ops.conv2d_direct_plan(xs, fs), (ops.conv2d_matrix_plan(xs, fs), ops.conv2d_tile_plan(xs, fs))
    ops.profile_enable(True)
    assert ops.conv2d_direct_plan(xs, fs) is None
    ops.set_merged_launches(1)
    assert ops.conv2d_direct_plan(xs, fs) == plan
    ops.profile_enable(False)
    assert ops.conv2d_direct_plan(xs, fs) == plan
    ops.set_merged_launches(-1)
    assert ops.conv2d_direct_plan(xs, fs) is None
    assert (ops.conv2d_matrix_plan(xs, fs), ops.conv2d_tile_plan(xs, fs)) == without
    ops.set_matrix_rows(4)
    assert ops.conv2d_direct_plan(xs, fs) is None
    for mode in (-2, 2):
        with pytest.raises(ValueError):
            ops.set_merged_launches(mode)


@pytest.mark.parametrize("seed", range(4))
def test_tiles_fit_the_kernel(ops, seed):
    rng = random.Random(seed)
    ops.set_matrix_rows(4)
    for _ in range(300):
        k = rng.choice((1, 1, 2, 3, 5, 7))
        h, w, c, co = rng.randint(k, 40), rng.randint(k, 40), rng.randint(1, 600), rng.randint(1, 600)
        n, stride = rng.randint(1, 40), rng.choice((1, 1, 2, 3))
        case = (n, h, w, c), (k, k, c, co), (1, stride, stride, 1), rng.choice(("SAME", "VALID"))
        p = ops.conv2d_direct_plan(*case, layer=rng.random() < 0.3)
        assert p is not None, case
        pt, ct, kc, chunks = (p[v] for v in ("pixels_per_tile", "columns_per_tile", "elements_per_chunk", "chunks"))
        assert pt in (16, 32, 64) and 1 <= ct <= 64
        assert p["column_tiles"] * ct >= co > (p["column_tiles"] - 1) * ct
        assert kc % 8 == 0 and kc * chunks >= k * k * c > kc * (chunks - 1)
        rows = pt * (4 * kc + 16 + 2 * kc + 16 * (kc // 8 % 2 == 0)) + ct * (4 * kc + 16 + kc + 8 * (kc // 8 % 2 == 0))
        assert rows <= (LDS_BESIDE_THE_TABLE if chunks == 1 else LDS_BESIDE_THE_TABLE // 2)
        # of a chunk that is not the only one a copying thread holds two quads of either kind
        assert chunks == 1 or max(pt, ct) * kc // 4 <= 2 * 384
        assert pt * ct * 4 <= LDS_BESIDE_THE_TABLE


# input, filter, stride, padding: layers of 2e8 products and more that the model of the other kernels puts too high
SLOWER = [
    ((30, 12, 3, 431), (3, 3, 431, 260), 1, "VALID"),          # 95 us as one launch, 75 with exchanged operands
    ((17, 11, 11, 65), (7, 7, 65, 257), 1, "VALID"),           # 103, 83
    ((3, 48, 2, 539), (7, 1, 539, 332), 1, "SAME"),           # 92, 75
    ((1, 20, 20, 457), (3, 3, 457, 270), 1, "VALID"),          # 102, 82
    ((10, 5, 6, 479), (3, 3, 479, 285), 1, "SAME"),            # 106, 85 with rows of its own
]


@pytest.mark.parametrize("xs,fs,stride,padding", SLOWER)
def test_large_layers_that_another_kernel_runs_faster(ops, xs, fs, stride, padding):
    assert ops.conv2d_direct_plan(xs, fs, (1, stride, stride, 1), padding) is None
