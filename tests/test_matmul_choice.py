"""Which kernel a strict MatMul takes, by the side of its output tile (16: the one launch of few
cells). The choice is made on the host, so it is checked without a GPU."""
import ctypes

import numpy as np
import pytest

IEEE, REJECT, GRADUAL = 0, 1, 2


@pytest.fixture(scope="module")
def tile(strict_tile):
    types = {"f32": np.float32, "f64": np.float64}
    return lambda dtype, *args, **kw: strict_tile(types[dtype], *args, **kw)


@pytest.mark.parametrize("engine", ["valu", "mfma_products"])
def test_a_chosen_engine_always_takes_the_tile_kernels(tile, engine):
    for dtype in ("f32", "f64"):
        for m in (1, 16, 64, 256, 1000, 4096):
            for k in (1, 8, 64, 256, 4096):
                for n in (1, 64, 512, 4096):
                    assert tile(dtype, m, k, n, engine=engine) in (32, 64, 128)


def test_no_choice_launches_more_threads_than_a_grid_holds(tile):
    """A launch holds fewer than 2^32 threads. The one-launch kernel takes one thread a cell, the
    32 x 32 and 64 x 64 binary32 tiles one for each 4 and 8 cells; outputs of that size fit the
    device's memory and run on 128 x 128 tiles."""
    threads = {16: 1 / 1, 32: 1 / 4, 64: 1 / 8, 128: 1 / 32}
    for m, k, n in ((65536, 8, 65536), (65537, 15, 70001), (1 << 20, 1, 1 << 14), (131073, 5000, 131073),
                    (185400, 5000, 185400), (1 << 18, 16, 1 << 16)):
        for policy in (IEEE, REJECT, GRADUAL):
            for dtype in ("f32", "f64"):
                assert m * n * threads[tile(dtype, m, k, n, policy=policy)] < 2 ** 32, (dtype, m, k, n)


@pytest.mark.parametrize("dtype", ["f32", "f64"])
def test_short_sums_of_many_cells_take_the_tiles(tile, dtype):
    """One launch pays for each of its 16 x 16 workgroups, however short the sum; above some 30 of
    them a CU the tile kernels are the faster at every K, at the smaller K of several too."""
    for k in (1, 8, 15, 16, 30, 32, 64, 100, 128, 256, 1024, 4096):
        for m, n in ((4096, 4096), (2048, 2048), (8192, 8192), (4096, 1024), (64, 65536)):
            assert tile(dtype, m, k, n) != 16, (m, k, n)
    for m, k, n in ((4096, 8, 512), (1024, 128, 1024), (1024, 256, 1024), (4096, 64, 512)):
        assert tile(dtype, m, k, n) != 16, (m, k, n)


def test_the_choice_counts_the_screen_where_there_is_one(tile):
    """AllowGradual needs no exponent screen, so its tiles are the faster way a little earlier."""
    for m, k, n in ((512, 256, 1024), (768, 19, 2270), (1024, 64, 1024), (512, 300, 512)):
        assert tile("f32", m, k, n, policy=GRADUAL) != 16
    for m, k, n in ((512, 8, 512), (512, 256, 512), (64, 4096, 1024)):
        for policy in (IEEE, REJECT, GRADUAL):
            assert tile("f32", m, k, n, policy=policy) == 16 and tile("f64", m, k, n, policy=policy) == 16


@pytest.mark.parametrize("dtype", ["f32", "f64"])
def test_few_cells_take_one_launch(tile, dtype):
    for m, k, n in ((64, 256, 64), (1, 1, 1), (64, 4096, 1024), (512, 8, 512), (1024, 8, 1024), (512, 64, 1024),
                    (256, 1024, 256), (64, 64, 2048), (100, 17, 300)):
        for tl in (False, True):
            for tr in (False, True):
                assert tile(dtype, m, k, n, tl, tr) == 16, (m, k, n)


def test_native_whole_tiles_need_aligned_operands(pcu_pkg):
    """A grid of whole 128 x 128 tiles is one only where both operands' rows are 16-byte aligned:
    the bound-checked form of that tile is slower than the 64 x 64 tiles at every size."""
    f = pcu_pkg.lib().pcu_internal_native_matmul_tile
    f.argtypes, f.restype = 2 * [ctypes.c_void_p] + 3 * [ctypes.c_uint64] + 2 * [ctypes.c_int], ctypes.c_int
    for tl in (0, 1):
        for tr in (0, 1):
            assert f(0x10000, 0x20000, 4096, 4096, 4096, tl, tr) == 128
            for a, b in ((0x10004, 0x20000), (0x10000, 0x20008), (0x10004, 0x20004)):
                assert f(a, b, 4096, 4096, 4096, tl, tr) == 64


@pytest.mark.gpu
@pytest.mark.parametrize("name,engine", [("auto", 0), ("valu", 1), ("mfma_products", 2)])
def test_a_context_runs_with_the_engine_it_was_given(pcu_pkg, name, engine):
    f = pcu_pkg.lib().pcu_internal_matmul_engine
    f.argtypes, f.restype = [ctypes.c_void_p], ctypes.c_int
    with pcu_pkg.Context(0) as ctx:
        ctx.set_matmul_engine(name)
        assert f(ctx.handle) == engine
