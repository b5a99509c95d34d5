"""The ordered sum of a large strict MSE where its first squares are folded one by one and where
crossing chunks fold from their run prefixes: dense binade crossings, first faults among the
first squares, and lengths around the fold's 64 squares and its limit. Bit-exact, and
first-fault-exact, against the oracle's dependent chain."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx(pcu_pkg):
    c = pcu_pkg.Context(0)
    yield c
    c.close()


def _check(ctx, pcu_pkg, p, policy):
    t = np.zeros_like(p)
    ref, rf = oracle.mse(p, t, policy=policy)
    try:
        got, fault = ctx.strict_mse(ctx.upload(p), ctx.upload(t), policy).numpy(), None
    except pcu_pkg.PcuExecutionError as e:
        f = e.tensor_fault
        fault = (f.element_index, f.reduction_index, int(f.step), int(f.kind))
    want = None if rf is None else (rf.element_index, rf.reduction_index, rf.step, rf.kind)
    assert fault == want
    if want is None:
        u = np.uint32 if p.dtype == np.float32 else np.uint64
        assert np.asarray(got).view(u).item() == np.asarray(ref).view(u).item()


@pytest.mark.parametrize("dtype", [np.float32, np.float64], ids=["f32", "f64"])
@pytest.mark.parametrize("policy", [0, 1, 2])
@pytest.mark.parametrize("n", [4 * 8192 + 77, 8192, 4096])
def test_first_squares(ctx, pcu_pkg, dtype, policy, n):
    rng = np.random.default_rng(3)
    info = np.finfo(dtype)
    base = rng.uniform(-1, 1, n).astype(dtype)
    for first in (0, 1, 63, 64, 65, 1000, 4000, 4095, 4096, 5000):
        if first + 3 > n:
            continue
        p = base.copy()
        p[:first] = 0  # the total leaves +0 at square `first`
        _check(ctx, pcu_pkg, p, policy)
        # A total that stays subnormal, an overflowing Add and a steep climb from there.
        q = p.copy()
        q[first] = dtype(2.0 ** ((info.minexp - 3) // 2))
        q[first + 1:first + 40] = 0
        _check(ctx, pcu_pkg, q, policy)
        q = p.copy()
        q[first:first + 3] = np.sqrt(info.max) * dtype(0.8)
        _check(ctx, pcu_pkg, q, policy)
        # A binade every few squares, for as far as the type's range carries it.
        steps = np.minimum(np.arange(n - first) / 7.0, info.maxexp / 2 - 40)
        q = p.copy()
        q[first:] = np.exp2(steps - 20).astype(dtype)
        _check(ctx, pcu_pkg, q, policy)


@pytest.mark.parametrize("dtype", [np.float32, np.float64], ids=["f32", "f64"])
def test_lengths_about_the_one_workgroup_kernel(ctx, pcu_pkg, dtype):
    rng = np.random.default_rng(9)
    for n in (1, 63, 65, 512, 513, 4095, 4096, 4097, 4160, 4161, 8191, 8192, 8193, 8192 + 63, 12289,
              16385, 40960 + 15):
        _check(ctx, pcu_pkg, rng.normal(0, 1, n).astype(dtype), 0)
        # Whole counts: a crossing at every power of two, at run and chunk edges.
        _check(ctx, pcu_pkg, np.ones(n, dtype), 0)
        # A first Subtract fault late in each quarter of the last chunk.
        for at in {n - 1, n - n // 4 - 1, n // 2}:
            p = rng.normal(0, 1, n).astype(dtype)
            p[at] = np.inf
            _check(ctx, pcu_pkg, p, 0)


@pytest.mark.parametrize("dtype", [np.float32, np.float64], ids=["f32", "f64"])
@pytest.mark.parametrize("policy", [0, 1, 2])
@pytest.mark.parametrize("n", [61, 121, 2048, 2049])
def test_first_squares_of_short_inputs(ctx, pcu_pkg, dtype, policy, n):
    test_first_squares(ctx, pcu_pkg, dtype, policy, n)


@pytest.mark.parametrize("dtype", [np.float32, np.float64], ids=["f32", "f64"])
@pytest.mark.parametrize("policy", [0, 1, 2])
def test_lengths_about_the_one_wave_kernel(ctx, pcu_pkg, dtype, policy):
    """Lengths about its chunks of 60 (binary64 30) squares, its four waves and its limit: random,
    whole counts, squares all zero, a first fault of each kind at the first, a middle and the last
    element."""
    rng = np.random.default_rng(13)
    info = np.finfo(dtype)
    for n in (1, 2, 29, 30, 31, 59, 60, 61, 119, 120, 121, 255, 256, 257, 2047, 2048, 2049):
        p = rng.normal(0, 1, n).astype(dtype)
        _check(ctx, pcu_pkg, p, policy)
        _check(ctx, pcu_pkg, np.ones(n, dtype), policy)
        _check(ctx, pcu_pkg, np.zeros(n, dtype), policy)
        for at in {0, n // 2, n - 1}:
            # Subtract of a NaN; a square that overflows, is tiny, is exactly subnormal; a mean that is.
            for special in (np.nan, info.max, np.sqrt(info.tiny) * dtype(0.7), dtype(2.0 ** ((info.minexp - 3) // 2))):
                q = p.copy()
                q[at] = special
                _check(ctx, pcu_pkg, q, policy)
                q[:] = 0
                q[at] = special
                _check(ctx, pcu_pkg, q, policy)
