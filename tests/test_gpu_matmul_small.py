"""The one-launch strict MatMul of few cells at the sizes where it can go wrong: the edges of its
16 x 16 blocks, of the chunks it stages (256 k for F32, 128 for F64), of the blocks it computes
(64 and 32 k) and of the groups in them, rows that are and are not 16-byte aligned, in every
layout, under every policy, with and without faults. Bit-exact against the oracle."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu

DTYPES = pytest.mark.parametrize("dtype", [np.float32, np.float64], ids=["f32", "f64"])
LAYOUTS = pytest.mark.parametrize("layout", [(False, False), (False, True), (True, False), (True, True)],
                                  ids=["nn", "nt", "tn", "tt"])


@pytest.fixture(scope="module")
def ctx(pcu_pkg):
    c = pcu_pkg.Context(0)
    yield c
    c.close()


def _check(ctx, pcu_pkg, a, b, tl, tr, policy, offset=0):
    """`offset`: elements between each operand's allocation and its first element."""
    ref, rf = oracle.matmul(a, b, tl, tr, policy=policy)
    held, args = [], []
    for x in (a, b):
        flat = ctx.upload(np.concatenate([np.zeros(offset, x.dtype), np.ascontiguousarray(x).reshape(-1)]))
        held.append(flat)
        args.append(pcu_pkg.DeviceArray(ctx, flat.ptr + offset * x.itemsize, x.shape, x.dtype))
    try:
        got = ctx.strict_matmul(args[0], args[1], tl, tr, policy).numpy()
        fault = None
    except pcu_pkg.PcuExecutionError as e:
        f = e.tensor_fault
        fault = (f.element_index, f.reduction_index, int(f.step), int(f.kind))
    for h in held:
        h.free()
    want = None if rf is None else (rf.element_index, rf.reduction_index, rf.step, rf.kind)
    assert fault == want, (a.shape, b.shape, tl, tr, policy, offset)
    if want is None:
        u = np.uint32 if a.dtype == np.float32 else np.uint64
        np.testing.assert_array_equal(got.view(u), ref.view(u))


def _operands(rng, m, k, n, tl, tr, dtype):
    a = rng.uniform(-1, 1, (k, m) if tl else (m, k)).astype(dtype)
    b = rng.uniform(-1, 1, (n, k) if tr else (k, n)).astype(dtype)
    return a, b


@DTYPES
@LAYOUTS
def test_block_chunk_and_group_edges(ctx, pcu_pkg, dtype, layout):
    tl, tr = layout
    rng = np.random.default_rng(5)
    for m, n in ((1, 1), (16, 16), (17, 15), (33, 48)):
        for k in (1, 2, 3, 4, 5, 31, 32, 33, 63, 64, 65, 127, 128, 129, 160, 255, 256, 257, 260, 511, 516):
            a, b = _operands(rng, m, k, n, tl, tr, dtype)
            _check(ctx, pcu_pkg, a, b, tl, tr, 0, offset=(m + k) % 3)


@DTYPES
@LAYOUTS
@pytest.mark.parametrize("policy", [0, 1, 2])
def test_first_fault_and_screen(ctx, pcu_pkg, dtype, layout, policy):
    """Values that fault or are screened, at the first and last k, across chunks: not a number,
    an infinity, an overflowing product, products that are tiny and inexact, exact subnormal
    ones, and rows of zeros and subnormals whose exponents the block folds itself."""
    tl, tr = layout
    rng = np.random.default_rng(11 + policy)
    info = np.finfo(dtype)
    root = dtype(2.0 ** (info.minexp // 2))
    for m, k, n in ((20, 70, 18), (16, 300, 33)):
        for special in (np.nan, np.inf, info.max, root * dtype(0.7), root * dtype(0.5),
                        info.smallest_subnormal, info.tiny * dtype(1.5), 0.0):
            for kk in (0, k - 1):
                a, b = _operands(rng, m, k, n, tl, tr, dtype)
                av, bv = (a.T if tl else a), (b.T if tr else b)
                av[m - 1, kk] = special
                bv[kk, n - 1] = special if np.isfinite(special) else 1
                _check(ctx, pcu_pkg, a, b, tl, tr, policy)
                if special == info.smallest_subnormal:
                    av[m - 1, :] = info.smallest_subnormal  # a whole row below the smallest normal
                    _check(ctx, pcu_pkg, a, b, tl, tr, policy)


@DTYPES
@LAYOUTS
@pytest.mark.parametrize("policy", [0, 1, 2])
def test_search_of_many_suspect_cells(ctx, pcu_pkg, dtype, layout, policy):
    """Every cell marked by the screen and clean; exact subnormal products everywhere (a fault
    under RejectSubnormal only) with an inexact one after them; subnormal partial sums; and faults
    of every kind in several workgroups at once, of which the lowest cell, k and step is the one."""
    tl, tr = layout
    rng = np.random.default_rng(23)
    f32 = dtype == np.float32
    low = dtype(2.0 ** (-120 if f32 else -1016))
    info = np.finfo(dtype)
    for m, k, n in ((33, 130, 50), (100, 40, 90), (18, 523, 34)):
        def base():
            a, b = _operands(rng, m, k, n, tl, tr, dtype)
            av, bv = (a.T if tl else a), (b.T if tr else b)
            av[:, 0], bv[0, :] = low, 1
            av[:, 1], bv[1, :] = 1, dtype(2.0 ** -20)
            return a, b, av, bv
        a, b, av, bv = base()
        _check(ctx, pcu_pkg, a, b, tl, tr, policy)
        av[:, 1], bv[1, :] = low, dtype(2.0 ** -9)
        _check(ctx, pcu_pkg, a, b, tl, tr, policy)
        av[m - 2, k - 1], bv[k - 1, n - 3] = low * dtype(1.3), dtype(1.3 * 2.0 ** -30)
        _check(ctx, pcu_pkg, a, b, tl, tr, policy)
        a, b, av, bv = base()
        # A sum that cancels to a subnormal at k 3 of one cell, its products normal.
        av[m - 1, :4], bv[:4, n - 1] = 0, 1
        av[m - 1, 2], av[m - 1, 3] = info.tiny * dtype(1.5), -info.tiny
        _check(ctx, pcu_pkg, a, b, tl, tr, policy)
        for _ in range(6):
            a, b, av, bv = base()
            for special in rng.choice(6, 4, replace=False):
                i, j, kk = rng.integers(m), rng.integers(n), rng.integers(2, k - 2)
                if special == 0:
                    av[i, kk] = np.nan
                elif special == 1:
                    bv[kk, j] = -np.inf
                elif special == 2:
                    av[i, kk], bv[kk, j] = info.max, 2
                elif special == 3:  # the Add overflows, not the Multiply
                    av[i, kk:kk + 2], bv[kk:kk + 2, j] = info.max, dtype(0.75)
                elif special == 4:
                    av[i, kk], bv[kk, j] = low * dtype(1.3), dtype(1.7 * 2.0 ** -30)
                else:
                    av[i, kk], bv[kk, j] = info.smallest_subnormal, dtype(0.5)
            _check(ctx, pcu_pkg, a, b, tl, tr, policy)


@DTYPES
@pytest.mark.parametrize("layout", [(False, False), (True, True)], ids=["nn", "tt"])
def test_many_workgroups_of_short_sums(ctx, pcu_pkg, strict_tile, dtype, layout):
    """Grids of more workgroups than run at once, at sums that stand in one chunk of each form and
    just past it: clean, a row of NaN after a tiny product in an earlier workgroup, and faults in
    several workgroups of which the last to be dispatched holds none of the first cells."""
    tl, tr = layout
    rng = np.random.default_rng(31)
    low = dtype(2.0 ** (-120 if dtype == np.float32 else -1016))
    per = 16 // np.dtype(dtype).itemsize
    for m, k, n in ((1000, 7, 1000), (33, 16 * per, 5000), (700, 16 * per + 1, 600), (500, 64 * per, 600),
                    (300, 64 * per + 3, 400)):
        assert strict_tile(dtype, m, k, n, tl, tr) == 16
        a, b = _operands(rng, m, k, n, tl, tr, dtype)
        av, bv = (a.T if tl else a), (b.T if tr else b)
        _check(ctx, pcu_pkg, a, b, tl, tr, 0)
        av[m - 2, k - 1] = np.nan
        bv[k - 1, n // 2] = np.inf
        _check(ctx, pcu_pkg, a, b, tl, tr, 0)
        av[m // 3, k // 2], bv[k // 2, n - 1] = low * dtype(1.3), dtype(1.7 * 2.0 ** -30)
        _check(ctx, pcu_pkg, a, b, tl, tr, 0)
        av[0, k - 1] = np.nan
        _check(ctx, pcu_pkg, a, b, tl, tr, 0)


@DTYPES
@pytest.mark.parametrize("policy", [0, 1])
def test_marked_cells_cost_a_bounded_multiple_of_the_call(ctx, pcu_pkg, dtype, policy):
    """A call whose every cell the screen marks, without a fault, takes no more than 8 times the
    clean call's time (a wave for each marked cell took 40 to 90 times as long)."""
    import time

    rng = np.random.default_rng(2)
    m, k, n = 64, 2048, 64
    a, b = _operands(rng, m, k, n, False, False, dtype)
    clean = ctx.upload(a), ctx.upload(b)
    a[:, 0], b[0, :] = dtype(2.0 ** (-120 if dtype == np.float32 else -1016)), 1
    a[:, 1], b[1, :] = 1, dtype(2.0 ** -20)
    marked = ctx.upload(a), ctx.upload(b)
    out = ctx.empty((m, n), dtype)
    best = []
    for ops in (clean, marked):
        times = []
        for _ in range(12):
            t = time.perf_counter()
            ctx.strict_matmul(ops[0], ops[1], False, False, policy, out=out)
            times.append(time.perf_counter() - t)
        best.append(min(times[2:]))
    assert best[1] < 8 * best[0], best
