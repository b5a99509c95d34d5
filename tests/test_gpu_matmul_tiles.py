"""The strict F32 MatMul's tiles at the sizes where they can go wrong: the edges of the 32 x 32, 64 x
64 and bound-checked 128 x 128 tiles, slabs of 32 (16) k and their remainders, operands whose rows are and are
not 16-byte aligned, in every layout, under every policy, with and without faults. Outputs are
bit-exact and first faults exact against the oracle."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx(pcu_pkg):
    c = pcu_pkg.Context(0)
    # The screened tile kernels at every size (the default engine computes outputs of few cells
    # in one launch).
    c.set_matmul_engine("mfma_products")
    yield c
    c.close()


def _check(ctx, pcu_pkg, a, b, tl, tr, policy):
    ref, rf = oracle.matmul(a, b, tl, tr, policy=policy)
    try:
        got = ctx.strict_matmul(ctx.upload(a), ctx.upload(b), tl, tr, policy).numpy()
        fault = None
    except pcu_pkg.PcuExecutionError as e:
        f = e.tensor_fault
        fault = (f.element_index, f.reduction_index, int(f.step), int(f.kind))
    want = None if rf is None else (rf.element_index, rf.reduction_index, rf.step, rf.kind)
    assert fault == want, (a.shape, b.shape, tl, tr, policy)
    if want is None:
        np.testing.assert_array_equal(got.view(np.uint32), ref.view(np.uint32))


def _operands(rng, m, k, n, tl, tr):
    a = rng.uniform(-1, 1, (k, m) if tl else (m, k)).astype(np.float32)
    b = rng.uniform(-1, 1, (n, k) if tr else (k, n)).astype(np.float32)
    return a, b


# 32 x 32 tiles, up to three a CU and more; 64 x 64 tiles, two a CU; 128 x 128 tiles, two a CU.
@pytest.mark.parametrize("m,n,tile", [(1, 1, 32), (31, 33, 32), (32, 64, 32), (36, 68, 32), (65, 127, 32),
                                      (896, 1024, 32), (900, 1028, 32), (897, 1031, 32), (1408, 1408, 64),
                                      (1400, 1404, 64), (1393, 1427, 64), (4092, 2036, 128), (4089, 2041, 128)])
@pytest.mark.parametrize("tl", [False, True])
@pytest.mark.parametrize("tr", [False, True])
def test_tile_edges_and_slab_remainders(ctx, pcu_pkg, strict_tile, m, n, tile, tl, tr):
    rng = np.random.default_rng(m * 7 + n)
    small = m * n < 100000
    # None, one, two, three, four and five slabs of 32, whole and with 1 to 31 k over.
    for k in (1, 4, 31, 32, 33, 64, 68, 95, 96, 100, 127, 128, 132, 161) if small else (4, 61, 96, 132, 163):
        assert strict_tile(np.float32, m, k, n, tl, tr, engine="mfma_products") == tile
        a, b = _operands(rng, m, k, n, tl, tr)
        _check(ctx, pcu_pkg, a, b, tl, tr, 0)


@pytest.mark.parametrize("m,k,n,tile", [(70, 100, 90, 32), (68, 132, 92, 32), (901, 70, 1030, 32),
                                        (904, 100, 1032, 32), (1401, 70, 1405, 64), (1408, 100, 1404, 64),
                                        (4089, 50, 2041, 128), (4092, 52, 2036, 128)])
@pytest.mark.parametrize("policy", [0, 1, 2])
@pytest.mark.parametrize("layout", [(False, False), (False, True), (True, False), (True, True)])
def test_tiles_first_fault_and_partial_sums(ctx, pcu_pkg, strict_tile, m, k, n, tile, policy, layout):
    """Operands next to the tiles' edges replaced by values that fault (not a number, an
    overflow, a tiny product) or leave a subnormal partial sum (rejected under policy 1 only):
    in the last row, column and k, inside the slab remainder."""
    tl, tr = layout
    assert strict_tile(np.float32, m, k, n, tl, tr, policy, "mfma_products") == tile
    rng = np.random.default_rng(m + 10 * policy + 100 * tl + 1000 * tr)
    for special in (np.nan, np.float32(3e38), np.float32(1e-30), None):
        a, b = _operands(rng, m, k, n, tl, tr)
        av, bv = (a.T if tl else a), (b.T if tr else b)
        if special is None:
            # One cell's sum is 2^-130 after the first k of the remainder, exactly.
            kk = k - 3
            av[m - 1, :], bv[:, n - 1] = 0, 0
            av[m - 1, kk], bv[kk, n - 1] = np.float32(2.0 ** -70), np.float32(2.0 ** -60)
            av[m - 1, kk + 1], bv[kk + 1, n - 1] = 1, 1
        else:
            av[m - 1, k - 1] = special
            bv[k - 1, n - 1] = special
        _check(ctx, pcu_pkg, a, b, tl, tr, policy)


# F64: 64 x 64 tiles of its own, slabs of 16 k.
@pytest.mark.parametrize("m,n", [(63, 1025), (64, 1024), (65, 1026), (513, 515)])
@pytest.mark.parametrize("layout", [(False, False), (False, True), (True, False), (True, True)])
def test_f64_tile_edges_and_slab_remainders(ctx, strict_tile, m, n, layout):
    tl, tr = layout
    rng = np.random.default_rng(m + n)
    for k in (1, 2, 15, 16, 17, 32, 47, 48, 50, 64, 65, 98):
        assert strict_tile(np.float64, m, k, n, tl, tr, engine="mfma_products") == 64
        a = rng.uniform(-1, 1, (k, m) if tl else (m, k))
        b = rng.uniform(-1, 1, (n, k) if tr else (k, n))
        got = ctx.strict_matmul(ctx.upload(a), ctx.upload(b), tl, tr).numpy()
        ref, fault = oracle.matmul(a, b, tl, tr)
        assert fault is None
        np.testing.assert_array_equal(got.view(np.uint64), ref.view(np.uint64))


@pytest.mark.parametrize("dtype", [np.float32, np.float64], ids=["f32", "f64"])
@pytest.mark.parametrize("m,n", [(33, 65), (200, 130), (900, 1030)])
@pytest.mark.parametrize("layout", [(False, False), (False, True), (True, False), (True, True)])
def test_native_tile_edges(ctx, dtype, m, n, layout):
    """Each native product within gamma_k (|A| |B|), gamma_k = k u / (1 - k u), of the exact one,
    whatever the order of its sum."""
    tl, tr = layout
    rng = np.random.default_rng(m)
    u = np.finfo(dtype).eps / 2
    for k in (1, 3, 16, 31, 32, 33, 64, 100, 161):
        a = rng.uniform(-1, 1, (k, m) if tl else (m, k)).astype(dtype)
        b = rng.uniform(-1, 1, (n, k) if tr else (k, n)).astype(dtype)
        got = ctx.native_matmul(ctx.upload(a), ctx.upload(b), tl, tr)
        ctx.synchronize()
        la, lb = (a.T if tl else a).astype(np.longdouble), (b.T if tr else b).astype(np.longdouble)
        la, lb = (la, lb) if dtype == np.float64 and m < 300 else (la.astype(np.float64), lb.astype(np.float64))
        exact, size = la @ lb, abs(la) @ abs(lb)
        # The reference's own sum is rounded too where it is in binary64.
        slack = (k * u / (1 - k * u) + k * 2.0 ** -52) * size
        assert np.all(abs(got.numpy() - exact) <= slack), (k, m, n, tl, tr)
