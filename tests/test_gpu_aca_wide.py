"""Wide blocks of the ACA (more than 1024 rows or columns): their ranks and factors do not
depend on whether a long row search suspends the block, nor on the team that resumes it."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


def _one_block(gpu, m1, m2, dim, k, ls=0.1):
    """Two point sets whose root block is the one admissible block.  In Morton order set 1
    begins with points too far from set 2 for any entry to count, a search of hundreds of rows."""
    X1 = 0.5 * O.uniform(8100 + m1, dim * m1).reshape(dim, m1)
    X2 = (0.9 if dim == 2 else 0.75) + 0.5 * O.uniform(8200 + m2, dim * m2).reshape(dim, m2)
    hm = gpu.HMatrix(X1, X2, 32 if dim == 2 else 20, 20.0, 50, 16, k)
    hm.setup()
    kern = gpu.Kernel(O.K_GAUSSIAN, 0.0, ls)
    hm.set_kernel(kern)
    assert hm.work()["aca"] == 1 and hm.work()["dense"] == 0
    return hm, kern


@pytest.mark.parametrize("m1,m2,dim", [(1500, 1300, 2), (3000, 2100, 2), (2000, 1100, 3), (9000, 2000, 2)])
def test_stop_of_a_suspended_block(gpu, m1, m2, dim):
    # the tolerance at which the stop comes one rank later, to the last bit, is the same
    # function of the factors with the row scan (the block is suspended and resumed) and without
    hm, kern = _one_block(gpu, m1, m2, dim, 24)
    hm.set_option(gpu.OPT_ACA_TOLERANCE, 2)

    def rank(scan, eps):
        hm.set_option(gpu.OPT_ACA_ROW_SCAN, scan)
        hm.data.epsilon = eps
        hm.precompute_aca()
        return hm.work()["rank_sum"]

    for target in (2, 5, 9):
        lo, hi = 1e-14, 1.0 - 1e-9  # rank(lo) > target >= rank(hi)
        assert rank(1, lo) > target >= rank(1, hi)
        while hi > np.nextafter(lo, 1.0):
            # halfway between their bit patterns
            a, b = np.float64(lo).view(np.int64), np.float64(hi).view(np.int64)
            mid = float(np.int64(a + (b - a) // 2).view(np.float64))
            lo, hi = (mid, hi) if rank(1, mid) > target else (lo, mid)
        assert rank(0, lo) > target >= rank(0, hi), (target, lo)
    hm.destroy()
    kern.free()


def _compare_scans(gpu, hm, om, ok, k, x, n_rank, bound):
    """The block's rank and product with the row scan (searches over suspended blocks) and
    without: bitwise the same, and the oracle's."""
    om.aca(ok, k)
    assert int(om.aca_factors()["keff"].sum()) == n_rank
    y = []
    for scan in (0, 1):
        hm.set_option(gpu.OPT_ACA_ROW_SCAN, scan)
        hm.precompute_aca()
        assert hm.work()["rank_sum"] == n_rank
        y.append(hm.apply(x))
    np.testing.assert_array_equal(y[0], y[1])
    ref = om.hmvp(ok, x)
    assert np.linalg.norm(y[1] - ref) <= bound * np.linalg.norm(ref)


def _two_sets(gpu, X1, X2, dim, k, kind, ls):
    hm = gpu.HMatrix(X1, X2, 32 if dim == 2 else 20, 20.0, 50, 16, k)
    hm.setup()
    kern = gpu.Kernel(kind, 0.0, ls)
    hm.set_kernel(kern)
    om = O.HMatrix(X1, X2, 32 if dim == 2 else 20, 20.0, 50, 16)
    assert om.naca == 1 and om.ndense == 0
    return hm, kern, om, O.kernel(kind, dim, 0.0, ls)


@pytest.mark.parametrize("k", [31, 32, 33, 48])
def test_resume_at_high_ranks(gpu, k):
    # k places with a hundred points each: once a row of a place is a pivot, the other 99 are
    # rejected, a search at every rank step, past the 32 U terms that a search holds in
    # registers.  (3D: the ranks are far from the block's numerical rank, so that the product
    # hardly moves with the last bits of exp; 1e-9 as for the oracle's comparisons there.)
    places = 0.5 * O.uniform(8300, 3 * k).reshape(3, k)
    X1 = np.repeat(places, 100, axis=1)
    X2 = 0.5 * O.uniform(8301, 3 * 1400).reshape(3, 1400) + np.array([0.7, 0.0, 0.0])[:, None]
    assert X1.shape[1] * X2.shape[1] > 1 << 22  # blocks of fewer entries search alone
    hm, kern, om, ok = _two_sets(gpu, X1, X2, 3, k, O.K_EXPONENTIAL, 1.0)
    _compare_scans(gpu, hm, om, ok, k, O.normal(8302, 1400), k, 1e-9)
    hm.destroy()
    kern.free()


def test_more_searches_than_rounds(gpu):
    # 5000 rows whose norms lie a little below the threshold of 1e-13, nearly all of it in
    # the first 150 of 1100 columns: a search by column segments finds every row worth
    # another look, the block evaluates it, rejects it and is suspended again some rows later,
    # until the rounds end and its team searches on alone.  The last row is acceptable.
    n1, n2 = 5000, 1100
    X1 = 1e-3 * O.uniform(8400, 2 * n1).reshape(2, n1)
    X1[:, 17] = 0.02
    d = 0.808 / np.sqrt(2.0)
    X2 = 0.95 + 1e-3 * O.uniform(8401, 2 * n2).reshape(2, n2)
    X2[:, :150] = d + 1e-4 * O.uniform(8402, 2 * 150).reshape(2, 150)
    norms = np.sqrt((np.exp(-50.0 * ((X1[:, :, None] - X2[:, None, :]) ** 2).sum(0)) ** 2).sum(1))
    low = np.delete(norms, 17)
    assert low.max() < 1e-13 and low.min() > 0.4e-13 and norms[17] > 2e-13
    hm, kern, om, ok = _two_sets(gpu, X1, X2, 2, 12, O.K_GAUSSIAN, 0.1)
    # one column of entries: each within a few eps of the oracle's, exp's argument of 33
    _compare_scans(gpu, hm, om, ok, 12, O.uniform(8403, n2), 1, 1e-12)
    hm.destroy()
    kern.free()


@pytest.mark.parametrize("prec_name", ["fp64", "mixed"])
def test_fewer_slabs_and_none(gpu, prec_name):
    # one slab at a time: the same factors; none: the memory form, the same ranks, and a
    # product that differs by the rounding of the norms at most (the factors agree as long as
    # no norm lies within rounding of its threshold, so by nothing, or as much as a changed
    # pivot row changes a product of this accuracy: 1e-8, the bar of the FP64 products)
    n, k = 20000, 16
    X = O.uniform(8500, 2 * n).reshape(2, n)
    x = O.normal(8501, n)
    kern = gpu.Kernel(O.K_EXPONENTIAL, 0.0, 0.1)
    hm = gpu.HMatrix(X, X, 32, 1.5, 50, 64, k)
    hm.set_precision(gpu.PREC_MIXED if prec_name == "mixed" else gpu.PREC_FP64)
    hm.setup()
    hm.set_kernel(kern)
    b = hm.blocks(O.WORK_ITEM_DTYPE)
    b = b[b["work_type"] == gpu.WT_ACA]
    assert (np.maximum(b["set1_u"] - b["set1_l"], b["set2_u"] - b["set2_l"]) >= 1024).sum() > 50
    got = []
    for slab in (3 << 30, 1 << 20, 1, 0):
        hm.set_option(gpu.OPT_ACA_SLAB_BYTES, slab)
        hm.precompute_aca()
        got.append((hm.work()["rank_sum"], hm.apply(x)))
    for ranks, y in got[1:]:
        assert ranks == got[0][0]
    np.testing.assert_array_equal(got[1][1], got[0][1])
    np.testing.assert_array_equal(got[2][1], got[0][1])
    assert np.linalg.norm(got[3][1] - got[0][1]) <= 1e-8 * np.linalg.norm(got[0][1])
    hm.destroy()
    kern.free()
