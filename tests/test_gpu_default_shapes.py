"""Default launch shapes of one system's solvers (lanes by rows and row length,
one row slab per workgroup) against an explicit shape, at the lines of the rule."""

import numpy as np
import pytest
import scipy.sparse as sp

pytestmark = pytest.mark.gpu


def _band(n, half):
    """Symmetric band with 2 half off-diagonals, diagonally dominant: condition
    below 5 after scaling by the diagonal."""
    rng = np.random.default_rng(n + half)
    d = {}
    for k in range(1, min(half, n - 1) + 1):
        d[k] = d[-k] = -rng.uniform(0.5, 1, n - k)
    a = sp.diags(list(d.values()), list(d.keys()), shape=(n, n)).tocsr() if d else sp.csr_matrix((n, n))
    return (a + sp.diags(1.5 * np.asarray(abs(a).sum(axis=1)).ravel() + 1)).tocsr()


# half 3: 6 off-diagonal entries, 4 lanes below 16,384 rows and 2 from there;
# 5: 10 entries, 8 lanes below 32,768 rows and 4 from there; 9: 18 entries, 16 lanes
@pytest.mark.parametrize("n,half", [(1, 0), (33, 3), (255, 5), (257, 9), (16383, 3), (16384, 3), (32767, 5), (32768, 5), (40001, 9)])
@pytest.mark.parametrize("name,nch,dtype", [("pcg", 1, np.float64), ("pcg", 2, np.float64), ("pcg_mixed", 2, np.float64),
                                            ("gs", 2, np.float32), ("pcg", 8, np.float64)])
def test_default_shape_equals_an_explicit_one(n, half, name, nch, dtype):
    from nsfem_amd import cu
    a = _band(n, half)
    b = np.random.default_rng(3).uniform(-1, 1, nch * n).astype(dtype)
    target = 1e-12 if dtype == np.float64 else 1e-4
    xs = []
    for shape in (None, (8, 128)):
        s = cu.createSolver(name, nch, a, 300, target, 1, dtype=dtype)
        if shape:
            s.reshape(*shape)
        s.getRhs().upload(b)
        s.getSol().memsetZero()
        s.solve()
        xs.append(s.getSol().download().astype(np.float64))
    # true residuals: the pcg target is relative to |b|, gs' the root mean
    # square over a column (summed over the columns at most); rounding of the
    # result adds a few ulps of |A||x|
    for x in xs:
        for c in range(nch):
            bc, xc = b[c * n:(c + 1) * n].astype(np.float64), x[c * n:(c + 1) * n]
            bound = 1.01 * target * (np.sqrt(n * nch) if name == "gs" else np.linalg.norm(bc))
            bound += 8 * np.finfo(dtype).eps * np.linalg.norm(abs(a) @ abs(xc))
            assert np.linalg.norm(bc - a @ xc) <= bound


# columns x workgroups of one slab (256 / columns rows) on both sides of 12,288
# and, from 16 columns on, 32,768: one, two and four slabs
@pytest.mark.parametrize("n,nch,slabs", [(49152, 8, 1), (49153, 8, 2), (12288, 16, 1), (12289, 16, 2), (32768, 16, 2), (32769, 16, 4),
                                         (3072, 32, 1), (3073, 32, 2), (8192, 32, 2), (8193, 32, 4), (200001, 4, 1)])
@pytest.mark.parametrize("name", ["pcg_mixed", "gs"])
def test_default_slabs_of_wide_tiles(n, nch, slabs, name):
    from nsfem_amd import cu
    a = _band(n, 3)
    b = np.random.default_rng(4).uniform(-1, 1, (nch, n))
    target = 1e-11
    s = cu.createSolver(name, nch, a, 300, target, 1)
    assert s.shape() == (nch, slabs * 256 // nch) and s.sweepShape() == (nch, 256 // nch)
    s.getRhs().upload(b.ravel())
    s.getSol().memsetZero()
    s.solve()
    x = s.getSol().download().reshape(nch, n)
    # true residuals, bounded as above
    for c in range(nch):
        bound = 1.01 * target * (np.sqrt(n * nch) if name == "gs" else np.linalg.norm(b[c]))
        bound += 8 * np.finfo(np.float64).eps * np.linalg.norm(abs(a) @ abs(x[c]))
        assert np.linalg.norm(b[c] - a @ x[c]) <= bound


# a row of more than 4 x mean + 16 off-diagonal entries keeps the lanes by the
# mean row length, 8 for 6 and 10 entries: fewer make wavefronts of more rows
@pytest.mark.parametrize("half,n,lanes", [(3, 20000, 2), (5, 40001, 4)])
@pytest.mark.parametrize("name", ["pcg", "pcg_mixed", "gs"])
def test_default_lanes_of_uneven_rows(half, n, lanes, name):
    from nsfem_amd import cu
    a = _band(n, half)
    longest = 4 * 2 * half + 16
    rng = np.random.default_rng(6)
    b = rng.uniform(-1, 1, n)
    target = 1e-11
    for extra, want in ((0, lanes), (longest - 2 * half - 2, lanes), (longest, 8)):
        far = n // 2 + 100 + 3 * np.arange(extra)
        e = sp.coo_matrix((np.full(extra, -0.1), (np.full(extra, n // 2), far)), shape=(n, n)).tocsr()
        m = (a + e + e.T + sp.diags(np.asarray((abs(e) + abs(e.T)).sum(axis=1)).ravel())).tocsr()
        s = cu.createSolver(name, 1, m, 400, target, 1)
        assert s.shape() == (want, 256 // want), extra
        s.getRhs().upload(b)
        s.getSol().memsetZero()
        s.solve()
        x = s.getSol().download()
        bound = 1.01 * target * (np.sqrt(n) if name == "gs" else np.linalg.norm(b)) + 8 * np.finfo(float).eps * np.linalg.norm(abs(m) @ abs(x))
        assert np.linalg.norm(b - m @ x) <= bound
