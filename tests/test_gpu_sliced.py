"""PCG with the approximate inverse on sliced rows in locality order (from four
channels on in CSR form, one lane per channel) against the general kernels
(two finalize launches per iteration): edges of the slices, empty and long
rows, several systems."""

import numpy as np
import pytest
import scipy.sparse as sp
import scipy.sparse.linalg as spla

pytestmark = pytest.mark.gpu


def _spd(n, seed, kind):
    """Symmetric, strictly diagonally dominant (so SPD): condition below 20."""
    rng = np.random.default_rng(seed)
    if kind == "diagonal":
        return sp.diags(rng.uniform(1, 2, n)).tocsr()
    a = sp.random(n, n, min(1.0, 6.0 / n), random_state=rng, format="lil" if kind == "long" else "csr")
    if kind == "long":  # rows of very different length, some empty off the diagonal
        for r in range(0, n, 97):
            a[r, rng.integers(0, n, min(n, 150))] = 0.3
        a[n // 2:, :] = 0
    a = a.tocsr()
    a = a + a.T
    a.setdiag(0)
    a.eliminate_zeros()
    return (a + sp.diags(np.asarray(abs(a).sum(axis=1)).ravel() * 1.2 + 1)).tocsr()


def _run(name, nch, mats, b, x0, fused, dtype, target):
    from nsfem_amd import cu
    make = cu.createSolver if len(mats) == 1 else cu.createBatchSolver
    s = make(name, nch, mats[0] if len(mats) == 1 else mats, 400, target, 1, dtype=dtype)
    s.setOption("preconditioner", 1)
    s.setOption("fusedReductions", fused)
    s.getRhs().upload(b)
    s.getSol().upload(x0)
    s.solve()
    return s, s.getSol().download().astype(np.float64)


# 64 rows are a slice; 2, 4 and 8 waves a workgroup up to 256, 1,024 and more
# slices; a window of 1,024 rows is sorted together
SIZES = [[1], [63], [64], [65], [1023], [1025], [257 * 64 + 1], [1025 * 64 + 5], [40, 1, 700, 64, 130]]
SOLVERS = [("pcg", 1, np.float64), ("pcg", 2, np.float64), ("pcg_mixed", 2, np.float64), ("pcg_mixed", 1, np.float64),
           ("pcg", 2, np.float32), ("pcg", 4, np.float64), ("pcg_mixed", 8, np.float64), ("pcg_mixed", 16, np.float64),
           ("pcg", 16, np.float32), ("pcg", 32, np.float64)]
# one or two channels and one pattern reach the largest sizes; from 262,144 rows
# on (4,096 slices) a workgroup walks its slices in more than one turn, and
# vectors of more than 8M values take twice the workgroups
CASES = [(kind, *solver, sizes) for kind in ("sparse", "long", "diagonal") for solver in SOLVERS for sizes in SIZES
         if max(sizes) < 20_000 or (kind == "sparse" and solver[1] <= 2)]
CASES += [("sparse", "pcg", 1, np.float64, [4097 * 64 + 3]), ("sparse", "pcg_mixed", 2, np.float64, [4097 * 64 + 3, 700]),
          ("sparse", "pcg_mixed", 32, np.float64, [4097 * 64 + 3])]


@pytest.mark.parametrize("kind,name,nch,dtype,sizes", CASES)
def test_sliced_solves_equal_the_general_kernels(sizes, name, nch, dtype, kind):
    mats = [_spd(n, 100 + n, kind) for n in sizes]
    n = sum(sizes)
    rng = np.random.default_rng(7)
    b = rng.uniform(-1, 1, nch * n).astype(dtype)
    x0 = rng.uniform(-1, 1, nch * n).astype(dtype)
    target = 1e-12 if dtype == np.float64 else 1e-5
    s, x = _run(name, nch, mats, b, x0, 1, dtype, target)
    g, xg = _run(name, nch, mats, b, x0, 0, dtype, target)
    # each solution is within cond * target of the exact one (cond < 20)
    bound = 2 * 20 * target
    assert np.linalg.norm(x - xg) <= bound * np.linalg.norm(xg)
    assert abs(s.getLastIterations() - g.getLastIterations()) <= 1
    # the true residual; in FP32 it drifts from the recursive one by a few roundings
    slack = 1.01 * target + (0 if dtype == np.float64 else 16 * np.finfo(np.float32).eps)
    start = 0
    for m in mats:
        rows = slice(start, start + m.shape[0])
        start += m.shape[0]
        for c in range(nch):
            bc, xc = b[c * n:(c + 1) * n].astype(np.float64)[rows], x[c * n:(c + 1) * n][rows]
            assert np.linalg.norm(bc - m @ xc) <= slack * np.linalg.norm(bc), (m.shape, c)


def test_non_finite_right_hand_side_is_reported():
    from nsfem_amd import cu
    m = _spd(500, 3, "sparse")
    s = cu.createSolver("pcg", 2, m, 50, 1e-10, 1)
    s.setOption("preconditioner", 1)
    b = np.ones(1000)
    b[77] = np.nan
    s.getRhs().upload(b)
    s.getSol().memsetZero()
    s.solve()
    assert not np.isfinite(s.getLastMse(0))


def test_preconditioner_switched_off_again_and_refinement_keep_working():
    """The colour-major rows serve the GS sweeps and the refinement path; the
    locality order only the approximate inverse."""
    from nsfem_amd import cu
    m = _spd(3000, 5, "sparse")
    rng = np.random.default_rng(9)
    b = rng.uniform(-1, 1, 3000)
    ref = spla.spsolve(m.tocsc(), b)
    s = cu.createSolver("pcg_mixed", 1, m, 400, 1e-11, 1)
    for precond, restart in ((0, 0), (1, 0), (0, 0), (1, 0), (1, 1), (1, 0)):
        s.setOption("mixedRestart", 0)
        s.setOption("preconditioner", precond)
        s.setOption("mixedRestart", restart)
        s.getRhs().upload(b)
        s.getSol().memsetZero()
        s.solve()
        x = s.getSol().download()
        assert np.linalg.norm(x - ref) <= 20 * 1e-11 * np.linalg.norm(ref), (precond, restart)


@pytest.mark.parametrize("sizes", [[3000], [700, 64, 1300]])
@pytest.mark.parametrize("name,nch", [("pcg", 2), ("pcg_mixed", 4)])
def test_sweeps_after_a_change_of_preconditioner_equal_a_fresh_solver(sizes, name, nch):
    """The colour sweeps' own shape, kept while the approximate inverse and back
    reallocates the block tables."""
    from nsfem_amd import cu
    mats = [_spd(n, 50 + n, "sparse") for n in sizes]
    b = np.random.default_rng(11).uniform(-1, 1, nch * sum(sizes))
    xs = []
    for switched in (False, True):
        s = cu.createSolver(name, nch, mats[0], 400, 1e-11, 1) if len(mats) == 1 else cu.createBatchSolver(name, nch, mats, 400, 1e-11, 1)
        s.reshapeSweeps(nch if nch > 2 else 4, 256)
        for kind in (1, 0) if switched else ():
            s.setOption("preconditioner", kind)
        s.getRhs().upload(b)
        s.getSol().memsetZero()
        s.solve()
        xs.append(s.getSol().download())
    assert np.array_equal(*xs)


def _with_long_rows(n, length, every, base):
    """base random neighbours a row and `length` of them every `every` rows."""
    rng = np.random.default_rng(n + length)
    r = np.repeat(np.arange(n), base)
    c = (r + rng.integers(1, 60, r.size)) % n
    for i in range(every // 2, n, every):
        far = rng.choice(np.setdiff1d(np.arange(n), [i]), length, replace=False)
        r, c = np.concatenate([r, np.full(length, i)]), np.concatenate([c, far])
    a = sp.coo_matrix((-rng.uniform(0.2, 1, r.size), (r, c)), shape=(n, n)).tocsr()
    a = a + a.T
    a.setdiag(0)
    a.eliminate_zeros()
    return (a + sp.diags(np.asarray(abs(a).sum(axis=1)).ravel() * 1.2 + 1)).tocsr()


# one row of about 200 and of 290 entries, an arrow of 700, many rows of 120 in
# short ones (padding of about 20): all but the first stay on the lane-split
# kernels, from four channels on none does
@pytest.mark.parametrize("args,sliced", [((4000, 190, 4000, 4), True), ((4000, 280, 4000, 4), False), ((701, 700, 701, 0), False),
                                         ((6000, 120, 700, 0), False)])
@pytest.mark.parametrize("name,nch", [("pcg", 1), ("pcg_mixed", 2), ("pcg_mixed", 4)])
@pytest.mark.parametrize("batch", [False, True])
def test_rows_too_uneven_for_slices(args, sliced, name, nch, batch):
    m = _with_long_rows(*args)
    mats = [m, _spd(130, 8, "sparse")] if batch else [m]
    n = sum(a.shape[0] for a in mats)
    rng = np.random.default_rng(13)
    b, x0 = rng.uniform(-1, 1, nch * n), rng.uniform(-1, 1, nch * n)
    s, x = _run(name, nch, mats, b, x0, 1, np.float64, 1e-12)
    assert (s.kindRows()[0] == 0) == (sliced or nch > 2)
    a = sp.block_diag(mats).tocsr()
    for c in range(nch):
        bc, xc = b[c * n:(c + 1) * n], x[c * n:(c + 1) * n]
        assert np.linalg.norm(bc - a @ xc) <= 1.01e-12 * np.linalg.norm(bc) * np.sqrt(len(mats))
    s.solve()  # from the solution: nothing left to do
    assert np.linalg.norm(s.getSol().download() - x) <= 1e-11 * np.linalg.norm(x)
