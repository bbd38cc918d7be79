"""The V-cycle's dense coarsest level inverted on the GPU, and the finest
level's sweeps fused with the residual and r.z: sizes at the edges of the
tiles (32 rows of the inversion, 64 of the product, 16 of the matrix-core
product) and of the hierarchy (one level, two levels), every channel count."""

import numpy as np
import pytest
import scipy.sparse as sp
import scipy.sparse.linalg as spla

pytestmark = pytest.mark.gpu


def _grid(nx, ny):
    """Five-point Laplacian with Dirichlet ends, mildly anisotropic (SPD)."""
    t = lambda n: sp.diags([-np.ones(n - 1), 2 * np.ones(n), -np.ones(n - 1)], [-1, 0, 1])
    return (sp.kron(sp.eye(ny), t(nx)) + 0.7 * sp.kron(t(ny), sp.eye(nx))).tocsr()


# up to 512 rows: one dense level; above: the finest level and a dense one (of
# 1,624 rows at the last shape, too many on four columns in FP64)
@pytest.mark.parametrize("shape", [(1, 1), (7, 9), (16, 32), (19, 27), (50, 61), (97, 101), (110, 115)])
@pytest.mark.parametrize("name,nch", [("amg_pcg", 1), ("amg_pcg_mixed", 1), ("amg_pcg", 2), ("amg_pcg_mixed", 4), ("amg_pcg", 4), ("amg_pcg", 8),
                                      ("amg_pcg_mixed", 8), ("amg_pcg", 16), ("amg_pcg_mixed", 16)])
def test_solutions_match_the_direct_solve(shape, name, nch):
    from nsfem_amd import cu
    m = _grid(*shape)
    n = m.shape[0]
    rng = np.random.default_rng(5)
    # columns of different scale; a guess has its column's, because the residual
    # recurrence rounds at eps times the first residual (1 against a right-hand
    # side of 1e-6 leaves 1e-10, above the target)
    scale = np.where(np.arange(nch) % 3 == 1, 1e-6, 1.0)[:, None]
    b = rng.uniform(-1, 1, (nch, n)) * scale
    target = 1e-11
    s = cu.createSolver(name, nch, m, 200, target, 1)
    ref = spla.splu(m.tocsc()).solve(b.T).T
    for guess in (0.0, 1.0):
        s.getRhs().upload(b.ravel())
        s.getSol().upload((guess * scale * np.ones((nch, n))).ravel())
        s.solve()
        x = s.getSol().download().reshape(nch, n)
        for c in range(nch):
            assert np.linalg.norm(b[c] - m @ x[c]) <= 1.01 * target * np.linalg.norm(b[c]), c
            # the residual bound times a condition number below 2 (n + 1)^2 per direction
            assert np.linalg.norm(x[c] - ref[c]) <= target * 8 * max(shape) ** 2 * np.linalg.norm(ref[c]) + 1e-14 * np.linalg.norm(ref[c]), c
        assert s.getLastIterations() <= 30
    first = s.getSol().download()
    s.getSol().upload((scale * np.ones((nch, n))).ravel())
    s.solve()
    assert np.array_equal(first, s.getSol().download())


@pytest.mark.parametrize("name", ["amg_pcg", "amg_pcg_mixed"])
def test_indefinite_operators_are_still_rejected(name):
    from nsfem_amd import cu
    from nsfem_amd._lib import NsfemError
    m = _grid(40, 41)
    m = (m - 0.5 * sp.diags(m.diagonal())).tocsr()  # the smooth modes' eigenvalues are negative
    with pytest.raises(NsfemError, match="not positive definite"):
        cu.createSolver(name, 1, m, 100, 1e-10, 1)
