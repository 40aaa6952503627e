"""Householder FGMRES against the oracle where its vectors' slabs end: one
slab (1024 rows) less and more a row, several, odd sizes, a slab count past
the one up to which a single workgroup sums the partials, and cycles of up to
63 columns (every remainder of the column groups is passed through).

One solve without preconditioner to a loose tolerance: the same Krylov space,
so the same number of steps, and solutions whose difference is rounding (1e-16
times the steps and the conditioning of the space, well under the 1e-6
checked); the residual norms agree to the same."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims,m", [((3, 3), 9), ((31, 33), 63), ((32, 32), 63), ((25, 41), 63), ((43, 47), 40),
                                    ((64, 64), 50), ((101, 83), 33), ((640, 830), 20)])
def test_householder_slabs(gpu, orc, dims, m):
    A = orc.laplace2d(*dims)
    n = A.n_rows
    ri = np.repeat(np.arange(n), np.diff(A.row))
    # diagonally dominant and not symmetric, so that m columns suffice
    val = A.val * np.random.default_rng(1).uniform(0.8, 1.2, A.nnz) + np.where(ri == A.col, 0.8, 0.0)
    A = orc.CSR(n, n, A.row, A.col, val)
    b = np.random.default_rng(2).standard_normal(n)
    o = gpu.default_opts()
    o.search_max, o.restart_max, o.rtol, o.trsv, o.inner_iters = m, 1, 1e-8, gpu.TRSV_NONE, 0
    S = gpu.Solver(gpu.HostCSR.from_csr(A), o)
    S.setup()
    x, st = S.solve(b)
    ref = orc.fgmres_householder(A, b, m=m, restart_max=1, rtol=1e-8, tol_type=1, choice=2)
    assert abs(st.iterations - ref.searches) <= 1, (st.iterations, ref.searches)
    if st.iterations == ref.searches:
        assert np.linalg.norm(x - ref.x) <= 1e-6 * np.linalg.norm(ref.x)
    r = np.linalg.norm(b - A.scipy() @ x)
    rr = np.linalg.norm(b - A.scipy() @ ref.x)
    assert r <= 1.05 * max(rr, 1e-8 * np.linalg.norm(b))
