"""32-column Jacobi sweeps, several to a launch plane by plane (option
"jacobi_march" 2: wherever there is such a form): bit-identical to one sweep
per launch ("jacobi_pair" 0) and to the single-vector solve.  Grids narrower than the sweeps' reach, of one and several
tiles along each axis, of one and several runs of planes with a short last one;
one launch and several; both factors and directions; infinities and NaN; a
pattern with gaps, which keeps the other kernels."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

GRIDS = [(2, 2, 2), (4, 3, 5), (9, 3, 17), (30, 30, 9), (31, 33, 8), (61, 18, 40), (17, 70, 25), (200, 5, 19), (3, 3, 100)]


def _opt(gpu, name, value):
    gpu.check(gpu.lib().lace_set_option(name, value))


def _both(gpu, P, R, sweeps, trans):
    out = []
    for march, pair in ((2, 1), (1, 0)):
        _opt(gpu, b"jacobi_march", march)
        _opt(gpu, b"jacobi_pair", pair)
        try:
            out.append(P.apply_block(R, gpu.TRSV_JACOBI, sweeps=sweeps, trans=trans))
        finally:
            _opt(gpu, b"jacobi_march", 1)
            _opt(gpu, b"jacobi_pair", 1)
    return out


def _launches(gpu, P, R, sweeps):
    """Launches of L's sweeps by kind: plane by plane, pairs, single ones."""
    lib = gpu.lib()
    gpu.check(lib.lace_timing_enable(1))
    gpu.check(lib.lace_timing_reset())
    try:
        P.apply_block(R, gpu.TRSV_JACOBI, sweeps=sweeps)
        out = []
        for kind in (b"march", b"pair", b"sweep"):
            calls = C.c_long(0)
            lib.lace_timing_get_calls(b"block_jacobi_" + kind + b"_lower", C.byref(calls))
            out.append(calls.value)
    finally:
        gpu.check(lib.lace_timing_enable(0))
    return tuple(out)


@pytest.mark.parametrize("dims,sweeps,want", [
    # few workgroups: the pair kernels
    ((2, 2, 2), 5, (0, 0, 4)),  # (no diagonal form)
    ((16, 16, 16), 5, (0, 2, 0)), ((16, 16, 16), 4, (0, 1, 1)), ((10, 10, 40), 3, (0, 1, 0)),
    ((5, 5, 4000), 5, (0, 2, 0)), ((64, 64, 16), 5, (0, 2, 0)), ((56, 56, 56), 5, (0, 2, 0)),
    # a single coupled sweep has nothing to save
    ((72, 72, 72), 2, (0, 0, 1)),
    # the chip is full
    ((200, 200, 4), 5, (1, 0, 0)), ((200, 200, 4), 6, (2, 0, 0)), ((72, 72, 72), 5, (1, 0, 0)), ((72, 72, 72), 3, (1, 0, 0)),
    ((72, 72, 72), 6, (2, 0, 0))])
def test_march_only_where_it_pays(gpu, orc, dims, sweeps, want):
    A = orc.convdiff3d(*dims)
    P = gpu.ParILU(gpu.HostCSR.from_csr(A), gpu.LACE_F32)
    P.sweeps(2)
    R = np.random.default_rng(1).standard_normal((A.n_rows, 32)).astype(np.float32)
    assert _launches(gpu, P, R, sweeps) == want


@pytest.mark.parametrize("dims", GRIDS)
def test_march_matches_single_sweeps(gpu, orc, dims):
    A = orc.convdiff3d(*dims)
    rng = np.random.default_rng(7)
    A = orc.CSR(A.n_rows, A.n_cols, A.row, A.col, A.val * rng.uniform(0.75, 1.25, A.nnz))
    print(f"march: {dims}", flush=True)
    P = gpu.ParILU(gpu.HostCSR.from_csr(A), gpu.LACE_F32)
    P.sweeps(3)
    R = rng.standard_normal((A.n_rows, 32)).astype(np.float32)
    for trans in (0, 1):
        for k in (1, 2, 3, 4, 5, 6, 9, 10):
            a, b = _both(gpu, P, R, k, trans)
            assert np.array_equal(a, b), (trans, k)
        z = P.apply(R[:, 13].copy(), gpu.TRSV_JACOBI, sweeps=5, trans=trans)
        assert np.array_equal(_both(gpu, P, R, 5, trans)[0][:, 13], z)


def test_march_special_values_and_gaps(gpu, orc):
    A = orc.convdiff3d(24, 19, 21)
    rng = np.random.default_rng(3)
    ri = A.rowidx()
    keep = (ri == A.col) | (rng.random(A.nnz) >= 0.1)
    row = np.zeros(A.n_rows + 1, dtype=np.int32)
    np.add.at(row, ri[keep] + 1, 1)
    gaps = orc.CSR(A.n_rows, A.n_cols, np.cumsum(row).astype(np.int32), A.col[keep].copy(), A.val[keep].copy())
    R = rng.standard_normal((A.n_rows, 32)).astype(np.float32)
    R[5, 3], R[4000, 17], R[9000, 31], R[70, 0] = np.inf, np.nan, -np.inf, -0.0
    for M in (A, gaps):
        P = gpu.ParILU(gpu.HostCSR.from_csr(M), gpu.LACE_F32)
        P.sweeps(3)
        for trans in (0, 1):
            a, b = _both(gpu, P, R, 5, trans)
            assert np.array_equal(a, b, equal_nan=True), trans


def test_march_quotients(gpu, orc):
    """Right-hand sides from the subnormal range to the largest: the sweeps'
    quotients round as IEEE division does, which the one-sweep launches use."""
    A = orc.convdiff3d(16, 8, 12)
    rng = np.random.default_rng(9)
    P = gpu.ParILU(gpu.HostCSR.from_csr(A), gpu.LACE_F32)
    P.sweeps(3)
    R = rng.standard_normal((A.n_rows, 32)) * 2.0 ** rng.integers(-150, 120, (A.n_rows, 32))
    R = R.astype(np.float32)
    for k in (2, 5):
        a, b = _both(gpu, P, R, k, 0)
        assert np.array_equal(a, b, equal_nan=True), k
        z = P.apply(R[:, 4].copy(), gpu.TRSV_JACOBI, sweeps=k)
        assert np.array_equal(a[:, 4], z, equal_nan=True), k


def test_march_zeros(gpu, orc):
    """Zeros of either sign, alone and beside quotients below the normal range:
    the same bits as one sweep per launch."""
    A = orc.convdiff3d(16, 8, 12)
    rng = np.random.default_rng(11)
    P = gpu.ParILU(gpu.HostCSR.from_csr(A), gpu.LACE_F32)
    P.sweeps(3)
    R = rng.standard_normal((A.n_rows, 32)).astype(np.float32)
    R[rng.random(R.shape) < 0.6] = 0.0
    R[rng.random(R.shape) < 0.2] = -0.0
    R[: A.n_rows // 2] = -0.0
    R[rng.random(R.shape) < 0.05] = np.float32(3e-39)
    for k in (2, 3, 5):
        for trans in (0, 1):
            a, b = _both(gpu, P, R, k, trans)
            assert np.array_equal(a.view(np.uint32), b.view(np.uint32)), (k, trans)
