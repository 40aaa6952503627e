"""Several Jacobi sweeps per launch on boxes of the grid (option
"jacobi_tile" 2: wherever there is such a form): bit-identical to one-sweep
launches of a row per thread ("jacobi_dia_vec" 0), which the other tests tie
to the oracle.  Grids whose sides fall short of, meet and pass the boxes'
(16 x 8 x 8, 12 x 12 x 12, 64 x 24, ...), lines that do and do not keep the
16-byte word, every factor storage, transposed solves, one launch and
several, a pattern with gaps (which keeps the one-sweep kernels), vectors off
the 16-byte boundary."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

GRIDS = [(16, 8, 8), (20, 9, 17), (17, 25, 13), (13, 12, 24), (4, 3, 2), (2, 2, 2), (64, 24, 1), (68, 49, 1), (29, 57, 1),
         (33, 4, 1)]
PRECS = ["F64", "F32", "BF16", "F16"]


def _matrix(orc, dims):
    return orc.convdiff3d(*dims) if dims[2] > 1 else orc.laplace2d(*dims[:2])


def _option(gpu, value):
    gpu.check(gpu.lib().lace_set_option(b"jacobi_dia_vec", value))


@pytest.fixture
def tile(gpu):
    gpu.check(gpu.lib().lace_set_option(b"jacobi_tile", 2))
    yield lambda v: _option(gpu, v)
    _option(gpu, 1)
    gpu.check(gpu.lib().lace_set_option(b"jacobi_tile", 1))


@pytest.mark.parametrize("prec", PRECS)
@pytest.mark.parametrize("dims", GRIDS)
def test_tiles_match_single_sweeps(gpu, orc, tile, dims, prec):
    A = _matrix(orc, dims)
    rng = np.random.default_rng(7)
    # values off the stencil's few constants
    A = orc.CSR(A.n_rows, A.n_cols, A.row, A.col, A.val * rng.uniform(0.75, 1.25, A.nnz))
    P = gpu.ParILU(gpu.HostCSR.from_csr(A), getattr(gpu, "LACE_" + prec))
    P.sweeps(3)
    r = rng.standard_normal(A.n_rows)
    for trans in (0, 1):
        for k in (1, 2, 3, 5, 6, 9, 10):
            out = []
            for v in (0, 1):
                tile(v)
                out.append(P.apply(r, gpu.TRSV_JACOBI, k, trans))
            assert np.array_equal(out[0], out[1]), (trans, k)


@pytest.mark.parametrize("prec", ["F64", "F32"])
def test_gaps_and_unaligned_vectors(gpu, orc, tile, prec):
    A = orc.convdiff3d(16, 12, 10)
    rng = np.random.default_rng(3)
    dt = np.float64 if prec == "F64" else np.float32
    ri = A.rowidx()
    keep = (ri == A.col) | (rng.random(A.nnz) >= 0.1)
    row = np.zeros(A.n_rows + 1, dtype=np.int32)
    np.add.at(row, ri[keep] + 1, 1)
    gaps = orc.CSR(A.n_rows, A.n_cols, np.cumsum(row).astype(np.int32), A.col[keep].copy(), A.val[keep].copy())
    for M in (A, gaps):
        P = gpu.ParILU(gpu.HostCSR.from_csr(M), getattr(gpu, "LACE_" + prec))
        P.sweeps(3)
        n, es = M.n_rows, np.dtype(dt).itemsize
        r = rng.standard_normal(n).astype(dt)
        # an infinity and a NaN travel as they do with one sweep per launch
        r[n // 2], r[n // 3] = np.inf, np.nan
        tile(0)
        want = P.apply(r, gpu.TRSV_JACOBI, 5)
        tile(1)
        assert np.array_equal(P.apply(r, gpu.TRSV_JACOBI, 5), want, equal_nan=True)
        dr, dz = gpu.DevVec(n + 1, dt, np.concatenate([[dt(0)], r])), gpu.DevVec(n + 1, dt, np.zeros(n + 1, dt))
        off = lambda d: C.c_void_p(d.ptr.value + es)  # noqa: E731
        gpu.check(gpu.lib().lace_parilu_apply(P.h, gpu.TRSV_JACOBI, 5, 0, off(dr), off(dz)))
        assert np.array_equal(dz.download()[1:], want, equal_nan=True)


@pytest.mark.parametrize("prec", PRECS)
@pytest.mark.parametrize("dims,least", [
    # sweeps from which boxes are taken, by (F64, F32, 16 bits)
    ((20, 9, 17), (2, 2, 2)), ((64, 24, 1), (2, 2, 2)), ((29, 57, 1), (2, 2, 2)),
    ((17, 25, 13), (2, 2, 2)), ((63, 64, 65), (2, 2, 2)), ((66, 64, 63), (2, 3, 3)), ((64, 66, 63), (2, 2, 2)),
    ((101, 102, 103), (2, 3, 4))])
def test_tiles_only_where_they_pay(gpu, orc, dims, least, prec):
    """The launches of L's sweeps: one for up to five sweeps on boxes, else one
    a sweep after the first; the results are those of one-sweep launches."""
    A = _matrix(orc, dims)
    P = gpu.ParILU(gpu.HostCSR.from_csr(A), getattr(gpu, "LACE_" + prec))
    P.sweeps(2)
    lib, r = gpu.lib(), np.random.default_rng(2).standard_normal(A.n_rows)
    for k in (2, 3, 4, 5):
        gpu.check(lib.lace_timing_enable(1))
        gpu.check(lib.lace_timing_reset())
        try:
            z = P.apply(r, gpu.TRSV_JACOBI, k)
            calls = gpu.timing_calls("trsv_jacobi_sweep_lower")
        finally:
            gpu.check(lib.lace_timing_enable(0))
        assert calls == (1 if k >= least[min(PRECS.index(prec), 2)] else k - 1), k
        _option(gpu, 0)
        try:
            assert np.array_equal(P.apply(r, gpu.TRSV_JACOBI, k), z), k
        finally:
            _option(gpu, 1)
