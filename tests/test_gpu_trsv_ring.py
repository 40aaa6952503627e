"""Exact triangular solves by one workgroup in level order (option
"trsv_exact_ring"): bit-identical to the persistent kernel, which the other
tests tie to substitution.  Levels of one row, of a chunk (64 rows) less and
more one, wider than a round of the waves; chains as long as the matrix; rows
of 0 to 16 off-diagonal entries; operands as far back as the ring in LDS
holds and one farther, and rows of 17 entries (which both keep the
persistent kernel); infinities and NaN; transposed solves, on patterns that
are symmetric and not (then L, U and their transposes have level orders of their
own); factor values that change; handles made by default, which hold the form
where it is expected to pay, and with the option at 2, which always do."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _opt(gpu, value):
    gpu.check(gpu.lib().lace_set_option(b"trsv_exact_ring", value))


@pytest.fixture
def ring(gpu):
    yield lambda v: _opt(gpu, v)
    _opt(gpu, 1)


def _band(orc, n, offs, seed=0, keep=1.0):
    """Symmetric pattern with entries at distances `offs` (a share of them)."""
    rng = np.random.default_rng(seed)
    rows, cols = [np.arange(n)], [np.arange(n)]
    for d in offs:
        i = np.arange(d, n)
        i = i[rng.random(len(i)) < keep]
        rows += [i, i - d]
        cols += [i - d, i]
    rows, cols = np.concatenate(rows), np.concatenate(cols)
    vals = np.where(rows == cols, 2.0 * len(offs) + 1.0, -1.0) * rng.uniform(0.75, 1.25, len(rows))
    return orc._coo_to_csr(n, rows, cols, vals)


def _nonsym(orc, A, seed=1):
    """A without a fifth of its entries above the diagonal."""
    ri = A.rowidx()
    keep = (ri >= A.col) | (np.random.default_rng(seed).random(A.nnz) < 0.8)
    return orc._coo_to_csr(A.n_rows, ri[keep], A.col[keep], A.val[keep])


CASES = {
    "one": lambda o: _band(o, 1, []),
    "diagonal": lambda o: _band(o, 5000, []),
    "chain": lambda o: _band(o, 3000, [1]),
    "level63": lambda o: _band(o, 1000, [63]),
    "level64": lambda o: _band(o, 1024, [64]),
    "level65": lambda o: _band(o, 1001, [65]),
    "level1500": lambda o: _band(o, 9000, [1500, 1501]),
    "lap2d": lambda o: o.laplace2d(67, 45),
    "conv3d": lambda o: o.convdiff3d(21, 18, 19),
    "rows16": lambda o: _band(o, 6000, [1, 2, 3, 60, 61, 62, 63, 64, 700, 701, 702, 703, 704, 705, 706, 707]),
    "ragged": lambda o: _band(o, 20000, [1, 38, 39, 40, 41, 1480, 1520, 1560, 1561], keep=0.5),
    "rows17": lambda o: _band(o, 3000, [1, 2, 3, 60, 61, 62, 63, 64, 700, 701, 702, 703, 704, 705, 706, 707, 708]),
    # rows of few entries, needed long after they are solved
    "late": lambda o: _band(o, 40000, [1, 130, 131, 132, 4000, 4090], keep=0.35),
    "nonsym": lambda o: _nonsym(o, o.convdiff3d(14, 13, 15)),
    "nonsym_ragged": lambda o: _nonsym(o, _band(o, 12000, [1, 38, 39, 40, 41, 1480, 1520, 1560, 1561], keep=0.5)),
    # two levels of h rows: an operand lies up to 2 h rows back from its level's end
    "span_f64": lambda o: _band(o, 16384, [8192]),
    "span_f64_over": lambda o: _band(o, 16386, [8193]),
    "span_f32": lambda o: _band(o, 32768, [16384]),
    "span_f32_over": lambda o: _band(o, 32770, [16385]),
}


@pytest.mark.parametrize("prec", ["F64", "F32"])
@pytest.mark.parametrize("name", list(CASES))
def test_ring_matches_persistent(gpu, orc, ring, name, prec):
    A = CASES[name](orc)
    print(f"ring: {name} {prec} n={A.n_rows}", flush=True)
    H, lp = gpu.HostCSR.from_csr(A), getattr(gpu, "LACE_" + prec)
    Q = gpu.ParILU(H, lp)
    ring(2)
    P = gpu.ParILU(H, lp)
    n = A.n_rows
    rng = np.random.default_rng(5)
    for sweeps in (2, 1):  # the factor values change in between
        P.sweeps(sweeps)
        Q.sweeps(sweeps)
        r = rng.standard_normal(n)
        for special in (False, True):
            if special:
                r[n // 2], r[n // 3], r[n // 5] = np.inf, np.nan, -0.0
            for trans in (0, 1):
                out = []
                for v in (0, 1, 2):  # 2: wherever the form exists
                    ring(v)
                    out.append(P.apply(r, gpu.TRSV_LEVEL, 0, trans))
                assert np.array_equal(out[0], out[1], equal_nan=True), (sweeps, special, trans)
                assert np.array_equal(out[0], out[2], equal_nan=True), (sweeps, special, trans)
                for v in (2, 1):
                    ring(v)
                    assert np.array_equal(out[0], Q.apply(r, gpu.TRSV_LEVEL, 0, trans), equal_nan=True), (v, trans)
