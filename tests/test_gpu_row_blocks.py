"""Kernels on general short-row patterns against the oracle, bit for bit: the
CSR product and Jacobi sweeps on blocks of rows and with 1, 2 and 4 rows a
thread (empty, short and long rows, a row longer than a block's entry capacity,
sizes around a block and the chip's block count), and ParILU sweeps whose positions have none, up to four and more
matches, taken from memory one after another or staged in LDS, in every factor
storage and both step modes."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _pattern(orc, n, offs, keep, seed, long_row=False):
    """Symmetric pattern with a share `keep` of the entries at distances offs;
    long_row: one row (and column) holds most of them."""
    rng = np.random.default_rng(seed)
    rows, cols = [np.arange(n)], [np.arange(n)]
    for d in offs:
        i = np.arange(d, n)
        i = i[rng.random(len(i)) < keep]
        rows += [i, i - d]
        cols += [i - d, i]
    if long_row:
        i = np.arange(2, n, 2)
        rows += [i, np.zeros_like(i)]
        cols += [np.zeros_like(i), i]
    key = np.unique(np.concatenate(rows).astype(np.int64) * n + np.concatenate(cols))
    rows, cols = key // n, key % n
    vals = rng.uniform(-1.2, -0.8, len(rows))
    deg = np.bincount(rows, minlength=n)
    vals[rows == cols] = 1.5 * deg
    return orc._coo_to_csr(n, rows, cols, vals)


WIDE = [1, 2, 3, 30, 31, 32, 33]
CASES = [("tiny", 1, [], 1.0, False), ("pair", 2, [1], 1.0, False), ("block", 256, WIDE[:4], 0.6, False),
         ("over", 257, WIDE[:4], 0.6, False), ("ragged", 5003, WIDE, 0.4, False), ("full", 3001, WIDE, 1.0, False),
         # FP64: matches staged in LDS, for their number and for the positions'
         ("wide", 20001, WIDE, 1.0, False), ("rounds", 350001, [1, 2, 3], 1.0, False),
         ("long", 9001, [1, 40, 41], 0.7, True), ("many", 300001, [1, 500, 501, 502], 0.5, False)]


# the kernels of a CSR form, and the default choice among them
KERNELS = [(b"row_blocks", 2, 1), (b"row_blocks", 0, 1), (b"stream_rows_per_thread", 1, 0),
           (b"stream_rows_per_thread", 2, 0), (b"stream_rows_per_thread", 4, 0), (b"row_blocks", 1, 1)]


def _each_kernel(gpu, call):
    for name, value, default in KERNELS:
        gpu.check(gpu.lib().lace_set_option(name, value))
        try:
            yield (name, value), call()
        finally:
            gpu.check(gpu.lib().lace_set_option(name, default))


def test_row_options(lace):
    """Every choice can be taken back to the default; others are refused."""
    lib = lace.lib()
    for name, ok, bad in ((b"row_blocks", (0, 2, 1), (-1, 3)), (b"stream_rows_per_thread", (1, 2, 4, 0), (-1, 3, 5))):
        assert all(lib.lace_set_option(name, v) == 0 for v in ok)
        assert all(lib.lace_set_option(name, v) != 0 for v in bad)


@pytest.mark.parametrize("prec", ["F64", "F32"])
@pytest.mark.parametrize("name,n,offs,keep,long_row", CASES)
def test_row_blocks(gpu, orc, name, n, offs, keep, long_row, prec):
    A = _pattern(orc, n, offs, keep, 3, long_row)
    print(f"row blocks: {name} {prec} n={n} nnz={A.nnz}", flush=True)
    dt = np.float64 if prec == "F64" else np.float32
    H = gpu.HostCSR.from_csr(A)
    rng = np.random.default_rng(4)
    x = rng.standard_normal(n).astype(dt)
    if A.nnz <= 16 * n:
        M = gpu.DevCSRMatrix(H, getattr(gpu, "LACE_" + prec))
        # each row summed in column order from zero, in the values' precision
        ri = A.rowidx()
        prod = (A.val.astype(dt) * x[A.col]).astype(dt)
        want = np.zeros(n, dt)
        at = A.row[:-1].astype(np.int64)
        for q in range(int(np.diff(A.row).max())):
            has = at + q < A.row[1:]
            want[has] = want[has] + prod[(at + q)[has]]
        assert len(ri) == A.nnz
        for kernel, y in _each_kernel(gpu, lambda: M.spmv(x)):
            assert np.array_equal(y, want), kernel
    P = gpu.ParILU(H, getattr(gpu, "LACE_" + prec))
    P.sweeps(3)
    st = orc.parilu(A, 3, dtype=dt)
    (_, _, lv), (_, _, uv) = P.factors()
    assert np.array_equal(lv, st.Lval.astype(lv.dtype)) and np.array_equal(uv, st.Uval.astype(uv.dtype))
    Lf = orc.CSR(n, n, st.L.row, st.L.col, st.Lval)
    Uc = orc.CSR(n, n, st.U.row, st.U.col, st.Uval)
    Ur, Lt = orc.transpose(Uc), orc.transpose(Lf)

    def jacobi(T, r, upper, k):
        """k sweeps from zero, rows summed in column order over the
        off-diagonal entries, then divided."""
        kd = T.row[:-1] if upper else T.row[1:] - 1
        first = (T.row[:-1] + 1 if upper else T.row[:-1]).astype(np.int64)
        last = (T.row[1:] if upper else T.row[1:] - 1).astype(np.int64)
        d, y = T.val[kd].astype(dt), np.zeros(n, dt)
        for s in range(k):
            acc = np.zeros(n, dt)
            if s:
                prod = (T.val.astype(dt) * y[T.col]).astype(dt)
                for q in range(int((last - first).max())):
                    has = first + q < last
                    acc[has] = acc[has] + prod[(first + q)[has]]
            y = ((r - acc) / d).astype(dt)
        return y

    for k in (2, 5):
        want = jacobi(Ur, jacobi(Lf, x, False, k), True, k)
        for kernel, got in _each_kernel(gpu, lambda: P.apply(x, gpu.TRSV_JACOBI, k)):
            assert np.array_equal(got, want), (kernel, k)
        want = jacobi(Lt, jacobi(Uc, x, False, k), True, k)
        for kernel, got in _each_kernel(gpu, lambda: P.apply(x, gpu.TRSV_JACOBI, k, trans=1)):
            assert np.array_equal(got, want), (kernel, k)


@pytest.mark.parametrize("prec", ["F64", "F32", "BF16", "F16"])
@pytest.mark.parametrize("name", ["block", "over", "ragged", "full", "wide", "long"])
def test_parilu_sweeps_with_matches(gpu, orc, name, prec):
    """Every sweep's factors, bit for bit, in every storage (the 16-bit ones
    round inside the sweep) and with and without the step, which sums up to
    3 10^5 squares in FP64 in another order (at most that many roundings)."""
    _, n, offs, keep, long_row = next(c for c in CASES if c[0] == name)
    A = _pattern(orc, n, offs, keep, 5, long_row)
    storage = prec.lower() if prec in ("BF16", "F16") else None
    dt = np.float64 if prec == "F64" else np.float32
    print(f"sweeps with matches: {name} {prec} n={n} nnz={A.nnz}", flush=True)
    P = gpu.ParILU(gpu.HostCSR.from_csr(A), getattr(gpu, "LACE_" + prec))
    st = orc.ParILUState(A, dtype=dt, storage=storage)
    anorm = np.linalg.norm(A.val)
    for k in range(4):
        got = P.sweeps(1, want_step=k % 2 == 0)
        step = st.sweep("jacobi") / anorm
        (_, _, lv), (_, _, uv) = P.factors()
        assert np.array_equal(lv.astype(dt), st.Lval), (k, "L")
        assert np.array_equal(uv.astype(dt), st.Uval), (k, "U")
        if k % 2 == 0:
            assert abs(got - step) <= 3e5 * 2.3e-16 * step, (k, got, step)
