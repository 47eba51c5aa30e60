"""Tile layout of large operators (at least 2^22 nonzeros per direction: the
built-in choice, and what the layout with every panel in one launch runs):
row sums accumulated in LDS, batches of entries with distinct rows.  Against
the float64 host product at the sizes where its units change: few rows in
many segments, tiles of the largest height, several rounds of tiles, odd
sizes, empty rows; rows that do not fit it (long or uneven) fall back to the
panels.  Tolerance: a row of len products summed one after another in FP64
is off by at most len * 2^-53 * sum |a x| (plus the products' own rounding),
and FP32 results by 2^-24 of the value on top."""
import ctypes as C

import numpy as np
import pytest

from propack_amd import api, synth

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def _matrix(m, n, lam, seed, dtype=np.float64, extra=()):
    """Poisson(lam) distinct uniform columns per row; extra: (row, column)
    arrays added."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    deg = torch.poisson(torch.full((m,), float(lam), device="cuda"), generator=g).long()
    deg = deg.clamp_(max=n)
    rows = torch.repeat_interleave(torch.arange(m, device="cuda"), deg)
    cols = torch.randint(0, n, (rows.numel(),), generator=g, device="cuda")
    key = rows * n + cols
    for r, c in extra:
        key = torch.cat([key, torch.as_tensor(r * n + c, device="cuda")])
    key = torch.unique(key)
    rows, cols = key // n, key % n
    rp = torch.zeros(m + 1, dtype=torch.int64, device="cuda")
    torch.cumsum(torch.bincount(rows, minlength=m), 0, out=rp[1:])
    vals = torch.randn(key.numel(), dtype=torch.float64, generator=g, device="cuda")
    A = synth.Csr(m, n, rp.int().cpu().numpy(), cols.int().cpu().numpy(),
                  vals.cpu().numpy().astype(dtype))
    return A, rows.cpu().numpy(), cols.cpu().numpy()


def _products(A, rows, cols, x, trans):
    """Row sums of op(A) x and of |op(A)| |x| in float64, and the lengths."""
    i, j, L = (rows, cols, A.m) if trans == "n" else (cols, rows, A.n)
    p = A.val.astype(np.float64) * x.astype(np.float64)[j]
    return (np.bincount(i, p, L), np.bincount(i, np.abs(p), L), np.bincount(i, minlength=L))


def _check(A, rows, cols, op, seed):
    rng = np.random.default_rng(seed)
    out = {}
    for trans, nin in (("n", A.n), ("t", A.m)):
        x = rng.standard_normal(nin).astype(A.val.dtype)
        want, mag, ln = _products(A, rows, cols, x, trans)
        tol = (ln + 1) * 2.0 ** -52 * mag
        if A.val.dtype == np.float32:
            tol = tol + 2.0 ** -24 * np.abs(want) + 2.0 ** -149
        got = op.spmv(x, trans)
        assert np.all(np.abs(got.astype(np.float64) - want) <= tol), (A.m, A.n, trans)
        assert np.array_equal(got, op.spmv(x, trans))
        dx = torch.from_numpy(x).cuda()
        dy = torch.full((want.size,), float("nan"), dtype=dx.dtype, device="cuda")
        rc = api.lib().pk_csr_spmv_noalloc(op.handle, C.c_char(trans.encode()),
                                           C.c_void_p(dx.data_ptr()), C.c_void_p(dy.data_ptr()),
                                           C.c_int(op.prec), C.c_void_p(0))
        assert rc == 0, api.lib().pk_last_error()
        torch.cuda.synchronize()
        assert np.array_equal(dy.cpu().numpy(), got)
        out[trans] = (x, got)
    return out


@pytest.mark.parametrize("m,n,lam", [
    (40009, 30011, 110.0),     # 16 segments of low tiles: many conflicts in a batch
    (300007, 260011, 16.0),    # odd sizes both ways
    (1000000, 320000, 5.0),    # five segments of tiles near the largest height
    (1020001, 1017003, 4.3),   # four segments; sparse columns
    (5130001, 900000, 0.9),    # past 256 full tiles: two rounds, many empty rows
])
@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_tile_products(m, n, lam, dtype):
    A, rows, cols = _matrix(m, n, lam, seed=m + n, dtype=dtype)
    assert A.nnz >= 1 << 22
    op = api.CsrOperator(A, api.PK_F64 if dtype == np.float64 else api.PK_F32)
    assert op.sort() == (0, 0) and op.lanes() == (0, 0)
    res = _check(A, rows, cols, op, 1)
    # the row-block layout, asked for, sums in another order
    op.set_sort(0, 0)
    differ = 0
    for trans, (x, got) in res.items():
        y = op.spmv(x, trans)
        _, mag, ln = _products(A, rows, cols, x, trans)
        differ += int((y != got).sum())
        eps = 2.0 ** -51 if dtype == np.float64 else 2.0 ** -23
        assert np.all(np.abs(y.astype(np.float64) - got) <= (ln + 2) * eps * mag)
    # FP32 results round both orders' FP64 sums to the same values nearly always
    assert differ > 0 or dtype == np.float32


def test_tile_stands_in_for_concurrent_panels():
    """Every panel in one launch, at a size the tile layout serves: the same
    products as the built-in choice bit for bit, the settings reported as
    asked, a solve against the row-block layout's to 1e-12 with its operator
    count, an engine made before the switch, and a batch on such operators
    (which runs the sorted panels) to rounding."""
    A, rows, cols = _matrix(320000, 280000, 15.0, seed=3)
    op = api.CsrOperator(A, panels=(4, 8), lanes=(0, -1), sort=(-8192, -8192))
    assert op.panels() == (4, 8) and op.sort() == (-8192, -8192) and op.lanes() == (0, -1)
    res = _check(A, rows, cols, op, 2)
    plain = api.CsrOperator(A)
    for trans, (x, got) in res.items():
        assert np.array_equal(plain.spmv(x, trans), got)
    u0 = synth.start_vector(A.m, 7)

    def solve(o, eng=None):
        eng = eng or api.Engine(o, kmax=48)
        eng.put_u1(u0)
        return api.lansvd_irl_dev(eng, 8, 48, tol=1e-8)
    a = solve(op)
    ref = api.CsrOperator(A, panels=(2, 2))
    early = api.Engine(ref, kmax=48)
    b = solve(ref)
    assert a.k == b.k == 8 and a.info == b.info == 0
    np.testing.assert_allclose(a.sigma, b.sigma, rtol=1e-12)
    assert a.counters["nopx"] == b.counters["nopx"]
    ref.set_sort(-8192, -8192)
    c = solve(ref, early)
    np.testing.assert_allclose(c.sigma, b.sigma, rtol=1e-12)
    engs = [api.Engine(op, kmax=48), api.Engine(plain, kmax=48)]
    for e in engs:
        e.put_u1(u0)
    bat = api.Batch(engs)
    for r in api.lansvd_irl_batch(bat, 8, 48, tol=1e-8):
        assert r.info == 0 and r.k == 8
        np.testing.assert_allclose(r.sigma, b.sigma, rtol=1e-10)
    bat.close()


def test_tile_falls_back():
    """Rows too long for a tile's batches (one of every column: 250,000
    entries of one row in some 30 batches) and a column half of the rows hit:
    the panels run those directions; bit for bit the row-block layout's."""
    m, n = 400000, 250000
    long_row = (np.full(n, 17), np.arange(n))
    A, rows, cols = _matrix(m, n, 11.0, seed=9, extra=[long_row])
    op = api.CsrOperator(A)
    res = _check(A, rows, cols, op, 4)
    op.set_sort(0, 0)
    x, got = res["n"]
    assert np.array_equal(op.spmv(x, "n"), got)
    # fewer rows in a tile than a batch has entries
    A, rows, cols = _matrix(9001, 1200, 700.0, seed=10)
    op = api.CsrOperator(A)
    res = _check(A, rows, cols, op, 5)
    op.set_sort(0, 0)
    for trans, (x, got) in res.items():
        assert np.array_equal(op.spmv(x, trans), got)


def test_tile_specials():
    """Infinities and NaN in x reach the rows that hold their columns and no
    other; subnormal products are kept; -0.0 adds to +0.0."""
    A, rows, cols = _matrix(270001, 260003, 16.5, seed=21)
    op = api.CsrOperator(A)
    x = np.ones(A.n)
    x[5], x[1000] = np.inf, np.nan
    got = op.spmv(x, "n")
    hit = np.zeros(A.m, bool)
    hit[rows[(cols == 5) | (cols == 1000)]] = True
    assert np.array_equal(~np.isfinite(got), hit)
    tiny = synth.Csr(A.m, A.n, A.rowptr, A.col, np.full(A.nnz, 2.0 ** -1070))
    got = api.CsrOperator(tiny).spmv(np.ones(A.n), "n")
    assert np.array_equal(got, np.diff(A.rowptr) * 2.0 ** -1070)
    neg = synth.Csr(A.m, A.n, A.rowptr, A.col, np.full(A.nnz, -0.0))
    got = api.CsrOperator(neg).spmv(np.ones(A.n), "n")
    assert not np.signbit(got).any()
