"""Rows past 1024 nonzeros: cut into parts and chunks that workgroups sum
apart, one list per XCD.  Lengths around the limits of the cut (1024 nonzeros
for a long row, parts of 4096, eight parts, chunks of 8192), alone and beside
short and empty rows, in every layout and direction, against FP64 sums on the
host."""
import numpy as np
import pytest

from propack_amd import api, synth

pytestmark = pytest.mark.gpu

LENGTHS = (1024, 1025, 4095, 4096, 8191, 8192, 8193, 28672, 32767, 32768, 65535, 65536, 65544,
           131073)
N = 140_001


def _matrix(lengths, seed):
    g = np.random.default_rng(seed)
    rows = []
    for k, length in enumerate(lengths):
        rows.append(np.sort(g.choice(N, length, replace=False)))
        rows.append(np.sort(g.choice(N, k % 3, replace=False)))  # short and empty rows
    rp = np.concatenate([[0], np.cumsum([len(r) for r in rows])]).astype(np.int32)
    return synth.Csr(len(rows), N, rp, np.concatenate(rows).astype(np.int32),
                     g.standard_normal(int(rp[-1])))


@pytest.mark.parametrize("prec", [api.PK_F64, api.PK_F32])
@pytest.mark.parametrize("kw", [{}, dict(sort=(1024, 1024)), dict(sort=(8192, 8192)),
                                dict(sort=(-1, -1)), dict(panels=(3, 2))])
@pytest.mark.parametrize("lengths", [LENGTHS, LENGTHS[:1], LENGTHS[1:2], LENGTHS[-1:],
                                     (1025,) * 9])
def test_long_rows(prec, kw, lengths):
    dt, u = (np.float64, 2.0 ** -53) if prec == api.PK_F64 else (np.float32, 2.0 ** -24)
    A = _matrix(lengths, len(lengths)).astype(dt)
    for B in (A, A.transpose()):  # long rows in A, then in A^T
        op = api.CsrOperator(B, prec, **kw)
        rows = np.repeat(np.arange(B.m), np.diff(B.rowptr))
        g = np.random.default_rng(7)
        x, w = g.standard_normal(B.n).astype(dt), g.standard_normal(B.m).astype(dt)
        for trans, v, r, c, size in (("n", x, rows, B.col, B.m), ("t", w, B.col, rows, B.n)):
            p = B.val.astype(np.float64) * v.astype(np.float64)[c]
            want = np.bincount(r, p, size)
            mass = np.bincount(r, np.abs(p), size)
            count = np.bincount(r, minlength=size)
            got = op.spmv(v, trans)
            # both sums in FP64, (count + 2) roundings each, and the store
            bound = 2 * (count + 2) * 2.0 ** -53 * mass + u * (np.abs(want) + mass * 2.0 ** -40)
            assert np.all(np.abs(got.astype(np.float64) - want) <= bound)


@pytest.mark.parametrize("prec", [api.PK_F64, api.PK_F32])
@pytest.mark.parametrize("empty", [1, 60])  # mean rows of about 90 and 3: many lanes a row, few
@pytest.mark.parametrize("kw", [dict(lanes=(s, s)) for s in range(-2, 3)]
                         + [dict(sort=(2048, 2048))])
def test_row_depth(prec, kw, empty):
    """Rows whose nonzeros per lane lie around the depths that a lane reads
    at a time (4 and 8), on 2 to 64 lanes a row, beside empty rows: whole
    numbers small enough that every product and sum is exact."""
    lengths = sorted({min(max(g * d + e, 0), 1024) for g in (2, 4, 8, 16, 32, 64)
                      for d in (1, 3, 4, 5, 7, 8, 9, 15, 16, 17) for e in (-1, 0, 1)})
    g = np.random.default_rng(5)
    rows = []
    for length in lengths:
        rows.append(np.sort(g.choice(4099, length, replace=False)))
        rows += [np.zeros(0, np.int64)] * empty
    rp = np.concatenate([[0], np.cumsum([len(r) for r in rows])]).astype(np.int32)
    dt = np.float64 if prec == api.PK_F64 else np.float32
    A = synth.Csr(len(rows), 4099, rp, np.concatenate(rows).astype(np.int32),
                  g.integers(-15, 16, int(rp[-1])).astype(dt))
    for B, trans in ((A, "n"), (A.transpose(), "t")):  # these rows in A, then in A^T
        op = api.CsrOperator(B, prec, **kw)
        x = g.integers(-15, 16, A.n).astype(dt)
        r = np.repeat(np.arange(A.m), np.diff(A.rowptr))
        want = np.bincount(r, A.val.astype(np.float64) * x.astype(np.float64)[A.col], A.m)
        assert np.array_equal(op.spmv(x, trans).astype(np.float64), want)
