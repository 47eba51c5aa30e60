"""Ritz vectors of a batched restarted solve: the small SVDs run on the host
threads and the basis products of all problems in one grouped launch per
side, with the same products as one problem's own, so values and vectors are
those of the problem solved alone, bit for bit.  Shapes with fewer than DIM
Lanczos steps (short sides, a low-rank matrix), a zero start vector and each
choice of sides."""
import numpy as np
import pytest

from propack_amd import api, synth

pytestmark = pytest.mark.gpu

NEIG, DIM, TOL = 8, 32, 1e-8


def _low_rank(m, n, rank):
    """Rows r of rank distinct columns, one nonzero each."""
    rp = np.minimum(np.arange(m + 1), rank).astype(np.int32)
    return synth.Csr(m, n, rp, np.arange(rank, dtype=np.int32) * 3,
                     np.linspace(9.0, 1.0, rank))


def _engines(prec):
    dt = np.float64 if prec == api.PK_F64 else np.float32
    mats = [synth.poisson_decay(m, n, lam, 0.8, seed=60 + m).astype(dt)
            for m, n, lam in ((61, 31, 4.0), (700, 1300, 9.0), (20011, 2003, 21.0))]
    mats.append(_low_rank(300, 90, 20).astype(dt))
    out = []
    for i, A in enumerate(mats):
        u0 = np.zeros(A.m) if i == 1 else synth.start_vector(A.m, 5 + i)
        out.append((api.Engine(api.CsrOperator(A, prec=prec), kmax=DIM, prec=prec), u0))
    return out


@pytest.mark.parametrize("prec", [api.PK_F64, api.PK_F32])
@pytest.mark.parametrize("jobu,jobv", [("y", "y"), ("y", "n"), ("n", "y"), ("n", "n")])
def test_batched_ritz_vectors_match_alone(prec, jobu, jobv):
    engs = _engines(prec)
    alone = []
    for e, u0 in engs:
        e.put_u1(u0)
        alone.append(api.lansvd_irl_dev(e, NEIG, DIM, tol=TOL, jobu=jobu, jobv=jobv))
    for e, u0 in engs:
        e.put_u1(u0)
    b = api.Batch([e for e, _ in engs])
    for _ in range(2):  # the second call finds its buffers allocated
        got = api.lansvd_irl_batch(b, NEIG, DIM, tol=TOL, jobu=jobu, jobv=jobv, fetch=True)
        for r, s in zip(got, alone):
            assert r.info == s.info and r.k == s.k and r.k >= NEIG
            assert np.array_equal(r.sigma, s.sigma) and np.array_equal(r.bnd, s.bnd)
            for x, y in ((r.U, s.U), (r.V, s.V)):
                assert (x is None) == (y is None)
                assert x is None or np.array_equal(x, y)
        for e, u0 in engs:
            e.put_u1(u0)
    b.close()
