"""Lanczos steps of a small operator in one resident launch (at most 512 row
blocks of 1024 nonzeros per direction): bit for bit the host executor's
singular values, bounds, vectors and counters -- both run the same control
code on the same sums -- at the sizes where the launch changes: one row block,
one and two blocks per workgroup, the largest grid, more blocks than it takes
(the chains), more rows than one projection slice, wide and tall shapes, rows
of one nonzero, restarts, calls that leave the launch (invariant subspaces,
Lanczos dimensions past the LDS window), FP32 bases, and several engines'
launches at once."""
import threading

import numpy as np
import pytest

from propack_amd import api, synth

pytestmark = pytest.mark.gpu


def _solve(A, mode, prec, k, dim, irl=True, op=None, **kw):
    op = op or api.CsrOperator(A, prec=prec)
    eng = api.Engine(op, kmax=dim, prec=prec)
    if mode == "host":
        eng.set_mode("host", 2)
    eng.put_u1(synth.start_vector(A.m, 3))
    run = api.lansvd_irl_dev if irl else api.lansvd_dev
    r = run(eng, k, dim, tol=1e-5 if prec == api.PK_F32 else 1e-10, **kw)
    out = (r, eng.stats(), eng.path_stats(), eng.get("u", r.k), eng.get("v", r.k))
    eng.close()
    return out


def _same(a, b):
    (ra, sa, pa, ua, va), (rb, sb, pb, ub, vb) = a, b
    assert (ra.info, ra.k) == (rb.info, rb.k)
    assert np.array_equal(ra.sigma, rb.sigma) and np.array_equal(ra.bnd, rb.bnd)
    assert np.array_equal(ua, ub) and np.array_equal(va, vb)
    for key in ("nopx", "nreorth", "ndot", "ncols", "nretry"):
        assert sa[key] == sb[key], key
    assert pa == pb


@pytest.mark.parametrize("m,n,lam,k,dim", [
    (90, 60, 4.0, 5, 30),          # one row block
    (1850, 712, 4.7, 10, 60),
    (5003, 9001, 24.0, 8, 40),     # wide: 118 blocks, one per workgroup
    (131000, 4000, 1.0, 6, 30),    # many rows per block, 64 projection slices
    (20011, 9973, 12.5, 8, 40),    # two blocks per workgroup
    (30000, 20000, 16.9, 8, 40),   # 506 of at most 512 blocks
    (30000, 20000, 18.0, 8, 40),   # past it: the chains
    (700, 701, 480.0, 8, 40),      # rows of half a block
])
@pytest.mark.parametrize("prec", [api.PK_F64, api.PK_F32])
def test_resident_matches_host_executor(m, n, lam, k, dim, prec):
    A = synth.poisson_decay(m, n, lam, 0.5, seed=m + n,
                            dtype=np.float64 if prec == api.PK_F64 else np.float32)
    _same(_solve(A, "device", prec, k, dim), _solve(A, "host", prec, k, dim))


@pytest.mark.parametrize("kw", [dict(delta=0.0), dict(elr=0), dict(which="S")])
def test_resident_options(kw):
    """Full reorthogonalization, no ELR, the smallest triplets."""
    A = synth.random_uniform(400, 120, 4000, seed=5)
    dim = 60 if "which" in kw else 40
    _same(_solve(A, "device", api.PK_F64, 6, dim, maxiter=40, **kw),
          _solve(A, "host", api.PK_F64, 6, dim, maxiter=40, **kw))


def test_resident_leaves_for_the_host():
    """An exact-rank matrix (new random directions on the host between
    resident stretches), a matrix smaller than the Lanczos dimension, a zero
    matrix's start, and dimensions past the control state's LDS window."""
    rng = np.random.default_rng(2)
    B, C = rng.standard_normal((300, 7)), rng.standard_normal((7, 200))
    D = B @ C
    r, c = np.nonzero(D)
    low = synth.from_coo(300, 200, r, c, D[r, c])
    a = _solve(low, "device", api.PK_F64, 12, 40, irl=False)
    _same(a, _solve(low, "host", api.PK_F64, 12, 40, irl=False))
    assert sum(a[2][key] for key in ("v_invariant", "u_invariant")) > 0
    tiny = synth.random_uniform(40, 30, 600, seed=3)
    _same(_solve(tiny, "device", api.PK_F64, 10, 48), _solve(tiny, "host", api.PK_F64, 10, 48))
    A = synth.random_uniform(1850, 712)
    _same(_solve(A, "device", api.PK_F64, 200, 713, irl=False),
          _solve(A, "host", api.PK_F64, 200, 713, irl=False))


def test_resident_several_engines_at_once():
    """Solves on several threads, engines sharing an operator: each as alone."""
    A = synth.poisson_decay(12007, 5003, 9.3, 0.4, seed=8)
    op = api.CsrOperator(A)
    want = _solve(A, "device", api.PK_F64, 8, 40, op=op)
    got = [None] * 6

    def work(i):
        got[i] = _solve(A, "device", api.PK_F64, 8, 40, op=op)
    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(got))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for g in got:
        _same(g, want)
