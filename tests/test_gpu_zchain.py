"""Complex Lanczos steps as gated device chains (one synchronization per
DLANBPRO call) against the host executor, bit for bit: the same control
stages on the same sums.  One and several column panels, both precisions,
restarts, full reorthogonalization, no ELR, a wide matrix, an exact-rank
matrix whose new directions run on the host in between, Lanczos dimensions
past the control state's LDS window, and steps that need a second
Gram-Schmidt pass (a chain of one pass leaves them to the host)."""
import numpy as np
import pytest

from propack_amd import api, synth

pytestmark = pytest.mark.gpu


def _solve(A, mode, prec, k, dim, irl=True, panels=None, tries=2, **kw):
    op = api.CsrOperator(A, prec, panels=panels)
    eng = api.Engine(op, kmax=dim)
    eng.set_mode(mode, tries)
    eng.put_u1(synth.start_vector(A.m, 3, np.complex128))
    run = api.lansvd_irl_dev if irl else api.lansvd_dev
    r = run(eng, k, dim, tol=1e-5 if prec == api.PK_C64 else 1e-10, **kw)
    out = (r, eng.stats(), eng.path_stats(), eng.get("u", r.k), eng.get("v", r.k))
    eng.close()
    return out


def _same(a, b, fewer_syncs=True):
    (ra, sa, pa, ua, va), (rb, sb, pb, ub, vb) = a, b
    assert (ra.info, ra.k) == (rb.info, rb.k)
    assert np.array_equal(ra.sigma, rb.sigma) and np.array_equal(ra.bnd, rb.bnd)
    assert np.array_equal(ua, ub) and np.array_equal(va, vb)
    for key in ("nopx", "nreorth", "ndot", "ncols", "nretry"):
        assert sa[key] == sb[key], key
    assert pa == pb
    if fewer_syncs:
        assert sa["nsync"] < sb["nsync"] / 3


@pytest.mark.parametrize("prec", [api.PK_C128, api.PK_C64])
@pytest.mark.parametrize("m,n,panels,k,dim", [
    (1850, 712, None, 8, 30), (1850, 712, (4, 8), 8, 30), (700, 1900, None, 6, 40),
    (30001, 20003, (2, 1), 8, 40),
])
def test_chain_matches_host_executor(m, n, panels, k, dim, prec):
    dt = np.complex128 if prec == api.PK_C128 else np.complex64
    A = synth.complex_uniform(m, n, 6 * m, seed=m, dtype=dt)
    _same(_solve(A, "device", prec, k, dim, panels=panels),
          _solve(A, "host", prec, k, dim, panels=panels))


@pytest.mark.parametrize("kw", [dict(delta=0.0), dict(elr=0), dict(tries=1)])
def test_chain_options(kw):
    A = synth.complex_poisson_decay(3000, 1500, 9.0, 0.9, seed=5)
    _same(_solve(A, "device", api.PK_C128, 8, 40, **kw),
          _solve(A, "host", api.PK_C128, 8, 40, **kw))


def test_chain_leaves_for_the_host():
    rng = np.random.default_rng(2)

    def z(*shape):
        return rng.standard_normal(shape) + 1j * rng.standard_normal(shape)
    D = z(300, 7) @ z(7, 200)
    r, c = np.nonzero(D)
    low = synth.from_coo(300, 200, r, c, D[r, c])
    a = _solve(low, "device", api.PK_C128, 12, 40, irl=False)
    _same(a, _solve(low, "host", api.PK_C128, 12, 40, irl=False), fewer_syncs=False)
    assert sum(a[2][key] for key in ("v_invariant", "u_invariant")) > 0
    A = synth.complex_uniform(1850, 712)
    _same(_solve(A, "device", api.PK_C128, 200, 713, irl=False),
          _solve(A, "host", api.PK_C128, 200, 713, irl=False))
