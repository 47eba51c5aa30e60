"""Performance cases of the truncated-SVD library.

Each case is work that a program gives the library through its public entry
points, at the sizes of this repository's workloads and between them:

* ``solve``   device-resident DLANSVD_IRL (or its S / Z / C twin) on an
  operator and an engine the program keeps; the start vector comes from the
  GPU, the singular vectors stay there.
* ``dropin``  the Fortran drop-in DLANSVD with a device operator, start vector
  and singular vectors in host memory.
* ``batch``   independent uneven problems solved together.
* ``spmv``    one application of A and one of A^T to device vectors, enqueued
  without allocation, as an iterative method of the caller's own does it.

Matrices are sparse with Poisson row lengths, uniform columns and decaying
columns (``poisson``), or with power-law rows and Zipf columns, whose heavy
columns make rows of A^T of 10^5 and more nonzeros (``powerlaw``).
"""
import ctypes as C
import math

import numpy as np
import torch

from propack_amd import api, synth

# precision code, element type of the operator and the bases, of their real
# parts, type string of the device views
TYPES = {
    "f64": (api.PK_F64, torch.float64, torch.float64, "<f8"),
    "f32": (api.PK_F32, torch.float32, torch.float32, "<f4"),
    "c128": (api.PK_C128, torch.complex128, torch.float64, "<c16"),
    "c64": (api.PK_C64, torch.complex64, torch.float32, "<c8"),
}
# The SpMV layouts a program asks for: the one the library picks by itself
# ("default"); the one its autotuner names for millions of uniform rows,
# passed as fixed settings so that every run sums alike ("tuned"); and the
# batched workload's ("blocks").
LAYOUTS = {
    "default": {},
    "tuned": dict(panels=(8, 8), lanes=(0, 0), sort=(-8192, -8192)),
    "blocks": dict(lanes=(-2, -2), sort=(8192, 8192)),
}


def listed():
    return [
        # The small correctness workload's shape, one drop-in call: launches,
        # set-up and latency are all of it.
        dict(name="dropin_1850x712_f64", kind="dropin", pattern="poisson", m=1850, n=712,
             lam=4.67, decay=0.0, dtype="f64", layout="default", k=10, dim=300, tol=1e-12),
        # A small restarted solve on a kept engine, odd sizes.
        dict(name="solve_12007x5003_f64", kind="solve", pattern="poisson", m=12007, n=5003,
             lam=9.3, decay=0.4, dtype="f64", layout="default", k=10, dim=40, tol=1e-10),
        # The ordinary size of the solver tests.
        dict(name="solve_200kx100k_f64", kind="solve", pattern="poisson", m=200000, n=100000,
             lam=16.0, decay=0.6, dtype="f64", layout="default", k=20, dim=60, tol=1e-10),
        # FP32 storage with FP64 accumulation, odd sizes.
        dict(name="solve_1000003x500009_f32", kind="solve", pattern="poisson", m=1000003,
             n=500009, lam=16.0, decay=0.6, dtype="f32", layout="default", k=32, dim=96,
             tol=1e-6),
        # The headline workload.
        dict(name="solve_2Mx1M_f64", kind="solve", pattern="poisson", m=2000000, n=1000000,
             lam=16.0, decay=0.6, dtype="f64", layout="tuned", k=50, dim=120, tol=1e-10),
        # Heavy columns: long rows of A^T, many empty ones.
        dict(name="solve_powerlaw_1Mx500k_f64", kind="solve", pattern="powerlaw", m=1000000,
             n=500000, lam=0.0, decay=0.0, dtype="f64", layout="default", k=32, dim=80,
             tol=1e-8),
        # Complex bases.
        dict(name="solve_250kx125k_c128", kind="solve", pattern="poisson", m=250000, n=125000,
             lam=16.0, decay=0.6, dtype="c128", layout="default", k=20, dim=60, tol=1e-10),
        # Part of the batched workload in its own layout and form.
        dict(name="batch_24_f32", kind="batch", pattern="poisson", m=200000, n=5000, lam=48.0,
             decay=1.0, dtype="f32", layout="blocks", k=16, dim=48, tol=1e-8, count=24,
             shapes=4096),
        # The operator alone: the headline matrix as a program without tuning has it.
        dict(name="spmv_2Mx1M_f64", kind="spmv", pattern="poisson", m=2000000, n=1000000,
             lam=16.0, decay=0.6, dtype="f64", layout="default"),
        # FP32 values, odd sizes, tuned.
        dict(name="spmv_3000017x1500007_f32", kind="spmv", pattern="poisson", m=3000017,
             n=1500007, lam=12.0, decay=0.6, dtype="f32", layout="tuned"),
        # A small operator: two launches' latency.
        dict(name="spmv_9973x4409_f64", kind="spmv", pattern="poisson", m=9973, n=4409, lam=11.0,
             decay=0.5, dtype="f64", layout="default"),
        # Long rows and empty rows.
        dict(name="spmv_powerlaw_2Mx1M_f64", kind="spmv", pattern="powerlaw", m=2000000,
             n=1000000, lam=0.0, decay=0.0, dtype="f64", layout="default"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["solve", "solve", "solve", "spmv", "spmv", "spmv", "dropin", "batch"])
    if kind == "batch":
        return dict(kind=kind, pattern="poisson", m=_log(rng, 20000, 200000), n=5000, lam=48.0,
                    decay=1.0, dtype=rng.choice(["f32", "f32", "f64"]),
                    layout=rng.choice(["blocks", "blocks", "default"]), k=rng.randint(4, 16),
                    dim=rng.randint(36, 56), tol=1e-8, count=rng.randint(3, 24),
                    shapes=rng.randrange(1 << 20))
    pattern = "powerlaw" if kind != "dropin" and rng.random() < 0.2 else "poisson"
    lam = round(rng.uniform(4.0, 48.0), 2)
    hi = {"solve": 1200000, "dropin": 20000, "spmv": 3000000}[kind]
    m = _log(rng, 1500, hi)
    most = 16e6 if kind == "solve" else 32e6
    m = min(m, int(most / max(lam, 1.0)))
    n = max(600, int(m * rng.uniform(0.25, 1.4)))
    case = dict(kind=kind, pattern=pattern, m=m, n=n, lam=lam, decay=round(rng.uniform(0.3, 1.0), 2),
                dtype=rng.choice(["f64", "f64", "f32"]), layout="default")
    if m >= 1000000 and n >= 500000 and pattern == "poisson" and rng.random() < 0.5:
        case["layout"] = "tuned"
    if kind == "spmv":
        return case
    if rng.random() < 0.25:
        case["dtype"] = rng.choice(["c128", "c128", "c64"])
    if pattern == "powerlaw":
        case["m"], case["n"] = max(m, 50000), max(n, 25000)
    k = rng.randint(4, 40)
    single = case["dtype"] in ("f32", "c64")
    case.update(k=k, dim=2 * k + rng.randint(20, 40),
                tol=1e-5 if single else 10.0 ** -rng.randint(8, 10))
    if kind == "dropin":
        case["dim"] = 10 * k  # the Lanczos vectors a scipy caller allows
    return case


# ------------------------------------------------------------------ inputs --
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _coo(pattern, m, n, lam, decay, dtype, g):
    """Rows, columns (sorted, distinct) and values on the GPU."""
    dev = dict(device="cuda")
    if pattern == "poisson":
        deg = torch.poisson(torch.full((m,), float(lam), dtype=torch.float32, **dev), generator=g)
        deg = deg.to(torch.int64).clamp_(max=n)
    else:
        d = torch.arange(1, min(100000, n) + 1, dtype=torch.float64, **dev)
        cdf = torch.cumsum(d ** -2.1, 0)
        u = torch.rand(m, dtype=torch.float64, generator=g, **dev) * cdf[-1]
        deg = (torch.searchsorted(cdf, u) + 1).clamp_(max=d.numel())
    rows = torch.repeat_interleave(torch.arange(m, **dev), deg)
    if pattern == "poisson":
        cols = torch.randint(0, n, (rows.numel(),), generator=g, **dev)
    else:
        cdf = torch.cumsum(torch.arange(1, n + 1, dtype=torch.float64, **dev) ** -1.8, 0)
        u = torch.rand(rows.numel(), dtype=torch.float64, generator=g, **dev) * cdf[-1]
        cols = torch.randperm(n, generator=g, **dev)[torch.searchsorted(cdf, u).clamp_(max=n - 1)]
    key = torch.unique(rows * n + cols)
    rows, cols = key // n, key % n
    elem, real = TYPES[dtype][1:3]
    if pattern == "powerlaw":
        vals = torch.ones(cols.numel(), dtype=elem, **dev)
        if elem.is_complex:
            th = torch.rand(cols.numel(), dtype=torch.float64, generator=g, **dev) * (2 * math.pi)
            vals = torch.polar(torch.ones_like(th), th).to(elem)
        return rows, cols, vals
    mag = torch.randn(cols.numel(), dtype=torch.float64, generator=g, **dev)
    mag *= (1.0 + cols.to(torch.float64)) ** -decay
    if elem.is_complex:
        th = torch.rand(cols.numel(), dtype=torch.float64, generator=g, **dev) * (2 * math.pi)
        return rows, cols, torch.polar(mag.abs(), th).to(elem)
    return rows, cols, mag.to(elem)


def _csr(m, n, coo):
    """Host CSR arrays of device coordinates (sorted by row, then column)."""
    rows, cols, vals = coo
    rp = torch.zeros(m + 1, dtype=torch.int64, device="cuda")
    torch.cumsum(torch.bincount(rows, minlength=m), 0, out=rp[1:])
    return synth.Csr(m, n, rp.to(torch.int32).cpu().numpy(), cols.to(torch.int32).cpu().numpy(),
                     vals.cpu().numpy())


def _start(m, dtype, g):
    wide = torch.complex128 if TYPES[dtype][1].is_complex else torch.float64
    return torch.randn(m, dtype=wide, generator=g, device="cuda")


def _matrix(case, seed):
    g = _gen(seed)
    return _coo(case["pattern"], case["m"], case["n"], case["lam"], case["decay"], case["dtype"], g), g


def _problems(case):
    """The shapes of a batched case: synth.batch_params up to case["m"] rows."""
    return synth.batch_params(case["count"], 5000, case["m"], seed=case["shapes"])


class _Columns:
    """The first k columns of an engine's basis as a device array (k x L)."""

    def __init__(self, eng, which, k, typestr):
        p, ld = C.c_void_p(), C.c_longlong()
        api._check(api.lib().pk_lbd_basis(eng.handle, C.c_char(which.encode()), C.byref(p),
                                          C.byref(ld)), "pk_lbd_basis")
        size = int(typestr[2:])
        self.__cuda_array_interface__ = dict(
            shape=(k, eng.m if which == "u" else eng.n), typestr=typestr, version=2,
            data=(p.value, False), strides=(ld.value * size, size))


def _columns(eng, which, k, dtype):
    t = torch.as_tensor(_Columns(eng, which, k, TYPES[dtype][3]), device="cuda")
    t.engine = eng  # the view lives in the engine's memory: it keeps the engine
    return t


def prepare(case, seed):
    prec = TYPES[case["dtype"]][0]
    layout = LAYOUTS[case["layout"]]
    s = dict(case=case)
    if case["kind"] == "batch":
        s["engines"], s["starts"] = [], []
        g = _gen(seed)
        for p in _problems(case):
            A = _csr(p["m"], p["n"], _coo("poisson", p["m"], p["n"], p["lam"], p["p"],
                                          case["dtype"], g))
            eng = api.Engine(api.CsrOperator(A, prec, **layout), case["dim"])
            if case["dtype"] == "f32":
                eng.set_rounding(1)
            s["engines"].append(eng)
            s["starts"].append(_start(p["m"], case["dtype"], g))
        s["batch"] = api.Batch(s["engines"])
        torch.cuda.synchronize()
        return s
    coo, g = _matrix(case, seed)
    s["op"] = op = api.CsrOperator(_csr(case["m"], case["n"], coo), prec, **layout)
    if case["kind"] == "spmv":
        elem = TYPES[case["dtype"]][1]
        s["x"] = torch.randn(case["n"], dtype=torch.float64, generator=g, device="cuda").to(elem)
        s["u"] = torch.randn(case["m"], dtype=torch.float64, generator=g, device="cuda").to(elem)
        s["y"] = torch.empty(case["m"], dtype=elem, device="cuda")
        s["z"] = torch.empty(case["n"], dtype=elem, device="cuda")
    elif case["kind"] == "dropin":
        s["u0"] = _start(case["m"], case["dtype"], g).cpu().numpy()
    else:
        s["eng"] = api.Engine(op, case["dim"])
        if case["dtype"] == "f32":
            s["eng"].set_rounding(1)
        s["u0"] = _start(case["m"], case["dtype"], g)
    torch.cuda.synchronize()
    return s


def _apply(op, trans, x, y):
    api._check(api.lib().pk_csr_spmv_noalloc(
        op.handle, C.c_char(trans), C.c_void_p(x.data_ptr()), C.c_void_p(y.data_ptr()),
        C.c_int(op.prec), C.c_void_p(torch.cuda.current_stream().cuda_stream)),
        "pk_csr_spmv_noalloc")


def run(state):
    case = state["case"]
    if case["kind"] == "spmv":
        _apply(state["op"], b"n", state["x"], state["y"])
        _apply(state["op"], b"t", state["u"], state["z"])
        return dict(y=state["y"], z=state["z"])
    if case["kind"] == "dropin":
        r = api.lansvd(state["op"], case["m"], case["n"], case["k"], min(case["dim"], case["n"]),
                       u0=state["u0"], tol=case["tol"], prec=TYPES[case["dtype"]][0])
        return dict(sigma=r.sigma, u=r.U, v=r.V)
    if case["kind"] == "batch":
        for eng, u0 in zip(state["engines"], state["starts"]):
            eng.put_u1(u0)
        got = api.lansvd_irl_batch(state["batch"], case["k"], case["dim"], tol=case["tol"],
                                   jobu="y", jobv="y")
        return dict(sigma=np.concatenate([r.sigma for r in got]),
                    u=[_columns(e, "u", r.k, case["dtype"]) for e, r in zip(state["engines"], got)],
                    v=[_columns(e, "v", r.k, case["dtype"]) for e, r in zip(state["engines"], got)])
    eng = state["eng"]
    eng.put_u1(state["u0"])
    r = api.lansvd_irl_dev(eng, case["k"], case["dim"], tol=case["tol"], fetch=False)
    return dict(sigma=r.sigma, u=_columns(eng, "u", r.k, case["dtype"]),
                v=_columns(eng, "v", r.k, case["dtype"]))


def _spmv_bytes(m, n, nnz, size):
    """A applied once and A^T applied once."""
    return 2 * nnz * (size + 4.0) + (m + n + 2) * 4.0 + 2 * (m + n) * size


def _solve_work(m, n, nnz, size, steps, k, flop):
    """One Lanczos pass of that many steps: both operator applications, half
    of the steps reorthogonalized against the columns so far (the basis read
    once), and the singular vectors out of the bases."""
    basis = (m + n) * size
    return dict(bytes=steps * _spmv_bytes(m, n, nnz, size) + steps * steps / 4 * basis
                + (steps + k) * basis,
                flops=flop * (4.0 * steps * nnz + (m + n) * (steps * steps + 2.0 * steps * k)))


def work(case):
    size = TYPES[case["dtype"]][1].itemsize
    flop = 4.0 if TYPES[case["dtype"]][1].is_complex else 1.0
    if case["kind"] == "batch":
        parts = [_solve_work(p["m"], p["n"], p["m"] * p["lam"], size, case["dim"], case["k"], flop)
                 for p in _problems(case)]
        return dict(bytes=sum(p["bytes"] for p in parts), flops=sum(p["flops"] for p in parts))
    # the power law's mean degree, less what its heavy columns repeat
    nnz = case["m"] * (case["lam"] if case["pattern"] == "poisson" else 3.2)
    if case["kind"] == "spmv":
        return dict(bytes=_spmv_bytes(case["m"], case["n"], nnz, size), flops=4.0 * nnz * flop)
    steps = case["dim"] if case["kind"] == "solve" else min(case["dim"], 8 * case["k"])
    return _solve_work(case["m"], case["n"], nnz, size, steps, case["k"], flop)


def exact(case, seed):
    if case["kind"] == "batch":
        return None
    wide = torch.complex128 if TYPES[case["dtype"]][1].is_complex else torch.float64
    if case["kind"] == "spmv":
        (rows, cols, vals), g = _matrix(case, seed)
        elem = TYPES[case["dtype"]][1]
        x = torch.randn(case["n"], dtype=torch.float64, generator=g, device="cuda").to(elem).to(wide)
        u = torch.randn(case["m"], dtype=torch.float64, generator=g, device="cuda").to(elem).to(wide)
        v = vals.to(wide)
        return dict(y=_rowsums(rows, v * x[cols], case["m"]),
                    z=_rowsums(cols, v * u[rows], case["n"]))
    if case["n"] > 6000 or case["m"] > 30000:
        return None  # a dense decomposition would take too long
    # singular values of the dense matrix; the vectors' signs follow the
    # start vector, so they have no value of their own
    (rows, cols, vals), _ = _matrix(case, seed)
    D = torch.zeros(case["m"], case["n"], dtype=wide, device="cuda")
    D[rows, cols] = vals.to(wide)
    G = D.conj().T @ D if case["n"] <= case["m"] else D @ D.conj().T
    s = np.sqrt(np.maximum(np.linalg.eigvalsh(G.cpu().numpy())[::-1][:case["k"]], 0.0))
    real = np.float32 if case["kind"] == "dropin" and case["dtype"] in ("f32", "c64") else np.float64
    return dict(sigma=s.astype(real), u=None, v=None)


def _rowsums(idx, prod, length):
    """Sums of prod by idx: sorted, then differences of nothing larger than
    one segment."""
    order = torch.argsort(idx, stable=True)
    counts = torch.bincount(idx, minlength=length)
    return torch.segment_reduce(prod[order], "sum", lengths=counts)
