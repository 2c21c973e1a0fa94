"""The work users of libukhip have it do, as cases that a timing program can run.

A case names one call pattern ("kind") and its sizes:

  device   ukhip_smooth_oddeven_noalloc: one problem whose inputs and outputs
           are in device memory, estimates and full covariances;
  batch    a device-resident batch (ukhip_batch_create in prepare, one
           smoothing and the download of its results per pass), by the FP64
           odd-even path (estimates, or estimates and covariance diagonals),
           the mixed-precision path, or the associative smoother;
  filter   the batched sequential filter fed from device memory;
  server   a burst of requests through the continuous-batching server;
  dropin   kalman_smooth_oddeven on host step equations, as a C client of the
           reference calls it.

The sizes are those of the benchmark workloads (n = 6; n = 48, m = 24; n = 64,
m = 32; batches of n in 4..32; requests of n in 3..16; 16-dimensional filters)
at lengths whose inputs take about a second to make.
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
for _d in (os.getcwd(), _ROOT):  # the tree it is run in, else the tree it is part of
    if os.path.isdir(os.path.join(_d, "ultimate-kalman_amd", "python")):
        sys.path.insert(0, os.path.join(_d, "ultimate-kalman_amd", "python"))
        break

from ukhip import capi, device, flops  # noqa: E402
from ukhip import problems as P  # noqa: E402

SCRATCH = 64 << 20  # UKHIP_NOALLOC_SCRATCH_BYTES
NO_COVARIANCE = capi.KALMAN_NO_COVARIANCE
COVARIANCE_DIAG = 1 << 25  # UKHIP_COVARIANCE_DIAG (include/ukhip.h)
INPUT_SETS = 8  # the filter cycles through this many steps' inputs


def listed():
    return [
        # the smallest call: a short track of a 4-state model (position and velocity in the plane)
        dict(name="device_n4_k64", kind="device", n=4, m=2, k=64, K="w", C="w", H=0, c=0, shared=1, unobserved=0.0),
        # a sensor-fusion state, inputs produced on the GPU, covariances consumed there
        dict(name="device_n16_k2500", kind="device", n=16, m=8, k=2500, K="w", C="w", H=0, c=1, shared=0,
             unobserved=0.1),
        # odd sizes, dense noise covariances and a general H: every block needs whitening
        dict(name="device_n45_k300_dense", kind="device", n=45, m=31, k=300, K="C", C="W", H=1, c=1, shared=0,
             unobserved=0.1),
        # a client of the reference's C API with its data in host memory
        dict(name="dropin_n6_k256", kind="dropin", n=6, m=6, k=256),
        # many independent tracks of mixed dimension, the headline's mixed-precision path
        dict(name="batch_mixed", kind="batch", path="mixed", refine=1, count=96, nmin=4, nmax=32, nstep=4, kmin=64,
             kmax=16384, half=1, seed=3),
        # the same kind of batch in FP64, estimates and variances
        dict(name="batch_fp64_diag", kind="batch", path="diag", refine=0, count=24, nmin=4, nmax=32, nstep=4, kmin=64,
             kmax=16384, half=1, seed=5),
        # one long, larger model in FP64, estimates and variances
        dict(name="long_n48_fp64", kind="batch", path="diag", refine=0, count=1, nmin=48, nmax=48, nstep=1, kmin=20000,
             kmax=20000, half=1, seed=2),
        # the largest dimension, mixed precision at the server's default of two refinements
        dict(name="long_n64_mixed", kind="batch", path="mixed", refine=2, count=1, nmin=64, nmax=64, nstep=1,
             kmin=10000, kmax=10000, half=1, seed=4),
        # the associative smoother on the long model
        dict(name="assoc_n48", kind="batch", path="assoc", refine=0, count=1, nmin=48, nmax=48, nstep=1, kmin=10000,
             kmax=10000, half=1, seed=7),
        # the associative smoother on a few requests of odd sizes
        dict(name="assoc_requests", kind="batch", path="assoc", refine=0, count=8, nmin=3, nmax=16, nstep=1, kmin=100,
             kmax=20000, half=0, seed=11),
        # a bank of filters advanced step by step as measurements arrive on the GPU
        dict(name="filter_n16", kind="filter", filters=1024, n=16, m=8, steps=200, history=0),
        # a burst of requests to the server, FP64 with covariances
        dict(name="server_fp64", kind="server", count=24, kmin=100, kmax=8000, mixed=-1, seed=13),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["device", "device", "batch", "batch", "batch", "batch", "filter", "server", "dropin"])
    if kind == "device":
        n = rng.randint(1, 60)
        most = int(0.9 * SCRATCH / (8 * (10 * n * n + 12 * n + 8)))
        return dict(kind=kind, n=n, m=rng.randint(max(1, n // 4), n), k=_log_int(rng, 16, min(most, 20000)),
                    K=rng.choice("wwWCU"), C=rng.choice("wwWCF"), H=rng.choice([0, 0, 1]), c=rng.randint(0, 1),
                    shared=rng.randint(0, 1), unobserved=rng.choice([0.0, 0.1]))
    if kind == "batch":
        path = rng.choice(["mixed", "mixed", "diag", "states", "assoc"])
        if rng.random() < 0.5:  # one long problem
            n = rng.randint(3, 64)
            k = _log_int(rng, 300, min(60000, int((8 if path == "assoc" else 18) * 2.3e6 / (n * n))))
            return dict(kind=kind, path=path, refine=2 if n > 48 else rng.randint(1, 2), count=1, nmin=n, nmax=n,
                        nstep=1, kmin=k, kmax=k, half=rng.randint(0, 1), seed=rng.randrange(1 << 30))
        lo, hi = rng.choice([(3, 16), (4, 32), (17, 32), (3, 12)])
        return dict(kind=kind, path=path, refine=1, count=_log_int(rng, 4, 8 if path == "assoc" else 40), nmin=lo,
                    nmax=hi, nstep=rng.choice([1, 1, 4]), kmin=64, kmax=_log_int(rng, 1000, 16384),
                    half=rng.randint(0, 1), seed=rng.randrange(1 << 30))
    if kind == "filter":
        n, history = rng.randint(2, 24), rng.randint(0, 1)
        return dict(kind=kind, filters=_log_int(rng, 64, 300 if history else 2000), n=n, m=rng.randint(1, n),
                    steps=rng.randint(20, 100), history=history)
    if kind == "server":
        return dict(kind=kind, count=rng.randint(4, 24), kmin=100, kmax=_log_int(rng, 500, 8000),
                    mixed=rng.choice([-1, -1, 2]), seed=rng.randrange(1 << 30))
    n = rng.randint(2, 16)
    return dict(kind=kind, n=n, m=rng.randint(1, n), k=rng.randint(64, 400))


# ---- inputs ------------------------------------------------------------------------
# Matrices are kept as the C layout has them: per step, column-major, so an
# array entry [i] holds the transpose of step i's matrix.

def _orthogonal(rng, n):
    q, r = np.linalg.qr(rng.standard_normal((n, n)))
    return q * np.where(np.diag(r) < 0, -1.0, 1.0)


def _noise(rng, kind, k, dim, var):
    """Per-step noise covariances of size dim about var in representation
    `kind`: (stored array, precision matrices or their diagonals)."""
    s = rng.uniform(0.7, 1.4, size=k)
    if kind == "w":
        d = s[:, None] * rng.uniform(0.8, 1.25, size=(1, dim)) / math.sqrt(var)
        return d, d * d
    a = 0.3 * rng.standard_normal((dim, dim)) / math.sqrt(dim) + np.eye(dim)
    low = np.linalg.cholesky(a @ a.T) * math.sqrt(var)  # covariance low low^T / s^2
    inv = np.linalg.inv(low)
    prec = s[:, None, None] ** 2 * (inv.T @ inv)[None]
    if kind == "W":
        return s[:, None, None] * inv.T[None], prec
    if kind == "C":
        return (low @ low.T).T[None] / s[:, None, None] ** 2, prec
    return low.T[None] / s[:, None, None], prec  # 'U', 'F'


def _arrays(rng, n, m, k, K="w", C="w", H=0, c=0, shared=1, unobserved=0.0, Kvar=1.0, Cvar=1.0, fscale=0.99):
    """One problem: the arrays of ukhip_problem_t, and what exact() needs."""
    d = dict(n=n, m=m, k=k, K_type=K, C_type=C, shared=shared)
    F = fscale * _orthogonal(rng, n)
    d["F"] = np.ascontiguousarray(F.T)
    if not shared:
        d["F"] = d["F"][None] * rng.uniform(0.9, 1.0, size=(k, 1, 1))
    d["H"] = None
    if H:
        Hm = np.eye(n)[None] + 0.2 / math.sqrt(n) * rng.standard_normal((k, n, n))
        d["H"] = Hm
    d["c"] = 0.1 * rng.standard_normal((k, n)) if c else np.zeros((k, n))
    d["K"], d["Kp"] = _noise(rng, K, k, n, Kvar)
    d["C"], d["Cp"] = _noise(rng, C, k, m, Cvar)
    d["G"] = rng.standard_normal((k, n, m)) * (1.0 / math.sqrt(n))
    d["o"] = rng.standard_normal((k, m))
    mi = np.where(rng.random(k) < unobserved, 0, m).astype(np.int32)
    mi[: -(-n // m)] = m  # the first steps determine the state, so that every smoother takes the problem
    d["m_i"] = mi
    return d


def _specs(case):
    """(n, m, k, options) of every problem of a batch, server or dropin case:
    sizes by the case alone, so that every pass of a case has the same work."""
    if case["kind"] == "dropin":
        return [(case["n"], case["m"], case["k"], {})]
    r = np.random.Generator(np.random.Philox(case["seed"]))
    out = []
    server = case["kind"] == "server"
    for _ in range(case["count"]):
        n = int(r.choice(np.arange(3, 17))) if server else int(r.choice(np.arange(case["nmin"], case["nmax"] + 1,
                                                                                 case["nstep"])))
        k = int(math.exp(r.uniform(math.log(case["kmin"]), math.log(case["kmax"] + 1))))
        m = max(1, n // 2) if not server and case["half"] else int(r.integers(max(1, n // 2), n + 1))
        opt = {}
        if server or not case["half"]:
            opt = dict(unobserved=0.05, Cvar=0.1)
        if not server and case["count"] == 1:
            opt = dict(opt, Kvar=1.0 if n <= 48 else 1e-2, unobserved=0.1 if n >= 17 else 0.0, shared=int(n >= 32))
        out.append((n, m, max(k, 1), opt))
    return out


def _inputs(case, seed):
    rng = np.random.Generator(np.random.Philox(seed))
    if case["kind"] == "device":
        return [_arrays(rng, case["n"], case["m"], case["k"], case["K"], case["C"], case["H"], case["c"],
                        case["shared"], case["unobserved"])]
    return [_arrays(rng, n, m, k, **opt) for n, m, k, opt in _specs(case)]


def _problem(d):
    """A packed problem as the package's batch and server classes take it."""
    n, k = d["n"], d["k"]
    packed = dict(n=n, m=d["m"], F=d["F"], G=d["G"], c=d["c"], o=d["o"], m_i=d["m_i"], K_steps=d["K"],
                  K_type=d["K_type"], C_steps=d["C"], C_type=d["C_type"], H=d["H"])
    if d["shared"]:
        packed["F_shared"] = d["F"].T
    p = P.Problem(k=k, n=[n] * k, H=[], F=[], c=[], K=[], K_type=[], G=[], o=[], C=[], C_type=[])
    p.packed = packed
    return p


def _step_lists(d):
    """The same problem as one matrix per step (the reference's form)."""
    n, m, k = d["n"], d["m"], d["k"]
    F = d["F"].T
    H = np.eye(n)
    return P.Problem(k=k, n=[n] * k, H=[None] + [H] * (k - 1), F=[None] + [F] * (k - 1),
                     c=[None] + [d["c"][i].reshape(n, 1) for i in range(1, k)],
                     K=[None] + [d["K"][i].reshape(n, 1) for i in range(1, k)], K_type=[None] + ["w"] * (k - 1),
                     G=[d["G"][i].T for i in range(k)], o=[d["o"][i].reshape(m, 1) for i in range(k)],
                     C=[d["C"][i].reshape(m, 1) for i in range(k)], C_type=["w"] * k)


def _filter_inputs(case, seed):
    rng = np.random.Generator(np.random.Philox(seed))
    nf, n, m = case["filters"], case["n"], case["m"]
    F = 0.98 * _orthogonal(rng, n)
    sets = [dict(K=rng.uniform(0.8, 1.25, size=(nf, n)), G=rng.standard_normal((nf, m, n)) / math.sqrt(n),
                 o=rng.standard_normal((nf, m)), C=rng.uniform(0.8, 1.25, size=(nf, m)))
            for _ in range(INPUT_SETS)]
    return F, sets


# ---- the calls ----------------------------------------------------------------------

def _library():
    L = device.lib()
    L.ukhip_smooth_oddeven_noalloc.argtypes = [ctypes.c_void_p, ctypes.c_uint32, ctypes.c_void_p, ctypes.c_void_p,
                                               ctypes.c_void_p]
    L.ukhip_smooth_oddeven_noalloc.restype = ctypes.c_int
    return L


def _check(rc):
    if rc != 0:
        raise RuntimeError(device.last_error())


def prepare(case, seed):
    L = _library()
    kind = case["kind"]
    st = dict(kind=kind, case=case, L=L)
    if kind == "device":
        d = _inputs(case, seed)[0]
        s = device.ProblemStruct()
        s.n, s.m, s.k, s.F_shared = d["n"], d["m"], d["k"], d["shared"]
        s.K_type, s.C_type = d["K_type"].encode(), d["C_type"].encode()
        keep = []
        for f in ("F", "H", "c", "K", "G", "o", "C", "m_i"):
            if d[f] is not None:
                t = torch.from_numpy(np.ascontiguousarray(d[f])).cuda()
                keep.append(t)
                setattr(s, f, t.data_ptr())
        x = torch.empty((d["k"], d["n"]), dtype=torch.float64, device="cuda")
        S = torch.empty((d["k"], d["n"], d["n"]), dtype=torch.float64, device="cuda")
        torch.cuda.synchronize()
        st.update(problem=s, keep=keep, x=x, S=S)
    elif kind == "batch":
        probs = [_problem(d) for d in _inputs(case, seed)]
        b = device.Batch(probs)
        # results go into one page-locked buffer that is kept, a piece per problem
        sizes = [p.k * p.n[0] for p in probs]
        want_d = case["path"] in ("diag", "assoc")
        x = torch.empty(sum(sizes), dtype=torch.float64, pin_memory=True)
        v = torch.empty(sum(sizes), dtype=torch.float64, pin_memory=True) if want_d else None
        st.update(batch=b, x=x, v=v, at=[8 * int(a) for a in np.cumsum([0] + sizes[:-1])])
    elif kind == "filter":
        F, sets = _filter_inputs(case, seed)
        st["sets"] = [device.Filter.upload(F=F, **s) for s in sets]
    elif kind == "server":
        st["problems"] = [_problem(d) for d in _inputs(case, seed)]
        st["server"] = device.Server(hbm_budget_bytes=4 << 30, max_batch=64, max_inflight=4,
                                     mixed_refinements=case["mixed"])
    else:
        st["equations"] = capi.EquationSet(_step_lists(_inputs(case, seed)[0]))
    return st


def run(state):
    L, case, kind = state["L"], state["case"], state["kind"]
    if kind == "device":
        _check(L.ukhip_smooth_oddeven_noalloc(ctypes.byref(state["problem"]), 0, state["x"].data_ptr(),
                                              state["S"].data_ptr(), None))
        return {"x": state["x"], "S": state["S"]}
    if kind == "batch":
        b, path = state["batch"], case["path"]
        if path == "mixed":
            b.smooth_mixed_opt(refinements=case["refine"], sync=False)
        elif path == "assoc":
            b.smooth("associative", sync=False)
        else:
            b.smooth("oddeven", COVARIANCE_DIAG if path == "diag" else NO_COVARIANCE, sync=False)
        x, v = state["x"].data_ptr(), state["v"].data_ptr() if state["v"] is not None else None
        for i, at in enumerate(state["at"]):
            _check(L.ukhip_batch_download(b.h, i, x + at, None))
            if v is not None:
                _check(L.ukhip_batch_download_cov(b.h, i, b"D", v + at))
        return {"x": state["x"]} if v is None else {"x": state["x"], "v": state["v"]}
    if kind == "filter":
        f = device.Filter(case["filters"], case["n"], case["m"])
        if case["history"]:
            f.keep_history(case["steps"])
        for t in range(case["steps"]):
            f.step_device(state["sets"][t % INPUT_SETS])
        if case["history"]:
            xs, W = f.smooth()
            out = {"xs": xs, "W": W}
        else:
            x, R = f.estimates()
            out = {"x": x, "R": R}
        f.close()
        return out
    if kind == "server":
        srv = state["server"]
        ids = [srv.submit(p) for p in state["problems"]]
        out = [srv.wait(r, want_cov=case["mixed"] < 0) for r in ids]
        return [[x, S] if S is not None else [x] for x, S, _ in out]
    eqs = state["equations"]
    L.ukhip_clear_error()
    L.kalman_smooth_oddeven(0, eqs.ptrs, eqs.problem.k)
    if device.last_error():
        raise RuntimeError(device.last_error())
    xs, Ss = eqs.collect(L.matrix_free)
    return {"x": np.stack(xs), "S": np.stack(Ss)}


# ---- what a pass cannot do without --------------------------------------------------------

def work(case):
    """Inputs read once and outputs written once; the reference's operations
    (ukhip.flops), counted over a short chain and scaled to the length."""
    kind = case["kind"]
    if kind == "filter":
        nf, n, m, T = case["filters"], case["n"], case["m"], case["steps"]
        # evolve: QR of 2n x n with n + 1 more columns; observe: QR of (n + m) x n with one more
        fl = nf * T * (2 * (2 * n) * n * n - 2 * n ** 3 / 3 + (n + 1) * 6 * n * n + 2 * (n + m) * n * n - 2 * n ** 3 / 3)
        by = 8 * (T * nf * (n + m * n + 2 * m) + n * n + nf * (n + n * n) * (T if case["history"] else 1))
        return {"bytes": by, "flops": fl}
    by = fl = 0
    if kind == "device":
        specs = [(case["n"], case["m"], case["k"], case)]
    else:
        specs = _specs(case)
    assoc = kind == "batch" and case["path"] == "assoc"
    full = kind in ("device", "dropin") or (kind == "server" and case["mixed"] < 0)
    diag = kind == "batch" and case["path"] in ("diag", "assoc")
    for n, m, k, opt in specs:
        Kt, Ct = opt.get("K", "w"), opt.get("C", "w")
        by += 8 * (k * (m * n + m + n) + k * (n if Kt == "w" else n * n) + k * (m if Ct == "w" else m * m))
        by += 8 * n * n * ((1 if opt.get("shared", 1) else k) + (k if opt.get("H") else 0)) + 4 * k
        by += 8 * k * (n + (n * n if full else n if diag else 0))
        q = min(k, 64)
        if assoc:
            fl += flops.associative_flops(n, [m] * q)["total"] * k / q
        else:
            fl += flops.oddeven_flops(n, [m] * q, [Kt] * q, [Ct] * q, cov=full or diag)["total"] * k / q
    return {"bytes": float(by), "flops": float(fl)}


# ---- the same results in plain torch, 64 bits ---------------------------------------------

def _cyclic(T, U, b):
    """Solution and the diagonal and first off-diagonal blocks of the inverse
    of the block tridiagonal system with diagonal blocks T, blocks (i, i+1) U
    and right-hand side b, by cyclic reduction."""
    L, n = T.shape[0], T.shape[1]
    if L == 1:
        Ti = torch.linalg.inv(T)
        return Ti @ b, Ti, U
    ne, no = (L + 1) // 2, L // 2
    Ti = torch.linalg.inv(T[0::2])
    A = torch.zeros((ne, n, n), dtype=T.dtype, device=T.device)  # block (j, j-1) of even j
    A[1:] = U[1::2][: ne - 1].transpose(1, 2)
    R = torch.zeros_like(A)  # block (j, j+1)
    R[:no] = U[0::2]
    Wl, Wr, y = Ti @ A, Ti @ R, Ti @ b[0::2]
    To = T[1::2] - R[:no].transpose(1, 2) @ Wr[:no]
    bo = b[1::2] - R[:no].transpose(1, 2) @ y[:no]
    q = ne - 1  # odd steps with an even step behind them
    To[:q] = To[:q] - A[1:].transpose(1, 2) @ Wl[1:]
    bo[:q] = bo[:q] - A[1:].transpose(1, 2) @ y[1:]
    Uo = -A[1:no].transpose(1, 2) @ Wr[1:no]
    xo, So, Xo = _cyclic(To, Uo, bo)
    x = torch.empty_like(b)
    S = torch.empty_like(T)
    X = torch.empty_like(U)
    x[1::2], S[1::2] = xo, So
    xl, xr = torch.zeros_like(y), torch.zeros_like(y)
    Sl, Sr, Sx = torch.zeros_like(A), torch.zeros_like(A), torch.zeros_like(A)
    xl[1:], xr[:no] = xo[: ne - 1], xo
    Sl[1:], Sr[:no] = So[: ne - 1], So
    Sx[1:no] = Xo  # Cov(left, right) where both are there
    x[0::2] = y - Wl @ xl - Wr @ xr
    Cl = Wl @ Sl + Wr @ Sx.transpose(1, 2)  # -Cov(j, j-1)
    Cr = Wl @ Sx + Wr @ Sr                  # -Cov(j, j+1)
    Sj = Ti + Cl @ Wl.transpose(1, 2) + Cr @ Wr.transpose(1, 2)
    S[0::2] = 0.5 * (Sj + Sj.transpose(1, 2))
    X[0::2] = -Cr[:no]
    X[1::2] = -Cl[1:].transpose(1, 2)[: L - 1 - no]
    return x, S, X


def _smoothed(d):
    """(estimates, covariances) of one problem from its normal equations."""
    dev = "cuda" if torch.cuda.is_available() else "cpu"

    def put(a):
        return torch.from_numpy(np.ascontiguousarray(a)).to(dev)

    n, m, k = d["n"], d["m"], d["k"]
    F = put(d["F"]).transpose(-1, -2)
    F = F.expand(k, n, n) if d["shared"] else F
    H = put(d["H"]).transpose(1, 2) if d["H"] is not None else torch.eye(n, dtype=torch.float64, device=dev).expand(k, n, n)
    G, c, o = put(d["G"]).transpose(1, 2), put(d["c"])[..., None], put(d["o"])[..., None]
    Kp, Cp, seen = put(d["Kp"]), put(d["Cp"]), put((d["m_i"] > 0).astype(np.float64))[:, None, None]

    def times(p, a):  # precision times a
        return p[..., None] * a if p.dim() == 2 else p @ a

    GC = times(Cp, G).transpose(1, 2) * seen
    T, b = GC @ G, GC @ o
    KH, KF = times(Kp, H)[1:], times(Kp, F)[1:]
    T[1:] += H[1:].transpose(1, 2) @ KH
    T[:-1] += F[1:].transpose(1, 2) @ KF
    b[1:] += KH.transpose(1, 2) @ c[1:]
    b[:-1] -= KF.transpose(1, 2) @ c[1:]
    U = -F[1:].transpose(1, 2) @ KH
    x, S, _ = _cyclic(T, U, b)
    return x[..., 0], S


def exact(case, seed):
    kind = case["kind"]
    if kind == "filter":
        dev = "cuda" if torch.cuda.is_available() else "cpu"
        if case["history"]:
            return None
        Fn, sets = _filter_inputs(case, seed)
        F = torch.from_numpy(Fn).to(dev)
        sets = [{q: torch.from_numpy(v).to(dev) for q, v in s.items()} for s in sets]
        nf, n = case["filters"], case["n"]
        Lam = torch.zeros((nf, n, n), dtype=torch.float64, device=dev)
        eta = torch.zeros((nf, n, 1), dtype=torch.float64, device=dev)
        for t in range(case["steps"]):
            s = sets[t % INPUT_SETS]
            if t:  # predict in information form
                Q = torch.diag_embed(s["K"] ** 2)
                QF = Q @ F
                M = torch.linalg.solve(Lam + F.T @ QF, torch.cat((QF.transpose(1, 2), eta), 2))
                Lam, eta = Q - QF @ M[..., :n], QF @ M[..., n:]
                Lam = 0.5 * (Lam + Lam.transpose(1, 2))
            GC = (s["C"][..., None] ** 2 * s["G"]).transpose(1, 2)
            Lam, eta = Lam + GC @ s["G"], eta + GC @ s["o"][..., None]
        if case["steps"] * case["m"] < n:
            return None
        return {"x": torch.linalg.solve(Lam, eta)[..., 0], "R": None}  # R's row signs are free
    res = [_smoothed(d) for d in _inputs(case, seed)]
    if kind == "batch":
        x = torch.cat([x.reshape(-1) for x, _ in res]).cpu()
        if case["path"] in ("mixed", "states"):
            return {"x": x}
        return {"x": x, "v": torch.cat([torch.diagonal(S, dim1=1, dim2=2).reshape(-1) for _, S in res]).cpu()}
    if kind == "server":
        return [[x.cpu(), S.cpu()] if case["mixed"] < 0 else [x.cpu()] for x, S in res]
    return {"x": res[0][0], "S": res[0][1]}
