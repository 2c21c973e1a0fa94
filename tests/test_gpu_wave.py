"""The kernels that give a wave, or a wave per matrix column tile, to a step
pair, a filter or an element: the elimination and back substitution for n <= 32
(oddeven_small.hip, oddeven_mid*.hip, k_backsub_small), the batched filter for
n <= 16 (filter_small.hip), the associative scan (associative.hip), and the
lanes of a composite batch. State dimensions at the edges of the register
granules (4) and tiles (16), lengths and batch sizes around the splits.

Bars: FP64 results within 1e-9 (per-step normwise relative) of the oracle or of
a square-root information filter in numpy, the bar of the other kernel tests;
the mixed path after three refinement steps within 1e-9 of the FP64 estimates;
a composite's results bit for bit those of its parts alone (the same launches).
An associative smoothing with process noise of condition 1e8 may lose what that
condition costs a covariance form, 64 * 2.2e-16 * 1e8 = 1.4e-6.
"""
import os

import numpy as np
import pytest

from checks import assoc_parity, max_rel_err, rel_err
from ukhip import capi
from ukhip import problems as P

pytestmark = pytest.mark.gpu

TOL = 1e-9
UKHIP_COVARIANCE_DIAG = 1 << 25


@pytest.fixture(scope="module")
def dev():
    from ukhip import device
    device.lib()
    return device


@pytest.fixture(autouse=True)
def threads(oracle):
    oracle.lib.oracle_set_threads(min(16, os.cpu_count() or 1))
    yield
    oracle.lib.oracle_set_threads(1)


def _iid(k, n, m, kind="w", unobserved=lambda i: i % 10 == 9):
    F = 0.97 * P.random_orthogonal(P.rng_for(1000 + n), n)
    return P.iid_problem(k, n, m, seed=1100 + k + m, F=F, G_scale=1 / np.sqrt(n), Cvar=0.1, K_kind=kind, C_kind=kind,
                         unobserved=unobserved, name=f"n{n}_m{m}_{kind}_k{k}")


def _check(dev, oracle, probs, mixed=True):
    b = dev.Batch(probs)
    try:
        b.smooth("oddeven")
        full = [b.download(i) for i in range(len(probs))]
        b.smooth("oddeven", options=capi.KALMAN_NO_COVARIANCE)
        est = [b.download(i, want_cov=False)[0] for i in range(len(probs))]
        b.smooth("oddeven", options=UKHIP_COVARIANCE_DIAG)
        diag = [b.download_cov(i, "D") for i in range(len(probs))]
        if mixed:
            b.smooth_mixed_opt(3, 0, False)
        for i, pr in enumerate(probs):
            (x, S), (ox, oc) = full[i], oracle.oddeven(pr)
            assert max_rel_err(list(x), ox) < TOL and max_rel_err(list(S), oc) < TOL, pr.name
            assert max_rel_err(list(est[i]), ox) < TOL, pr.name
            assert max_rel_err(list(diag[i]), [np.diag(c) for c in oc]) < TOL, pr.name
            if mixed:
                assert max_rel_err(list(b.download(i, want_cov=False)[0]), list(x)) < TOL, pr.name
    finally:
        b.free()


@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 8, 9, 12, 13, 16, 17, 20, 21, 24, 25, 28, 29, 32])
def test_wave_elimination(dev, oracle, n):
    """'w' weights with H = I (B formed on load, D diagonal), full weights with
    H = I, and a dense H; few rows, half of the rows and one more, all, more than n; lone
    steps, one pair, odd chains."""
    half = 4 * (((n + 3) // 4 + 1) // 2)  # the rows of the half-block kernels
    for m in sorted({1, min(half, n), min(half + 1, n), n}):
        ks = (1, 2, 40) if m == n else (2 * (n // m) + 3, 2 * (n // m) + 40)
        for kind in "wC":
            _check(dev, oracle, [_iid(k, n, m, kind) for k in ks], mixed=2 * m >= n)
    if n > 1:  # n = 1: the problems' random H may be singular
        pr = P.random_problem(1200 + n, 19, n, n, K_kind="W", C_kind="w", H_kind="R", unobserved=(3, 17))
        (xs, Ss), (ox, oc) = dev.smooth_equations(pr, "oddeven"), oracle.oddeven(pr)
        assert max_rel_err(xs, ox) < TOL and max_rel_err(Ss, oc) < TOL, pr.name
    _check(dev, oracle, [_iid(9, n, n + 3)])


@pytest.mark.parametrize("n,k", [(3, 2047), (3, 2050), (16, 2050), (17, 2048), (17, 2053), (32, 2053)])
def test_long_and_short_levels(dev, oracle, n, k):
    """Level 0 at 1024 and 1025 pairs (n <= 16: where three waves share a pair);
    level 1 at 512 and 514 (17 <= n <= 32: one launch a level or three)."""
    _check(dev, oracle, [_iid(k, n, (n + 1) // 2)])


def _whiten(kind, v):
    """V with V cov V^T = I for a covariance in representation `kind`."""
    if kind == "w":
        return np.diag(v.ravel())
    return v if kind == "W" else np.linalg.inv(np.linalg.cholesky(v))


@pytest.mark.parametrize("n,m", [(1, 1), (2, 2), (4, 1), (5, 5), (8, 8), (9, 4), (12, 12), (13, 2), (15, 15), (16, 8),
                                 (16, 16)])
@pytest.mark.parametrize("kt,ct,full", [("w", "w", False), ("C", "W", True), ("w", "C", True)])
def test_wave_filter(dev, n, m, kt, ct, full):
    """Estimates and information matrices of 70 filters over 9 steps, some steps
    unobserved, against the square-root information filter (QR of the stacked
    rows) in numpy. (In information form, Lam = W - W F (..) F^T W, numpy itself
    loses up to 1e-8 of the estimates with full covariances here.)"""
    nf, steps = 70, 9
    rng = P.rng_for(1300 + 17 * n + m)

    def cov(kind, d):
        if kind == "w":
            return rng.uniform(0.5, 2.0, d)
        a = 0.3 * rng.standard_normal((d, d)) + 1.5 * np.eye(d)
        return a @ a.T if kind == "C" else np.linalg.inv(np.linalg.cholesky(a @ a.T))

    rows = [np.zeros((0, n + 1)) for _ in range(nf)]  # [R | y]
    flt = dev.Filter(nf, n, m)
    try:
        for t in range(steps):
            F = 0.9 * P.random_orthogonal(P.rng_for(1400 + t), n)
            H = np.stack([np.eye(n) + 0.05 * rng.standard_normal((n, n)) for _ in range(nf)]) if full else None
            c = rng.standard_normal((nf, n)) if full else None
            K = np.stack([cov(kt, n) for _ in range(nf)])
            C = np.stack([cov(ct, m) for _ in range(nf)])
            G, o = rng.standard_normal((nf, m, n)) / np.sqrt(n), rng.standard_normal((nf, m))
            mi = np.full(nf, m, dtype=np.int32)
            if t:
                mi[(np.arange(nf) + t) % 5 == 0] = 0
            flt.step(K=K, G=G, o=o, C=C, F=np.stack([F] * nf), H=H, c=c, m_i=mi, K_type=kt, C_type=ct)
            for p in range(nf):
                if t:  # H x_t = F x_(t-1) + c + noise, past state eliminated
                    V = _whiten(kt, K[p])
                    A, cc = (H[p], c[p]) if full else (np.eye(n), np.zeros(n))
                    old = np.column_stack((rows[p][:, :n], np.zeros((len(rows[p]), n)), rows[p][:, n]))
                    q = np.linalg.qr(np.vstack((old, np.column_stack((-V @ F, V @ A, V @ cc)))), mode="r")
                    rows[p] = q[n:, n:]
                if mi[p]:
                    V = _whiten(ct, C[p])
                    q = np.linalg.qr(np.vstack((rows[p], np.column_stack((V @ G[p], V @ o[p])))), mode="r")
                    rows[p] = q[:n]
        x, R = flt.estimates()
        for p in range(nf):
            U, y = rows[p][:n, :n], rows[p][:n, n]
            assert rel_err(R[p].T @ R[p], U.T @ U) < TOL and rel_err(x[p], np.linalg.solve(U, y)) < TOL, p
    finally:
        flt.close()


@pytest.mark.parametrize("n", [1, 4, 5, 8, 12, 13, 16, 17, 31, 32, 33, 47, 48, 49, 64])
def test_associative_tiles(dev, oracle, n):
    """The model taken from the inputs ('w', H = I) and solved for (full weights,
    dense H); priors over one and several steps; one step, one element, chunks
    with remainders."""
    m = max(1, n // 3)
    sets = [[_iid(k, n, n) for k in (1, 2, 3, 6, 41)], [_iid(k, n, m, "C") for k in (-(-n // m) + 1, 30)],
            [_iid(9, n, m, "w", None)]]
    if n > 1:
        pr = P.random_problem(1500 + n, 11, n, n, K_kind="W", C_kind="w", H_kind="R", unobserved=(2, 10))
        got = dev.smooth_equations(pr, "associative")
        ok, what = assoc_parity(got, oracle.associative(pr), oracle.oddeven(pr), tol=TOL)
        assert ok, (pr.name, what)
    for probs in sets:
        b = dev.Batch(probs)
        try:
            for _ in range(2):  # the first makes the plan, the second finds it
                b.smooth("associative")
                for i, pr in enumerate(probs):
                    x, S = b.download(i)
                    ok, what = assoc_parity((list(x), list(S)), oracle.associative(pr), oracle.oddeven(pr), tol=TOL)
                    assert ok, (pr.name, what)
        finally:
            b.free()


@pytest.mark.parametrize("n", [12, 24, 48, 60])
def test_associative_ill_conditioned_noise(dev, n):
    rng = P.rng_for(1600 + n)
    U = P.random_orthogonal(rng, n)
    Q = (U * np.logspace(0, -8, n)) @ U.T
    pr = P.uniform_problem(300, n, n // 2, seed=1601, F=0.99 * P.random_orthogonal(rng, n), Cvar=0.01,
                           G_fn=lambda r, i: r.standard_normal((n // 2, n)) / np.sqrt(n), unobserved=lambda i: i % 3 == 2)
    pr.K = [None] + [(Q + Q.T) / 2] * (pr.k - 1)
    pr.K_type = [None] + ["C"] * (pr.k - 1)
    xa, Sa = dev.smooth_equations(pr, "associative")
    xo, So = dev.smooth_equations(pr, "oddeven")
    assert max_rel_err(xa, xo) < 1.4e-6 and max_rel_err(Sa, So) < 1.4e-6


@pytest.mark.parametrize("dims", [(3,), (3, 16), (2, 5, 17, 33), (1, 4, 8, 12, 20, 48)])
def test_lanes(dev, dims):
    probs = [_iid(k, n, n) for n in dims for k in (5, 130 + n)]
    whole, alone = dev.Batch(probs), [dev.Batch(probs[2 * i:2 * i + 2]) for i in range(len(dims))]
    try:
        for run in (lambda b: b.smooth("oddeven"), lambda b: b.smooth("associative"), lambda b: b.smooth_mixed_opt(1, 0, True)):
            for b in [whole] + alone:
                run(b)
            for i in range(len(probs)):
                (x, S), (y, T) = whole.download(i), alone[i // 2].download(i % 2)
                assert np.array_equal(x, y) and np.array_equal(S, T), probs[i].name
    finally:
        for b in [whole] + alone:
            b.free()


def test_associative_refusal_in_a_lane(dev):
    """A part whose observations do not determine its states is refused, and
    leaves the library in order."""
    bad = _iid(2, 9, 1)
    b = dev.Batch([_iid(60, 4, 4), bad, _iid(60, 17, 17)])
    for _ in range(2):
        with pytest.raises(dev.UkhipError, match="do not determine"):
            b.smooth("associative")
    b.free()
    b = dev.Batch([_iid(60, 4, 4), _iid(60, 17, 17)])
    b.smooth("associative")
    assert np.all(np.isfinite(b.download(0)[0])) and np.all(np.isfinite(b.download(1)[1]))
    b.free()
