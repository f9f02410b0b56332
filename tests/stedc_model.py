"""The divide and conquer of a symmetric tridiagonal matrix (Cuppen's method with
LAPACK dlaed2's deflation) down to single rows, in numpy: a reference for the signs
of the eigenvectors, which LAPACK's drivers with other leaves do not give.

At every merge a vector that is not deflated has v^T x < 0 with v = [last row of
the first child; sign(e) first row of the second]; a deflated one keeps its
child's sign; a single row is [1]."""
import numpy as np

EPS = np.finfo(np.float64).eps / 2


def _secular(d, z, rho):
    """Roots of 1 + rho sum z_k^2 / (d_k - lambda) as (origin pole, offset from it)."""
    K = len(d)
    org, off = np.zeros(K, int), np.zeros(K)
    for i in range(K):
        if i < K - 1:
            gap = d[i + 1] - d[i]
            f = 1.0 + rho * np.sum(z * z / ((d - d[i]) - gap / 2))
            org[i], lo, hi = (i, 0.0, gap / 2) if f >= 0 else (i + 1, -gap / 2, 0.0)
        else:
            org[i], lo, hi = i, 0.0, rho * np.sum(z * z)
        for _ in range(300):
            mid = 0.5 * (lo + hi)
            if mid in (lo, hi):
                break
            if 1.0 + rho * np.sum(z * z / ((d - d[org[i]]) - mid)) < 0:
                lo = mid
            else:
                hi = mid
        off[i] = 0.5 * (lo + hi)
    return org, off


def _solve(d, e):
    n = len(d)
    if n == 1:
        return d.copy(), np.ones((1, 1))
    m = n // 2
    w1, V1 = _solve(d[:m], e[:m - 1])
    w2, V2 = _solve(d[m:], e[m:])
    V = np.zeros((n, n))
    V[:m, :m], V[m:, m:] = V1, V2
    sgn = 1.0 if e[m - 1] >= 0 else -1.0
    rho = 2.0 * abs(e[m - 1])
    w = np.concatenate([w1, w2])
    z = np.concatenate([V1[-1], sgn * V2[0]]) / np.sqrt(2.0)
    at = np.argsort(w, kind="stable")
    w, z, V = w[at], z[at], V[:, at]
    tol = 8.0 * EPS * max(np.abs(w).max(), np.abs(z).max())
    keep = [j for j in range(n) if rho * np.abs(z).max() > tol and rho * abs(z[j]) > tol]
    nd, p = [], None
    for j in keep:
        if p is not None:
            t = np.hypot(z[j], z[p])
            c, s = z[j] / t, -z[p] / t
            if abs((w[j] - w[p]) * c * s) <= tol:
                z[j], z[p] = t, 0.0
                V[:, [p, j]] = np.stack([c * V[:, p] + s * V[:, j], c * V[:, j] - s * V[:, p]], axis=1)
                w[p], w[j] = w[p] * c * c + w[j] * s * s, w[p] * s * s + w[j] * c * c
            else:
                nd.append(p)
        p = j
    if p is not None:
        nd.append(p)
    if nd:
        dk, zk = w[nd], z[nd]
        org, off = _secular(dk, zk, rho)
        lam_minus = (dk[org][None, :] - dk[:, None]) + off[None, :]  # [j, i] = lambda_i - d_j
        zhat = np.empty(len(nd))
        for j in range(len(nd)):
            rest = np.arange(len(nd)) != j
            zhat[j] = np.sqrt(abs(lam_minus[j, j] / rho * np.prod(lam_minus[j, rest] / (dk[rest] - dk[j]))))
        X = -np.copysign(zhat, zk)[:, None] / lam_minus
        V[:, nd] = V[:, nd] @ (X / np.linalg.norm(X, axis=0))
        w[nd] = dk[org] + off
    at = np.argsort(w, kind="stable")
    return w[at], V[:, at]


def stedc(d, e):
    """(w, Z) of the tridiagonal (d, e)."""
    d, e = np.array(d, np.float64), np.array(e, np.float64)
    s = max(np.abs(d).max(), np.abs(e).max() if len(e) else 0.0)
    if s == 0.0:
        return d, np.eye(len(d))
    d, e = d / s, e / s
    d[:-1] -= np.abs(e)
    d[1:] -= np.abs(e)
    w, Z = _solve(d, e)
    return w * s, Z


def tridiagonal(kind, n, rng):
    """(d, e) of order n: 'gaussian' as from a dense Gaussian matrix, 'decoupled' with
    couplings of zero among the others, 'weak' with couplings of 1e-15, 'decades' with
    entries spread over 300 decades."""
    if kind == "decades":
        return tuple(10.0 ** rng.uniform(-300, 0, k) * rng.choice([-1.0, 1.0], k) for k in (n, n - 1))
    d, e = rng.standard_normal(n), np.sqrt(rng.chisquare(np.arange(n - 1, 0, -1)) / 2)
    if kind != "gaussian":
        e *= rng.choice([-1.0, 1.0], n - 1)
        e[rng.random(n - 1) < 0.4] *= 0.0 if kind == "decoupled" else 1e-15
    return d, e
