"""The tridiagonal solver around its leaf size and merge shapes, and the
eigenvalues-only form (which carries two rows of the vectors instead of the
vectors) against the form with vectors and LAPACK, on spectra that deflate in
every way: none, all, and long chains of rotations."""
import numpy as np
import pytest

from tests.helpers import to_dev, to_host

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2, 3, 15, 16, 17, 18, 31, 32, 33, 34, 63, 64, 65, 129, 511, 513, 1030])
def test_stedc_sizes(ctx, n):
    import evd4sc2025_amd as E

    rng = np.random.default_rng(n)
    for kind in ("random", "graded", "zero couplings"):
        d, e = rng.standard_normal(n), rng.standard_normal(n - 1)
        if kind == "graded":
            d, e = d * 10.0 ** -np.linspace(0, 12, n), e * 10.0 ** -np.linspace(0, 12, n - 1)
        if kind == "zero couplings":
            e[::3] = 0.0
        T = np.diag(d) + np.diag(e, 1) + np.diag(e, -1)
        w, Z = (to_host(x) for x in E.stedc(ctx, to_dev(d), to_dev(e)))
        nrm = np.abs(T).max()
        assert np.all(np.diff(w) >= 0)
        assert np.abs(w - np.linalg.eigvalsh(T)).max() < 1e-13 * nrm * np.sqrt(n)
        assert np.abs(T @ Z - Z * w).max() < 1e-13 * nrm * np.sqrt(n)
        assert np.abs(Z.T @ Z - np.eye(n)).max() < 1e-13 * np.sqrt(n)


def _matrix(kind, n, rng):
    X = rng.standard_normal((n, n))
    if kind == "random":
        return (X + X.T) / 2
    if kind == "diagonal":
        return np.diag(rng.standard_normal(n))
    if kind == "multiple":  # every eigenvalue many times over: long rotation chains
        m = 20
        B = rng.standard_normal((m, m))
        return np.kron(np.eye(n // m), (B + B.T) / 2)
    Q = np.linalg.qr(X)[0]
    return (Q * np.where(np.arange(n) < n // 2, 1.0, 1e-7 * np.arange(n))) @ Q.T


@pytest.mark.parametrize("kind,n", [("random", 17), ("random", 40), ("random", 600), ("diagonal", 300), ("multiple", 2000),
                                    ("clustered", 500)])
def test_values_only_equal_values_with_vectors(ctx, kind, n):
    import evd4sc2025_amd as E

    A = _matrix(kind, n, np.random.default_rng(n)).astype(np.float32)
    A = (A + A.T) / 2
    with_vectors = to_host(E.syevd(ctx, to_dev(A), nb=128, jobz="V").w)
    only = to_host(E.syevd(ctx, to_dev(A), nb=128, jobz="N").w)
    ref = np.linalg.eigvalsh(A.astype(np.float64))
    nrm = np.abs(ref).max()
    # the same tridiagonal, FP64 in both forms; the reduction to it is FP32
    assert np.abs(only - with_vectors).max() < 1e-14 * nrm * np.sqrt(n)
    assert np.abs(only - ref).max() < 1e-5 * nrm
    batch = to_host(E.syevd_batched(ctx, [to_dev(A)] * 2, nb=128, jobz="N")[0])
    assert np.array_equal(batch[0], only) and np.array_equal(batch[1], only)
