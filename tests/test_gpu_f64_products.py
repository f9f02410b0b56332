"""The FP64 band reduction's products (two operand pairs in one K loop, K
split over workgroups) at bandwidths that are no multiple of the K slab,
orders that end in partial tiles, and W, Y with leading dimensions of their
own; the FP64 SYR2K at the edges of its triangle of tiles."""
import numpy as np
import pytest

from oracle import evd_oracle as O
from tests.helpers import to_dev, to_host

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,b,nb,pad", [(130, 8, 32, 0), (257, 24, 96, 0), (257, 24, 96, 3), (500, 33, 66, 0),
                                        (300, 64, 64, 5), (66, 64, 64, 0), (700, 32, 32, 1), (1100, 32, 256, 0)])
def test_sy2sb_f64_shapes(ctx, n, b, nb, pad):
    import evd4sc2025_amd as E

    A = O.gen_symmetric(n, n + b, 0).astype(np.float64)
    dA = to_dev(A)
    W, Y = (E.colmajor(n + pad, n, dtype=dA.dtype)[:n] for _ in range(2))
    E.sy2sb(ctx, dA, b, nb, W, Y)
    B, W, Y = np.tril(np.triu(to_host(dA), -b)), to_host(W), to_host(Y)
    B = B + np.tril(B, -1).T
    Q = O.q_sbr(W, Y, b)
    nrm = np.linalg.norm(A, 2)
    # FP64 throughout: orthogonal similarity to rounding
    assert np.abs(Q.T @ Q - np.eye(n)).max() < 1e-13 * np.sqrt(n)
    assert np.abs(Q.T @ A @ Q - B).max() < 1e-13 * np.sqrt(n) * nrm


@pytest.mark.parametrize("n,k", [(1, 1), (63, 5), (64, 16), (65, 17), (200, 0), (129, 300)])
def test_syr2k_f64_edges(ctx, n, k):
    import evd4sc2025_amd as E

    rng = np.random.default_rng(n + k)
    A, B, C = rng.standard_normal((n, max(k, 1)))[:, :k], rng.standard_normal((n, max(k, 1)))[:, :k], rng.standard_normal((n, n))
    C = (C + C.T) / 2
    dC = to_dev(C)
    dA, dB = (to_dev(X) if k else E.colmajor(n, 1, dtype=dC.dtype)[:, :0] for X in (A, B))
    E.tc_ozimmu_syr2k(ctx, -1.5, dA, dB, 0.5, dC)
    got = to_host(dC)
    assert np.array_equal(got, got.T)
    assert np.abs(got - (-1.5 * (A @ B.T + B @ A.T) + 0.5 * C)).max() < 1e-14 * (10 + k)
