"""Rank-deficient panels, which the column-exchange kernel factors: panels of one
workgroup with one and two rows per thread, of several that work together or of
which one works alone (as where the others find no room), and batches in which
only some of the problems need it, against single solves and LAPACK."""
import numpy as np
import pytest

from tests.helpers import to_dev, to_host

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m", [64, 200, 256, 257, 512, 513])
def test_rank_deficient_single_panels(ctx, m):
    import evd4sc2025_amd as E

    b = 32
    P = np.random.default_rng(m).standard_normal((m, b)).astype(np.float32)
    P[:, 9] = P[:, 4]
    P[:, 30] = 0.0
    dA, dW, dR = to_dev(P), E.colmajor(m, b, fill=0.0), E.colmajor(b, b, fill=0.0)
    E.panelQR(ctx, dA, dW, dR)
    Y, W, R = (to_host(x).astype(np.float64) for x in (dA, dW, dR))
    Y = np.tril(Y, -1) + np.eye(m, b)
    Rf = np.zeros((m, b))
    Rf[:b] = np.triu(R)
    # the sums of the factorisation have m terms, those of its products b
    tol = 4 * b * np.finfo(np.float32).eps * np.sqrt(m) * np.abs(P).max()
    assert np.abs(Rf - W @ (Y.T @ Rf) - P).max() < tol
    Qt = np.eye(m, b) - W @ Y[:b].T
    assert np.abs(Qt.T @ Qt - np.eye(b)).max() < tol


@pytest.mark.parametrize("n", [200, 1100])
def test_batches_with_some_panels_rank_deficient(ctx, n):
    import torch

    import evd4sc2025_amd as E

    rng = np.random.default_rng(n)
    mats = []
    for q in range(4):
        X = rng.standard_normal((n, n if q % 2 else 5))
        A = (X @ X.T if q % 2 == 0 else (X + X.T) / 2).astype(np.float32)
        mats.append(to_dev((A + A.T) / 2))
    w, Z = E.syevd_batched(ctx, mats, b=32, nb=256)
    for q in range(4):
        r = E.syevd(ctx, mats[q], b=32, nb=256)
        assert torch.equal(w[q], r.w) and torch.equal(Z[q], r.Z), q
        ref = np.linalg.eigvalsh(to_host(mats[q]).astype(np.float64))
        assert np.abs(to_host(w[q]) - ref).max() < 1e-5 * np.abs(ref).max()
        Zq = to_host(Z[q]).astype(np.float64)
        assert np.linalg.norm(Zq.T @ Zq - np.eye(n)) / n < 1e-6


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("m,b", [(257, 32), (513, 32), (700, 17), (4096, 32), (16384, 31), (17000, 32)])
def test_one_group_alone_equals_the_groups_together(ctx, m, b, dtype):
    import torch

    import evd4sc2025_amd as E

    print(f"panel alone m={m} b={b} {dtype.__name__}", flush=True)
    P = np.random.default_rng(m + b).standard_normal((m, b)).astype(dtype)
    P[:, b // 2] = P[:, 1]
    P[:, b - 1] = 0.0
    tt = torch.float32 if dtype == np.float32 else torch.float64
    out = []
    for alone in (0, 1, 0):
        dA, dW, dR = to_dev(P), E.colmajor(m, b, dtype=tt, fill=0.0), E.colmajor(b, b, dtype=tt, fill=0.0)
        ctx.set_knob("panel_alone", alone)
        try:
            E.panelQR(ctx, dA, dW, dR)
        finally:
            ctx.set_knob("panel_alone", 0)
        torch.cuda.synchronize()
        out.append((dA, dW, dR))
    for x in out[1:]:
        assert all(torch.equal(a, b) for a, b in zip(out[0], x))


def test_solves_with_one_group_alone_equal_the_others(ctx):
    import torch

    import evd4sc2025_amd as E

    n = 1500
    X = np.random.default_rng(5).standard_normal((n, 40)).astype(np.float32)
    mats = [to_dev(X @ X.T), to_dev((X @ X.T)[::-1, ::-1])]
    ref = E.syevd(ctx, mats[0], b=32, nb=256)
    w, Z = E.syevd_batched(ctx, mats, b=32, nb=256)
    ctx.set_knob("panel_alone", 1)
    try:
        r = E.syevd(ctx, mats[0], b=32, nb=256)
        wa, Za = E.syevd_batched(ctx, mats, b=32, nb=256)
    finally:
        ctx.set_knob("panel_alone", 0)
    assert torch.equal(ref.w, r.w) and torch.equal(ref.Z, r.Z)
    assert torch.equal(w, wa) and torch.equal(Z, Za)
