"""Eigenvector signs of the tridiagonal solver follow from its merges down to single
rows (as the model's do), its vectors are orthogonal on entries of any spread, and
problems of a batch equal their single solves."""
import numpy as np
import pytest

from tests.helpers import to_dev, to_host
from tests.stedc_model import stedc, tridiagonal

pytestmark = pytest.mark.gpu


# orders of one leaf (its sizes and uneven halves), of leaves below one and several merges
@pytest.mark.parametrize("n", [2, 3, 5, 9, 15, 16, 17, 33, 64, 130])
@pytest.mark.parametrize("kind", ["gaussian", "decoupled", "weak"])
def test_signs_are_those_of_the_merges(ctx, kind, n):
    import evd4sc2025_amd as E

    for seed in range(4):
        d, e = tridiagonal(kind, n, np.random.default_rng(1000 * n + seed))
        wm, Zm = stedc(d, e)
        w, Z = (to_host(x) for x in E.stedc(ctx, to_dev(d), to_dev(e)))
        assert np.abs(w - wm).max() <= 1e-13 * np.abs(wm).max() * np.sqrt(n)
        # a vector's error is that of the matrix over its gap
        gap = np.diff(wm, prepend=-np.inf, append=np.inf)
        gap = np.minimum(gap[:-1], gap[1:])
        clear = gap > 1e-6 * np.abs(wm).max()
        dots = np.sum(Z * Zm, axis=0)
        assert clear.sum() >= n // 2
        assert np.all(dots[clear] > 0.999), (seed, np.flatnonzero(clear & (dots <= 0.999)))


@pytest.mark.parametrize("n", [8, 13, 16, 24, 100])
def test_vectors_orthogonal_over_300_decades(ctx, n):
    import evd4sc2025_amd as E

    for seed in range(40):
        d, e = tridiagonal("decades", n, np.random.default_rng(77 * n + seed))
        w, Z = (to_host(x) for x in E.stedc(ctx, to_dev(d), to_dev(e)))
        assert np.abs(Z.T @ Z - np.eye(n)).max() <= 1e-14 * np.sqrt(n), seed
        T = np.diag(d) + np.diag(e, 1) + np.diag(e, -1)
        assert np.abs(T @ Z - Z * w).max() <= 1e-13 * np.sqrt(n) * np.abs(T).max(), seed


def test_batches_equal_single_solves_over_seeds(ctx):
    import torch

    import evd4sc2025_amd as E

    for seed in range(6):
        g = torch.Generator(device="cuda")
        g.manual_seed(seed)
        mats = []
        for _ in range(32):
            x = torch.randn(256, 256, generator=g, device="cuda")
            mats.append(((x + x.t()) / 2).t())
        w, Z = E.syevd_batched(ctx, mats, b=32, nb=256)
        w2, Z2 = E.syevd_batched(ctx, mats, b=32, nb=256)
        assert torch.equal(w, w2) and torch.equal(Z, Z2), seed
        for q in range(0, 32, 5):
            r = E.syevd(ctx, mats[q], b=32, nb=256)
            assert torch.equal(w[q], r.w) and torch.equal(Z[q], r.Z), (seed, q)
