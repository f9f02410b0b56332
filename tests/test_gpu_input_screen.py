"""The input screen at the edges of its 64 x 64 tiles, in batches of more
matrices than one launch takes, and whole solves whose back transformation
merges fewer panels than the padding holds."""
import numpy as np
import pytest

from oracle import evd_oracle as O
from tests.helpers import to_dev, to_host

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [3, 63, 64, 65, 96, 129, 257, 300, 513, 1030])
def test_upper_triangle_is_not_read(ctx, n):
    import evd4sc2025_amd as E

    print(f"screen n={n}", flush=True)
    A = O.gen_symmetric(n, 11 + n)
    B = np.tril(A) + np.triu(np.full((n, n), np.nan, np.float32), 1)
    r = E.syevd(ctx, to_dev(B), b=32, nb=256)
    w = np.linalg.eigvalsh(A.astype(np.float64))
    assert np.abs(to_host(r.w) - w).max() <= 1e-5 * np.abs(w).max()
    assert E.backward_error(ctx, to_dev(A), r.w, r.Z) <= 1e-6 and E.checkOrthogonality(ctx, r.Z) <= 1e-6


@pytest.mark.parametrize("where", [(0, 0), (69, 31), (64, 70)])
def test_batch_of_seventy(ctx, where):
    import evd4sc2025_amd as E

    n, count = 71, 70
    mats = [to_dev(O.gen_symmetric(n, 500 + q)) for q in range(count)]
    w, _ = E.syevd_batched(ctx, mats, b=32, nb=64, jobz="N")
    for q in (0, 63, 64, 69):
        ref = np.linalg.eigvalsh(to_host(mats[q]).astype(np.float64))
        assert np.abs(to_host(w[q]) - ref).max() <= 1e-5 * np.abs(ref).max()
    q, c = where  # a non-finite entry of the lower triangle of any matrix is reported
    mats[q][n - 1, c] = float("inf")
    with pytest.raises(Exception):
        E.syevd_batched(ctx, mats, b=32, nb=64, jobz="N")
