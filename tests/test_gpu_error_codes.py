"""Device-side causes come back as their own status: the tridiagonal solver on NaN (orders
of one leaf and of every way a merge is sorted) ends with no other cause than no
convergence, and a request's failure comes with its message through the server."""
import numpy as np
import pytest

from oracle import evd_oracle as O
from tests.helpers import to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2, 13, 40, 300, 700])
def test_stedc_on_nan_ends_within_its_matrices(ctx, n):
    import evd4sc2025_amd as E

    rng = np.random.default_rng(n)
    for at in (0, n // 2, n - 1):
        d, e = rng.standard_normal(n), rng.standard_normal(n - 1)
        d[at] = np.nan
        print(f"stedc NaN n={n} at={at}", flush=True)
        # a root that does not converge is reported as that; a NaN that deflates
        # away with its row is not a root
        try:
            E.stedc(ctx, to_dev(d), to_dev(e))
        except E.EvdError as ex:
            assert ex.code == 6
        # the context stays usable
        w, _ = E.stedc(ctx, to_dev(np.ones(n)), to_dev(e))
        assert np.isfinite(w.cpu().numpy()).all()


def test_server_names_the_failed_request():
    import evd4sc2025_amd as E

    A = O.gen_symmetric(64, 3, 0).copy()
    A[5, 2] = A[2, 5] = np.nan
    srv = E.Server(0, slots=1)
    try:
        good, _, _ = srv.submit(to_dev(O.gen_symmetric(96, 4, 0)), b=32, nb=32)
        bad, _, _ = srv.submit(to_dev(A), b=32, nb=32)
        assert srv.wait(good) == 0
        with pytest.raises(E.EvdError) as ei:
            srv.wait(bad)
        assert ei.value.code == 3
        assert f"request {bad}" in str(ei.value) and "order 64" in str(ei.value) and "NaN" in str(ei.value)
        with pytest.raises(E.EvdError) as ei:
            srv.wait_all()
        assert ei.value.code == 3 and "order 64" in str(ei.value)
    finally:
        srv.close()
