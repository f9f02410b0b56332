"""The WY back transformation at every workgroup width (64, 32 and 16 columns,
chosen by the number of columns): a column's result does not depend on how
many columns are transformed with it, and agrees with the oracle."""
import numpy as np
import pytest

from oracle import evd_oracle as O
from tests.helpers import to_dev, to_host

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,b,precision", [(130, 32, 0), (97, 32, 2), (200, 64, 0)])
def test_widths_agree(n, b, precision):
    import torch

    import evd4sc2025_amd as E

    A = O.gen_symmetric(n, n).astype(np.float64)
    U = O.sb2st(np.tril(np.triu(A, -b), b), b)[2].astype(np.float32)
    rng = np.random.default_rng(n)
    cols = 8203  # 129 workgroups of 64 columns, the last of 11
    X = (rng.standard_normal((n, cols)) / np.sqrt(n)).astype(np.float32)
    with E.Context(0) as ctx:
        ctx.set_precision(precision)
        dU = to_dev(U)
        whole = to_dev(X)
        E.bc_back(ctx, whole, dU, n, b, 1)
        for c0, c1 in [(0, 1), (0, 15), (3, 20), (0, 33), (8000, 8203), (0, 5000), (100, 8200)]:
            part = to_dev(X[:, c0:c1])
            E.bc_back(ctx, part, dU, n, b, 1)
            assert torch.equal(part, whole[:, c0:c1]), (c0, c1)
    want = O.bc_back(X[:, :64].astype(np.float64), U.astype(np.float64), n, b, 1)
    # FP32 products over n reflectors of unit columns (split FP16 keeps 22 bits)
    assert np.abs(to_host(whole[:, :64]) - want).max() < 2e-6 * np.sqrt(n)
