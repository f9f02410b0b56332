"""The chase's tridiagonal keeps its last bits: the digests are those of the plain
forms of its sums (butterflies by lane ^ 32 ... 1) and of its roots and quotients."""
import hashlib

import numpy as np
import pytest

from tests.helpers import to_dev, to_host

pytestmark = pytest.mark.gpu

DIGESTS = {
    (70, 32): "33e26fc63768236351c1",
    (257, 32): "f988dbd4f93720c8119e",
    (130, 64): "716c9b57a23848615b03",
    (300, 64): "52cc48436893192d15e9",
    (100, 5): "1185715ad29e20f1c1df",
    (150, 33): "268c7ef2c3d4e0327576",
}


@pytest.mark.parametrize("n,b", [(70, 32), (257, 32), (130, 64), (300, 64), (100, 5), (150, 33)])
def test_tridiagonal_bits(ctx, n, b):
    import evd4sc2025_amd as E

    band = np.random.RandomState(n + b).standard_normal((n, 2 * b))
    for c in range(n):
        band[c, min(b, n - 1 - c) + 1:] = 0.0
    D, Eo, U = E.sb2st(ctx, to_dev(band.T), n, b)
    m = hashlib.sha256()
    for x in (to_host(D), to_host(Eo), np.ascontiguousarray(to_host(U).T)):
        m.update(np.ascontiguousarray(x).tobytes())
    assert m.hexdigest()[:20] == DIGESTS[n, b]
