"""The bulge chase over XCDs: runs of sweeps on one XCD, on several, batches
that take several launches, and single chases too large for the XCDs' boxes.
However the sweeps are handed out, each problem's arithmetic is the same, so a
batch equals its problems chased one by one, and a chase with boxes equals the
one without (the form without allocation never has any), bit for bit."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _bands(count, n, b):
    import torch

    gen = torch.Generator(device="cuda")
    gen.manual_seed(n + b)
    band = torch.randn(count, n, 2 * b, generator=gen, device="cuda", dtype=torch.float64)
    off = torch.arange(2 * b, device="cuda").view(1, 1, -1)
    return band * ((off <= b) & (off + torch.arange(n, device="cuda").view(1, -1, 1) < n))


@pytest.mark.parametrize("count,n,b", [(2, 100, 32), (36, 200, 32), (37, 200, 32), (80, 200, 32), (20, 900, 32), (50, 96, 24),
                                       (40, 400, 64)])
def test_batches_equal_singles(ctx, count, n, b):
    import torch

    import evd4sc2025_amd as E

    print(f"chase batch count={count} n={n} b={b}", flush=True)
    band = _bands(count, n, b)
    own = band.clone()
    U = torch.empty(count, n, n + b, device="cuda")
    D, Eo = (torch.empty(count, n, device="cuda", dtype=torch.float64) for _ in range(2))
    ctx.call("evd_sb2st_batched_f64", count, n, b, C.c_void_p(own.data_ptr()), 2 * b, 2 * b * n, C.c_void_p(U.data_ptr()),
             n + b, (n + b) * n, C.c_void_p(D.data_ptr()), n, C.c_void_p(Eo.data_ptr()), n)
    for q in sorted({0, 1, count // 2, count - 1}):
        d, e, u = E.sb2st(ctx, band[q].clone().t(), n, b)
        assert torch.equal(d, D[q]) and torch.equal(e, Eo[q, :n - 1]) and torch.equal(u.t(), U[q])


@pytest.mark.parametrize("n,b", [(1000, 32), (3001, 32), (2100, 64)])
def test_boxes_change_nothing(ctx, n, b):
    import torch

    import evd4sc2025_amd as E

    print(f"chase n={n} b={b}", flush=True)
    band = _bands(1, n, b)[0]
    with_boxes = E.sb2st(ctx, band.clone().t(), n, b)
    without = E.sb2st(ctx, band.clone().t(), n, b, noalloc=True)
    assert all(torch.equal(x, y) for x, y in zip(with_boxes, without))
