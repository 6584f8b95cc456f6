"""The plan's product is finished when the call returns.

A plan made while PyTorch's default stream is current has a stream of its
own, and side streams do not wait for either: what reads y or overwrites x
there right after the call must meet a finished product. The product takes
several times as long as the copies that follow take to reach the device, and
y holds NaN before it. x holds integers below 2^20 and A is scaled to integers,
so that every sum is exact and the comparison is of equal values.
"""
import numpy as np
import pytest

import clique_amd as cq
from clique_amd import problems as P

torch = pytest.importorskip("torch")


@pytest.mark.gpu
@pytest.mark.parametrize("own", [True, False])
def test_product_is_finished_on_return(device, own):
    k = 64
    ip, ind, v, dims = P.stencil7(61, 58, 63, 7.0, -1.0)
    N = ip.size - 1
    sym = cq.NaturalNestedDissection(*dims, ip, ind, cutoff=128)
    side = torch.cuda.Stream()
    with torch.cuda.stream(torch.cuda.default_stream() if own else torch.cuda.Stream()):
        ft = cq.DistSymmFrontTree(sym, ip, ind)
        ft.factor(torch.tensor(v, device=device), precision="f32")
    x0 = np.random.default_rng(8).integers(-2 ** 20, 2 ** 20, (N, k)).astype(np.float64)
    want = P.to_scipy(ip, ind, v) @ x0
    src = cq.colmajor(torch.tensor(x0, device=device))
    x, y = torch.empty_like(src), torch.empty_like(src)
    for _ in range(5):
        x.copy_(src)
        y.fill_(float("nan"))
        torch.cuda.synchronize()
        ft.multiply(x, y)
        with torch.cuda.stream(side):
            seen = y.clone()
            x.zero_()
        torch.cuda.synchronize()
        assert np.array_equal(seen.cpu().numpy(), want)
        assert np.array_equal(y.cpu().numpy(), want)


@pytest.mark.gpu
@pytest.mark.skipif(torch.cuda.device_count() < 2, reason="needs two devices")
def test_product_is_refused_on_another_device(device):
    """A plan with its own stream runs its products on the default stream of
    the current device, which has to be the plan's."""
    ip, ind, v, dims = P.stencil7(9, 8, 7, 7.0, -1.0)
    sym = cq.NaturalNestedDissection(*dims, ip, ind, cutoff=32)
    ft = cq.DistSymmFrontTree(sym, ip, ind)
    ft.factor(torch.tensor(v, device=device))
    x = torch.ones(ip.size - 1, dtype=torch.float64, device=device)
    y = torch.zeros_like(x)
    with torch.cuda.device(1), pytest.raises(Exception, match="device current"):
        ft.multiply(x, y)
