"""FP32 updates keep FP32's accuracy entry by entry, also in rows of wide range.

Two dense fronts (1,024 and 128 columns, unit D, no coupling inside) under a
dense one of 1,792: its entries are S - L L^T with known L. Every row of L has
one entry of size 1 and all others 2^-34 of it, so off the few places where
two large entries meet, a sum consists of terms 2^-34 below the product of its
rows' largest entries.

Tolerance: an FP32 sum of K products in any order is within (K + 2) u
sum |w| |l| of the exact one, u = 2^-24 (Higham, ch. 3). A complex product
by three real ones (Gauss) forms its parts from P1, P2 and P3 with operands of
up to sqrt(2) times the moduli: |Re| errs by at most 1 and |Im| by 3 times
that, sqrt(10) < 4 together. Fourteen roundings more cover the division by
the pivot and the way through the fronts.
"""
import numpy as np
import pytest

import clique_amd as cq
from clique_amd.problems import stencil7

torch = pytest.importorskip("torch")
U32 = 2.0 ** -24


def two_fronts(kind, nA=1024, nB=128, nS=1792):
    """CSR pattern and values: A and B coupled to S only, A's coupling of wide range."""
    rng = np.random.default_rng(17)
    herm, cplx = kind == "herm", kind != "real"
    g = rng.uniform(1, 2, (nS, nA)).astype(np.float32) * 2.0 ** -34
    if cplx:
        g = (g * np.exp(1j * rng.uniform(0, 2 * np.pi, g.shape))).astype(np.complex64)
    g = g.astype(np.complex128 if cplx else np.float64)
    g[np.arange(nS), np.arange(nS) % nA] = 1.0
    cA, cB = np.r_[0:nA, nA + nB:nA + nB + nS], np.arange(nA, nA + nB + nS)
    N = nA + nB + nS
    ip = np.zeros(N + 1, np.int64)
    np.cumsum(np.repeat([cA.size, cB.size, N], [nA, nB, nS]), out=ip[1:])
    ind = np.concatenate([np.tile(cA, nA), np.tile(cB, nB), np.tile(np.arange(N), nS)])
    top = np.concatenate([np.eye(nA), (g.conj() if herm else g).T], axis=1)
    mid = np.concatenate([np.eye(nB), np.zeros((nB, nS))], axis=1)
    low = np.concatenate([g, np.zeros((nS, nB)), 4.0 * np.eye(nS)], axis=1)
    return ip, ind.astype(np.int32), np.concatenate([top.ravel(), mid.ravel(), low.ravel()])


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["real", "complex", "herm"])
def test_fp32_updates_entry_by_entry(device, kind):
    ip, ind, v = two_fronts(kind)
    sym = cq.NestedDissection(ip, ind, cutoff=1024)
    sizes = [sym.node(s)["size"] for s in range(sym.num_nodes)]
    assert sorted(sizes) == [128, 1024, 1792] and sizes[-1] == 1792, sizes
    ft = cq.DistSymmFrontTree(sym, ip, ind, is_complex=kind != "real", conjugate=kind == "herm")
    vals = torch.tensor(v, device=device)
    ft.factor(vals, precision="f32")
    L32 = ft.front(sym.num_nodes - 1)[0][:, 0]
    ft.factor(vals)
    L64, d64 = ft.front(sym.num_nodes - 1)
    w = np.abs(ft.front(sizes.index(1024))[0][1024:])   # rows in the order of the front above
    scale = w @ w[0] / abs(d64[0])
    err = np.abs(L32 - L64[:, 0])[1:] / scale[1:]
    bound = (1 if kind == "real" else 4) * (1024 + 16) * U32
    print(f"{kind}: largest error {err.max():.2e} of sum |w l|, bound {bound:.2e}")
    assert err.max() <= bound, (err.max(), bound)


@pytest.mark.gpu
def test_fp32_far_field(device):
    """A point source in a screened Laplacian, 64^3, one FP32 solve.

    The solution falls by 10^-30 across the grid. A is an M-matrix and the
    source positive: L <= 0 off its diagonal, the inverted blocks >= 0, and
    neither the factorization nor the sweeps subtract anything but in the
    pivots (FP64 inside a block), so each entry keeps its digits. With sums of at
    most m_s terms at every front s of a path to the root, in the factor and in
    either sweep, and as many again from the pivots, it is within 4 u sum m_s
    of the exact one; 8 leaves room for the inverted blocks.
    """
    n = 64
    ip, ind, v, dims = stencil7(n, n, n, 6.3, -1.0)
    N = ip.size - 1
    sym = cq.NaturalNestedDissection(*dims, ip, ind, cutoff=128)
    nodes = [sym.node(s) for s in range(sym.num_nodes)]
    path = [0] * sym.num_nodes
    for s in range(sym.num_nodes - 1, -1, -1):
        path[s] = nodes[s]["size"] + nodes[s]["lower_size"]
        if nodes[s]["parent"] >= 0:
            path[s] += path[nodes[s]["parent"]]
    ft = cq.DistSymmFrontTree(sym, ip, ind)
    vals = torch.tensor(v, device=device)
    x = {}
    for prec in ("f32", "f64"):
        ft.factor(vals, precision=prec)
        b = torch.zeros((2, N), dtype=torch.float64, device=device).t()
        b[0, 0] = b[N // 2 + n // 2, 1] = 1.0
        x[prec] = ft.solve(b).cpu().numpy()
    err = np.abs(x["f32"] / x["f64"] - 1).max()
    bound = 8 * max(path) * U32
    print(f"largest relative error of an entry {err:.2e}, bound {bound:.2e}")
    assert x["f64"].min() > 0 and err <= bound, (err, bound)
