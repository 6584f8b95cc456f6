"""The allocation-free solve at the edge of its scratch array.

20,538 small fronts and 16 right-hand sides: 126.4 MiB of vectors, workspace
and launch descriptors for a scratch array of 128. The descriptors take 7 of
them, and tile arrays kept for every tile shape by itself took 48 KB more than
there was.
"""
import ctypes

import numpy as np
import pytest

import clique_amd as cq
from clique_amd import problems as P

torch = pytest.importorskip("torch")


@pytest.mark.gpu
def test_noalloc_solve_of_many_small_fronts(device):
    k, syms, ips, inds, vals, o, e = 16, [], [np.zeros(1, np.int64)], [], [], 0, 0
    for nx, ny in [(30, 29)] * 325 + [(7, 98)]:
        ip, ind, v, dims = P.laplacian5(nx, ny, 0.1)
        syms.append(cq.NaturalNestedDissection(*dims, ip, ind, cutoff=32))
        ips.append(ip[1:] + e)
        inds.append(ind + np.int32(o))
        vals.append(v)
        o, e = o + ip.size - 1, e + ind.size
    sym = cq.Symbolic.concat(syms)
    ft = cq.DistSymmFrontTree(sym, np.concatenate(ips), np.concatenate(inds))
    ft.factor(torch.tensor(np.concatenate(vals), device=device))
    b = torch.tensor(np.random.default_rng(2).standard_normal((k, o)), device=device).t()
    x = cq.colmajor(b)
    st = cq.lib().cliqg_plan_solve_noalloc(ft._h, ctypes.c_void_p(x.data_ptr()), o, k)
    assert st == 0, cq.lib().cliqg_last_error()
    assert torch.equal(x, ft.solve(cq.colmajor(b)))
