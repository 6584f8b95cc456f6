"""Solves past the streaming and chain kernels: more than 64 right-hand sides,
and 33 to 64 with a front of more than 8,192 columns.

They run the fused panel steps (launch_panel_step), one product per
super-panel with K split into slices (k_reduce_slices), or two products per
panel. The environment chooses the panels per super-panel and the width of the
inverted blocks, so each choice is a process of its own. One dense front of
2,450 columns takes two super-panels and a part of a third by default, ten or
more of 256 columns, and products with K of 1,024 and more.

Tolerance: A = d + (at most four entries of modulus 1 a row), |d| >= 5, is
diagonally dominant, so ||A^-1|| <= 1 in the largest-entry norm and cond(A) <=
|d| + 4. A computed solution is within c cond(A) N u of the exact one; c = 4
covers the two triangular sweeps with explicitly inverted diagonal blocks. An
update left out or taken twice is an error of a tenth or more next to its rows.
"""
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

_RUN = r"""
import sys, numpy as np, torch
import scipy.sparse.linalg as sl
sys.path.insert(0, sys.argv[1])
import clique_amd as cq
from clique_amd import problems as P
nx, ny, widths = int(sys.argv[2]), int(sys.argv[3]), [int(k) for k in sys.argv[4].split(",")]
for kind in sys.argv[5].split(","):
    ip, ind, v, dims = P.laplacian5(nx, ny, 1.0)
    N = ip.size - 1
    row = np.repeat(np.arange(N), np.diff(ip))
    if kind == "cplx":
        v = v * np.where(row == ind, 1 + 0.3j, 0.8 + 0.6j)
    if kind == "herm":
        v = v * np.where(row == ind, 1, np.exp(1j * np.sign(ind - row) * (row + ind)))
    cplx = kind != "real"
    lu = sl.splu(P.to_scipy(ip, ind, v).tocsc())
    for prec, u in (("f64", 2.0 ** -53), ("f32", 2.0 ** -24)):
        sym = cq.NaturalNestedDissection(*dims, ip, ind, cutoff=N)
        assert sym.num_nodes == 1
        ft = cq.DistSymmFrontTree(sym, ip, ind, is_complex=cplx, conjugate=kind == "herm")
        ft.factor(torch.tensor(v, device="cuda:0"), precision=prec)
        rng = np.random.default_rng(N)
        for k in widths:
            b = rng.standard_normal((N, k)) + (1j * rng.standard_normal((N, k)) if cplx else 0)
            x = cq.colmajor(torch.tensor(b, device="cuda:0"))
            ft.set_profiling(True)
            ft.solve(x)
            fams = ",".join(sorted(ft.profile()))
            ft.set_profiling(False)
            want = lu.solve(b)
            err = (np.abs(x.cpu().numpy() - want).max(axis=0) / np.abs(want).max(axis=0)).max()
            bound = 4 * (np.abs(v).max() + 4) * N * u
            print("CASE", kind, prec, k, "%.3e" % err, "%.3e" % bound, fams, flush=True)
        del ft
"""


@pytest.mark.gpu
@pytest.mark.parametrize("nx,ny,widths,kinds,env,has,lacks", [
    (50, 49, "65,70,130", "real,cplx,herm", {}, ["solve_panel", "solve_reduce"], ["solve_chain"]),
    (50, 49, "65", "real,cplx", {"CLIQG_SPLIT_TILES": "0"}, ["solve_panel"],
     ["solve_chain", "solve_reduce"]),
    (50, 49, "65", "cplx,herm", {"CLIQG_SOLVE_CHAIN": "2"}, ["solve_panel"], ["solve_chain"]),
    (50, 49, "96", "real,herm", {"CLIQG_SOLVE_CHAIN": "3", "CLIQG_SOLVE_BLOCK": "64"},
     ["solve_panel"], ["solve_chain"]),
    (50, 49, "65", "real,cplx", {"CLIQG_SOLVE_CHAIN": "0"}, [], ["solve_chain", "solve_panel"]),
    (92, 90, "33,64", "real", {}, ["solve_panel"], ["solve_chain"]),
    (92, 90, "32", "real", {}, ["solve_chain"], ["solve_panel"])])
def test_wide_solves(device, nx, ny, widths, kinds, env, has, lacks):
    clean = {k: x for k, x in os.environ.items() if not k.startswith("CLIQG_")}
    r = subprocess.run([sys.executable, "-c", _RUN, ROOT, str(nx), str(ny), widths, kinds],
                       env=dict(clean, **env), capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-2000:]
    cases = [t.split() for t in r.stdout.splitlines() if t.startswith("CASE")]
    assert len(cases) == 2 * len(widths.split(",")) * len(kinds.split(","))
    for _, kind, prec, k, err, bound, fams in cases:
        print(kind, prec, k, err, bound, fams)
        assert float(err) <= float(bound), (kind, prec, k)
        for name in has:
            assert name in fams.split(","), (kind, prec, k, name, fams)
        for name in lacks:
            assert name not in fams.split(","), (kind, prec, k, name, fams)
