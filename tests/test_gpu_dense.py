"""The dense exact solve of the bottom level against the oracle: one application of
the preconditioner whose V-cycle ends in it, at bottoms of every form the inversion
takes (one workgroup up to 64 cells, 32-column tiles above, with and without
padding; axes of one to nine cells).

Bound: the inverse of an n-cell operator of condition number kappa is exact to
about kappa * eps * sqrt(n); with at most 9 cells an axis and coefficients within a
factor 20, kappa is below 20 * (2 * 9 / pi)^2 * 3 = 2000, so 2000 * 2.2e-16 *
sqrt(512) = 1e-11."""
import numpy as np
import pytest

import tbfsolver_amd as T
from tbfsolver_amd import fields as F
from oracle import pyoracle as O
from conftest import to_dev, to_host

pytestmark = pytest.mark.gpu


def setup(n, stretch, seed=5):
    g, go = T.channel_grid(n, stretch_y=stretch, gamma=1.5), O.desc(n, stretch=(0, stretch, 0), gamma=1.5)
    rho, _ = F.make_bubble_density(g, 4, 0.3, seed, nref=4)
    q = O.divergence(go, *F.make_velocity(g, seed))
    return g, go, q, O.beta_from_rho(go, 1e-3, rho)


def rel(a, b):
    a, b = a - a.mean(), b - b.mean()
    return np.linalg.norm(a - b) / np.linalg.norm(b)


@pytest.mark.parametrize("n,stretch,bottom", [((8, 4, 2), 0, 8), ((24, 24, 24), 0, 27), ((32, 32, 32), 1, 64),
                                              ((20, 12, 12), 1, 45), ((12, 20, 44), 0, 165), ((16, 32, 18), 1, 1152),
                                              ((20, 20, 20), 0, 125), ((56, 64, 72), 1, 504), ((72, 40, 56), 1, 315)])
def test_dense_bottom_matches_oracle(torch_gpu, n, stretch, bottom):
    print("case dense bottom", n, bottom, flush=True)
    g, go, q, beta = setup(n, stretch)
    kw = dict(nLevels=2, precision="fp64", coarse_max_iter=0)
    if bottom > 512:
        with pytest.raises(T.TbfgError):
            T.PCG(g, **kw)
        return
    zr = O.mg_apply(go, O.params(n_levels=2, coarse_mode=1, coarse_cycles=1), beta, q)
    s = T.PCG(g, **kw)
    z = torch_gpu.zeros_like(to_dev(q, torch_gpu))
    s.precondition(to_dev(beta, torch_gpu), to_dev(q, torch_gpu), z)
    torch_gpu.cuda.synchronize()
    s.close()
    e = rel(to_host(z), zr)
    print("  rel error", e, flush=True)
    assert e < 1e-11


@pytest.mark.parametrize("n,nlev,cells", [((48, 32, 48), 4, 144), ((48, 40, 48), 3, 1440), ((128, 64, 128), 4, 2048)])
def test_direct_coarsest_solve_matches_inner_cg(torch_gpu, monkeypatch, n, nlev, cells):
    """The reference algorithm with its coarsest level solved by the dense inverse and by
    the inner CG (TBFG_INNER_IN_TAIL): the same outer iterations within one, pressures to
    1e-12 residual equal to 1e-10; a looser coarse_tol or fewer iterations keep the CG."""
    print("case direct coarsest", n, cells, flush=True)
    g, go, q, beta = setup(n, 1)
    b, r = to_dev(beta, torch_gpu), to_dev(q, torch_gpu)

    def solve(**kw):
        s = T.PCG(g, nLevels=nlev, tolPCG=1e-12, maxIterPCG=200, flexible=1, **kw)
        psi = torch_gpu.zeros_like(r)
        s.solvePCG(psi, b, r)
        out = (s.iterations, s.coarse_stats(), to_host(psi))
        assert s.converged
        s.close()
        return out

    it, cs, psi = solve()
    assert cs["calls"] >= it and cs["iters_max"] == 1 and cs["iters"] == cs["calls"] and cs["res_max"] <= 1e-10
    assert solve(coarse_tol=1e-3)[1]["iters_max"] > 1
    assert solve(coarse_max_iter=39)[1]["iters_max"] > 1
    monkeypatch.setenv("TBFG_INNER_IN_TAIL", "1")
    it_cg, cs_cg, psi_cg = solve()
    print("  iterations", it, it_cg, cs, cs_cg, flush=True)
    assert cs_cg["iters_max"] > 1 and abs(it - it_cg) <= 1
    assert rel(psi, psi_cg) < 1e-10


@pytest.mark.parametrize("kw", [dict(), dict(mg_cycles=2), dict(unfused=True)], ids=["fused", "two cycles", "unfused"])
def test_direct_coarsest_diagnostics_counted_once_per_solve(torch_gpu, monkeypatch, kw):
    """The diagnostics of the dense coarsest solves, formed beside the dot products or by a launch of their
    own: one call and one iteration per V-cycle, each to round-off."""
    kw = dict(kw)
    if kw.pop("unfused", False):
        monkeypatch.setenv("TBFG_UNFUSED_DOTS", "1")
    print("case direct diagnostics", kw, flush=True)
    g, go, q, beta = setup((48, 32, 48), 1)
    s = T.PCG(g, nLevels=3, tolPCG=1e-10, maxIterPCG=200, flexible=1, **kw)
    psi = torch_gpu.zeros(48, 32, 48, dtype=torch_gpu.float64, device="cuda")
    s.solvePCG(psi, to_dev(beta, torch_gpu), to_dev(q, torch_gpu))
    cs, it = s.coarse_stats(), s.iterations
    s.close()
    # (an application follows every update but the last, plus the first)
    assert cs["calls"] == it * kw.get("mg_cycles", 1), (cs, it)
    assert cs["iters"] == cs["calls"] and cs["iters_max"] == 1 and cs["res_max"] <= 1e-10
