"""The two sweep kernels without LDS staging against the two half-sweep launches: one
preconditioner application at the remainders of their tiles and chunks -- rows from 16
cells to a full wavefront, several rows to a wavefront, heights and depths that leave the
last tile and chunk partly filled, axes of two cells.  The same arithmetic up to fused
multiply-adds, so the bounds of the other sweep tests (1e-13 in FP64, 1e-6 in FP32)."""
import numpy as np
import pytest

import tbfsolver_amd as T
from tbfsolver_amd import fields as F
from conftest import to_dev, to_host

pytestmark = pytest.mark.gpu


def case(torch, n, seed=9):
    g = T.channel_grid(n, stretch_y=1, gamma=1.5)
    r = np.random.default_rng(seed)
    beta = to_dev(np.exp(r.uniform(-1.5, 1.5, n)), torch)
    q = torch.zeros_like(beta)
    F.computeSource(g, *(to_dev(a, torch) for a in F.make_velocity(g, seed)), q)
    return g, beta, q


def apply(torch, g, beta, q, **kw):
    s = T.PCG(g, nLevels=2, nPreSweep=2, nPostSweep=3, coarse_max_iter=0, **kw)
    z = torch.zeros_like(q)
    s.precondition(beta, q, z)
    out = to_host(z)
    s.close()
    return out


def rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


@pytest.mark.parametrize("precision,bound", [("fp64", 1e-13), ("mixed", 1e-6)])
@pytest.mark.parametrize("n", [(16, 6, 8), (20, 10, 4), (36, 14, 6), (44, 18, 4), (100, 4, 8), (16, 62, 4), (72, 40, 56),
                               (252, 2, 4), (256, 12, 8), (128, 20, 8)])
def test_row_sweep_matches_half_sweeps(torch_gpu, monkeypatch, n, precision, bound):
    print("case row sweep", n, precision, flush=True)
    c = case(torch_gpu, n)
    monkeypatch.setenv("TBFG_SWEEP_MIN_CELLS", "0")
    a = apply(torch_gpu, *c, precision=precision)
    monkeypatch.setenv("TBFG_HALF_SWEEPS", "1")
    b = apply(torch_gpu, *c, precision=precision)
    assert np.all(np.isfinite(a)) and rel(a, b) < bound


@pytest.mark.parametrize("precision,bound", [("fp64", 1e-13), ("mixed", 1e-6)])
@pytest.mark.parametrize("n", [(2, 2, 2), (2, 6, 8), (6, 10, 4), (18, 14, 10), (34, 2, 6), (260, 4, 2), (72, 40, 56)])
def test_point_sweep_matches_half_sweeps(torch_gpu, monkeypatch, n, precision, bound):
    print("case point sweep", n, precision, flush=True)
    c = case(torch_gpu, n)
    monkeypatch.setenv("TBFG_SWEEP_MIN_CELLS", str(10 ** 12))
    a = apply(torch_gpu, *c, precision=precision)
    monkeypatch.setenv("TBFG_HALF_SWEEPS", "1")
    b = apply(torch_gpu, *c, precision=precision)
    assert np.all(np.isfinite(a)) and rel(a, b) < bound


@pytest.mark.parametrize("precision,bound", [("mixed-bf16", 1e-6), ("mixed", 1e-6), ("fp64", 1e-13)])
def test_row_sweep_matches_staged_tiles(torch_gpu, monkeypatch, precision, bound):
    """The same level by rows and by a tile shape of the staged kernel, which the shape
    switch (or an entry of the tuning table) selects, bf16 storage included."""
    n = (64, 48, 64)
    print("case row sweep vs staged tiles", precision, flush=True)
    c = case(torch_gpu, n)
    monkeypatch.setenv("TBFG_SWEEP_MIN_CELLS", "0")
    a = apply(torch_gpu, *c, precision=precision)
    monkeypatch.setenv("TBFG_SWEEP_SHAPE", "64x8x256")
    b = apply(torch_gpu, *c, precision=precision)
    assert rel(a, b) < bound


@pytest.mark.parametrize("n", [(64, 48, 64), (32, 16, 16), (256, 32, 32), (96, 48, 96)])
def test_row_sweep_rounds_as_tiles(torch_gpu, monkeypatch, n):
    """Under bf16 storage the rows give the staged kernel's bits: its preferred shape
    named (32x16 tiles for the plain sweep), against the rows that run unasked."""
    print("case rows round as tiles", n, flush=True)
    c = case(torch_gpu, n)
    monkeypatch.setenv("TBFG_SWEEP_MIN_CELLS", "0")
    a = apply(torch_gpu, *c, precision="mixed-bf16")
    monkeypatch.setenv("TBFG_SWEEP_SHAPE", "32x16x256")
    b = apply(torch_gpu, *c, precision="mixed-bf16")
    assert np.array_equal(a, b)


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("n,min_cells", [((72, 40, 56), 0), ((72, 40, 56), 10 ** 12), ((36, 12, 20), 0), ((18, 14, 10), 0)])
def test_dots_in_row_and_point_sweeps(torch_gpu, monkeypatch, n, min_cells, precision):
    """A solve with the dot products formed by the last sweep against the separate pass:
    the same iterations and, to 1e-11 residual, the same pressure to 1e-9 (the sums'
    order alone differs)."""
    print("case dots in sweeps", n, min_cells, precision, flush=True)
    g, beta, q = case(torch_gpu, n)
    monkeypatch.setenv("TBFG_SWEEP_MIN_CELLS", str(min_cells))
    out = []
    for unfused in (False, True):
        if unfused:
            monkeypatch.setenv("TBFG_UNFUSED_DOTS", "1")
        s = T.PCG(g, nLevels=2, tolPCG=1e-11, maxIterPCG=200, precision=precision, flexible=1, coarse_max_iter=0)
        psi = torch_gpu.zeros_like(q)
        s.solvePCG(psi, beta, q)
        assert s.converged
        p = to_host(psi)
        out.append((s.iterations, p - p.mean()))
        s.close()
    assert abs(out[0][0] - out[1][0]) <= 1
    assert rel(out[0][1], out[1][1]) < 1e-9


@pytest.mark.parametrize("n", [(2, 4, 2), (4, 2, 6), (12, 10, 2), (66, 6, 4), (132, 4, 8), (256, 4, 8)])
def test_beta_aligned_to_its_elements(torch_gpu, n):
    """A caller's beta and q at an address that is no multiple of 16: the paired loads of the restriction
    read the same values, so the application is the same to the bit."""
    print("case element alignment", n, flush=True)
    g, beta, q = case(torch_gpu, n)

    def shifted(t):
        b = torch_gpu.empty(t.numel() + 1, dtype=t.dtype, device=t.device)[1:].view(t.shape)
        b.copy_(t)
        return b

    a = apply(torch_gpu, g, beta, q, precision="fp64")
    b = apply(torch_gpu, g, shifted(beta), shifted(q), precision="fp64")
    assert np.all(np.isfinite(a)) and np.array_equal(a, b)


@pytest.mark.parametrize("n", [(2, 4, 2), (4, 2, 6), (12, 10, 2), (66, 6, 4), (132, 4, 8), (256, 4, 8), (32, 32, 32)])
def test_cycle_with_one_sweep_matches_oracle_at_remainders(torch_gpu, n):
    """One V-cycle (two levels, one sweep each way, so that the residual and the correction carry it) on axes
    of two cells and rows that leave the last workgroup partly filled, against the oracle to 1e-12."""
    from oracle import pyoracle as O

    print("case restriction, prolongation", n, flush=True)
    g, beta, q = case(torch_gpu, n)
    s = T.PCG(g, nLevels=2, nPreSweep=1, nPostSweep=1, coarse_max_iter=0)
    z = torch_gpu.zeros_like(q)
    s.precondition(beta, q, z)
    s.close()
    go = O.desc(n, stretch=(0, 1, 0), gamma=1.5)
    prm = O.params(n_levels=2, n_pre=1, n_post=1, coarse_mode=1, coarse_cycles=1)
    ref = O.mg_apply(go, prm, to_host(beta), to_host(q))
    out = to_host(z)
    e = rel(out - out.mean(), ref - ref.mean())
    print("  rel error", e, flush=True)
    assert e < 1e-12


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("n", [(2, 4, 2), (4, 2, 6), (12, 10, 2), (66, 6, 4), (72, 40, 56), (256, 4, 8)])
def test_pair_operator_matches_columns(torch_gpu, monkeypatch, n, precision):
    """The direction, operator and pressure update by a thread per pair against the separate kernels with
    the column operator (TBFG_OP_TILE=columns): the solves take the same iterations and agree to 1e-9, the
    target of their residual being 1e-11; the caller's arrays aligned to their elements only."""
    print("case pair operator", n, precision, flush=True)
    g, beta, q = case(torch_gpu, n)

    def shifted(t):
        b = torch_gpu.empty(t.numel() + 1, dtype=t.dtype, device=t.device)[1:].view(t.shape)
        b.copy_(t)
        return b

    def solve(beta, psi):
        s = T.PCG(g, nLevels=2, tolPCG=1e-11, maxIterPCG=200, flexible=1, coarse_max_iter=0, precision=precision)
        s.solvePCG(psi, beta, q)
        it = s.iterations
        s.close()
        return it, to_host(psi)

    ia, a = solve(shifted(beta), shifted(torch_gpu.zeros_like(q)))
    monkeypatch.setenv("TBFG_OP_TILE", "columns")
    ib, b = solve(beta, torch_gpu.zeros_like(q))
    print("  iterations", ia, ib, "rel", rel(a, b), flush=True)
    assert abs(ia - ib) <= 1 and rel(a, b) < 1e-9


@pytest.mark.parametrize("sweeps", ["pairs", "rows"])
@pytest.mark.parametrize("unfused", [False, True], ids=["fused", "unfused"])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_breakdown_ends_the_solve_and_leaves_psi(torch_gpu, monkeypatch, precision, unfused, sweeps):
    """A breakdown of the first step (beta zero: d.Ad is not a number) is found by every workgroup of the
    residual update alike: the solve ends with a numeric error, blocking and queued, psi keeps its bits, and
    the handle solves as a new one afterwards."""
    n = (64, 48, 64)
    print("case breakdown", precision, unfused, sweeps, flush=True)
    if unfused:
        monkeypatch.setenv("TBFG_UNFUSED_OP", "1")
    monkeypatch.setenv("TBFG_SWEEP_MIN_CELLS", "0" if sweeps == "rows" else str(10 ** 12))
    g, beta, q = case(torch_gpu, n)
    kw = dict(nLevels=4, precision=precision, flexible=1, tolPCG=1e-8, maxIterPCG=100)
    start = to_dev(np.random.default_rng(3).normal(size=n), torch_gpu)
    s = T.PCG(g, **kw)
    for queued in (False, True):
        psi = start.clone()
        with pytest.raises(T.TbfgError) as e:
            if queued:
                s.solvePCG_queued(psi, torch_gpu.zeros_like(beta), q, 3)
                torch_gpu.cuda.synchronize()
                s.result()
            else:
                s.solvePCG(psi, torch_gpu.zeros_like(beta), q)
        assert "non-finite" in str(e.value)
        assert torch_gpu.equal(psi, start)
    out = []
    for h in (s, T.PCG(g, **kw)):
        psi = torch_gpu.zeros_like(q)
        h.solvePCG(psi, beta, q)
        assert h.converged
        out.append((h.iterations, h.coarse_stats(), psi))
        h.close()
    assert out[0][:2] == out[1][:2] and torch_gpu.equal(out[0][2], out[1][2])


def _solve(torch, g, beta, q, **kw):
    s = T.PCG(g, flexible=1, coarse_max_iter=0, **kw)
    psi = torch.zeros_like(q)
    s.solvePCG(psi, beta, q)
    out = (s.iterations, s.converged, psi)
    s.close()
    return out


@pytest.mark.parametrize("most", [1, 3, 200])
def test_stop_test_in_the_sweep_ends_as_its_own_launch(torch_gpu, most):
    """bf16 storage, where the rows round as the tiles do: with the first sweep's tile shape entered in the
    tuning table the stop test is a launch of its own, without it a workgroup of that sweep.  Converged or at
    the iteration limit, the iterations and the bits of psi are the same."""
    from tbfsolver_amd import tune as Tu

    n = (128, 64, 128)
    print("case folded stop test", most, flush=True)
    g, beta, q = case(torch_gpu, n)
    kw = dict(nLevels=4, precision="mixed-bf16", tolPCG=1e-8, maxIterPCG=most)
    Tu.clear()
    try:
        a = _solve(torch_gpu, g, beta, q, **kw)
        Tu.set_entry("sweep_edge", n, "mixed", (64, 8, 256))  # the built-in choice, by name
        b = _solve(torch_gpu, g, beta, q, **kw)
    finally:
        Tu.clear()
    assert a[:2] == b[:2] and a[1] == (most == 200) and (a[1] or a[0] == most), (a[:2], b[:2])
    assert torch_gpu.equal(a[2], b[2])


@pytest.mark.parametrize("sweeps", ["pairs", "rows"])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_stop_test_in_pair_and_row_sweeps(torch_gpu, monkeypatch, precision, sweeps):
    """The same on levels smoothed by pairs and rows, against the half-sweep launches (which leave the stop
    test to its own launch): the iterations, at the limit and converged; psi to ten times the residual bound."""
    n = (48, 32, 64)
    print("case folded stop test", precision, sweeps, flush=True)
    monkeypatch.setenv("TBFG_SWEEP_MIN_CELLS", "0" if sweeps == "rows" else str(10 ** 12))
    g, beta, q = case(torch_gpu, n)
    for most in (1, 2, 5, 200):
        kw = dict(nLevels=3, precision=precision, tolPCG=1e-10, maxIterPCG=most)
        monkeypatch.delenv("TBFG_HALF_SWEEPS", raising=False)
        a = _solve(torch_gpu, g, beta, q, **kw)
        monkeypatch.setenv("TBFG_HALF_SWEEPS", "1")
        b = _solve(torch_gpu, g, beta, q, **kw)
        assert a[1] == b[1] == (most == 200)
        if most < 200:
            assert a[0] == b[0] == most
        else:
            assert abs(a[0] - b[0]) <= 1
            assert rel(to_host(a[2] - a[2].mean()), to_host(b[2] - b[2].mean())) < 1e-9


@pytest.mark.parametrize("precision", ["fp64", "mixed", "mixed-bf16"])
def test_shapes_entered_while_solves_run(torch_gpu, precision):
    """Another thread enters and removes the first sweep's tile shape all the while: the stop test is neither
    lost nor made twice.  Iterations within one (the shapes round differently), converged to the same psi."""
    import threading

    from tbfsolver_amd import tune as Tu

    n = (128, 64, 128)
    print("case tuning during solves", precision, flush=True)
    g, beta, q = case(torch_gpu, n)
    kw = dict(nLevels=4, precision=precision, tolPCG=1e-8, maxIterPCG=200)
    key, shape = ("fp64", (64, 4, 128)) if precision == "fp64" else ("mixed", (64, 8, 256))
    Tu.clear()
    stop, turns = threading.Event(), [0]

    def toggle():
        while not stop.is_set():
            Tu.set_entry("sweep_edge", n, key, shape)
            Tu.set_entry("sweep_edge", n, key, (0, 0, 0))
            turns[0] += 1

    quiet = _solve(torch_gpu, g, beta, q, **kw)
    t = threading.Thread(target=toggle)
    t.start()
    try:
        out = [_solve(torch_gpu, g, beta, q, **kw) for _ in range(5)]
    finally:
        stop.set()
        t.join()
        Tu.clear()
    assert quiet[1] and turns[0] > 0
    for it, converged, psi in out:
        assert converged and abs(it - quiet[0]) <= 1
        assert rel(to_host(psi - psi.mean()), to_host(quiet[2] - quiet[2].mean())) < 1e-6
