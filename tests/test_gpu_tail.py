"""The tail kernel that smooths its levels from registers against the form that keeps them
in global memory: one preconditioner application where its first level has one or two
pairs of cells per thread (up to 4096 cells) or more (loops over the cells), with bottoms of
one cell, up to 64 and beyond, axes of two cells, sweep counts that include none.  The same
arithmetic up to the order of the bottom's FP64 sums: 1e-13 in FP64, 1e-6 in FP32."""
import numpy as np
import pytest

import tbfsolver_amd as T
from conftest import to_dev, to_host

pytestmark = pytest.mark.gpu


def apply(torch, n, precision, **kw):
    g = T.channel_grid(n, stretch_y=1, gamma=1.5)
    r = np.random.default_rng(11)
    beta = to_dev(np.exp(r.uniform(-1.5, 1.5, n)), torch)
    q = r.standard_normal(n)
    q = to_dev(q - q.mean(), torch)
    s = T.PCG(g, precision=precision, coarse_max_iter=0, **kw)
    z = torch.zeros_like(q)
    s.precondition(beta, q, z)
    out = to_host(z)
    s.close()
    return out


@pytest.mark.parametrize("precision,bound", [("fp64", 1e-13), ("mixed", 1e-6)])
@pytest.mark.parametrize("n,cells", [
    ((72, 40, 56), 4096),   # 2520 cells above a bottom of 315
    ((64, 48, 64), 4096),   # 1536 cells, bottom of 36
    ((32, 32, 32), 4096),   # 4096 cells down to one
    ((32, 32, 32), 20000),  # more than two pairs per thread
    ((128, 16, 16), 4096),  # 4096 cells in long rows, bottom of 8
    ((36, 20, 12), 4096),   # 1080 cells, bottom of 135
    ((64, 8, 8), 4096),     # 512 cells, levels of two cells along two axes
    ((8, 4, 4), 4096),      # 16 cells
    ((2, 6, 8), 4096),      # the bottom alone
])
def test_tail_from_registers(torch_gpu, monkeypatch, n, cells, precision, bound):
    print("case tail", n, cells, precision, flush=True)
    monkeypatch.setenv("TBFG_TAIL_CELLS", str(cells))
    for pre, post in ((2, 2), (0, 1), (3, 0)):
        a = apply(torch_gpu, n, precision, nLevels=2, nPreSweep=pre, nPostSweep=post)
        monkeypatch.setenv("TBFG_TAIL_HBM", "1")
        b = apply(torch_gpu, n, precision, nLevels=2, nPreSweep=pre, nPostSweep=post)
        monkeypatch.delenv("TBFG_TAIL_HBM")
        assert np.all(np.isfinite(a))
        assert np.linalg.norm(a - b) <= bound * np.linalg.norm(b)
