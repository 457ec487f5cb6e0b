"""Material properties on the device (updateMaterialProps + smoothVF,
VOF.f90:197-262) against the oracle: the smoothed volume fraction, rho and mu
to round-off (1e-14 of the values' scale) on a stretched channel grid."""
import numpy as np
import pytest

import tbfsolver_amd as T
from tbfsolver_amd import fields as F
from oracle import pyoracle as O
from conftest import to_dev, to_host

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,stretch", [((48, 40, 32), 1), ((32, 16, 24), 0), ((256, 192, 256), 1)])
def test_material_props_match_oracle(torch_gpu, n, stretch):
    print("case material props", n, stretch, flush=True)
    g = T.channel_grid(n, stretch_y=stretch, gamma=1.5)
    go = O.desc(n, stretch=(0, stretch, 0), gamma=1.5)
    rng = np.random.default_rng(9)
    c = np.clip(rng.random(n) * 1.4 - 0.2, 0.0, 1.0)  # with runs of pure 0 and 1
    cs_r, rho_r, mu_r = O.material_props(go, c, rho_l=1.0, rho_g=0.05, mu_l=1.0, mu_g=0.02)
    dc = to_dev(c, torch_gpu)
    cs, rho, mu = (torch_gpu.zeros_like(dc) for _ in range(3))
    F.updateMaterialProps(g, dc, cs, rho, mu, rho_l=1.0, rho_g=0.05, mu_l=1.0, mu_g=0.02)
    torch_gpu.cuda.synchronize()
    for a, b in ((cs, cs_r), (rho, rho_r), (mu, mu_r)):
        assert np.abs(to_host(a) - b).max() <= 1e-14 * max(1.0, np.abs(b).max())
    # without mu, and the second call reuses the cached coordinate tables
    rho2 = torch_gpu.zeros_like(dc)
    F.updateMaterialProps(g, dc, cs, rho2, None, rho_l=1.0, rho_g=0.05)
    torch_gpu.cuda.synchronize()
    assert torch_gpu.equal(rho2, rho)


@pytest.mark.parametrize("n,stretch", [((5, 3, 2), 1), ((2, 1, 3), 0), ((33, 17, 9), 1), ((96, 50, 31), 1),
                                       ((130, 33, 70), 0), ((64, 16, 4), 1)])
def test_material_props_ragged_sizes_and_aliases(torch_gpu, n, stretch):
    """Remainders of the tiles and axes shorter than the filter; outputs over the input
    (rho in place of c) give the same values.  Bound: three five-point filters of values
    up to 1 round to 15 eps, the oracle's four passes of eight products and a division to
    20 eps, together below 1e-14."""
    print("case material props ragged", n, stretch, flush=True)
    g = T.channel_grid(n, stretch_y=stretch, gamma=1.5)
    go = O.desc(n, stretch=(0, stretch, 0), gamma=1.5)
    c = np.clip(np.random.default_rng(10).random(n) * 1.4 - 0.2, 0.0, 1.0)
    cs_r, rho_r, mu_r = O.material_props(go, c, rho_l=1.0, rho_g=0.05, mu_l=1.0, mu_g=0.02)
    dc = to_dev(c, torch_gpu)
    cs, rho, mu = (torch_gpu.zeros_like(dc) for _ in range(3))
    F.updateMaterialProps(g, dc, cs, rho, mu, rho_l=1.0, rho_g=0.05, mu_l=1.0, mu_g=0.02)
    torch_gpu.cuda.synchronize()
    for a, b in ((cs, cs_r), (rho, rho_r), (mu, mu_r)):
        assert np.abs(to_host(a) - b).max() <= 1e-14
    cs2, mu2 = torch_gpu.zeros_like(dc), torch_gpu.zeros_like(dc)
    F.updateMaterialProps(g, dc, cs2, dc, mu2, rho_l=1.0, rho_g=0.05, mu_l=1.0, mu_g=0.02)
    torch_gpu.cuda.synchronize()
    assert torch_gpu.equal(cs2, cs) and torch_gpu.equal(dc, rho) and torch_gpu.equal(mu2, mu)
