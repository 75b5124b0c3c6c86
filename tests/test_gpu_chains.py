"""The radial recurrences of the sweeps (qz_chain.hpp: blocks of 128 rows, 8 rows per lane) at the sizes where a block,
a lane or a pair of rows ends, in the one-workgroup and the multi-workgroup sweep, modes 0 and 1, against the oracle
bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def qa():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import quarz_amd
    quarz_amd.lib()
    return quarz_amd


@pytest.mark.parametrize("modes,groups", [(0, 1), (0, 2), (1, 1), (1, 2)])
@pytest.mark.parametrize("N", [4, 7, 8, 9, 63, 64, 126, 127, 128, 129, 254, 255, 256, 383, 500])
def test_rows(qa, oracle, decks, N, modes, groups):
    ov = {"modes": modes, "grid.rmax": 4, "grid.dr": 4.0 / N, "xi.min": -1.2, "xi.step": 0.03, "driver.n0": 1.5,
          "driver.sigma_r": 0.4, "driver.sigma_xi": 0.2, "driver.xi0": -0.5, "driver.cut": 3, "driver.nparticles": 4000,
          "driver.x0": 0.05 if modes else 0, "electrons.ppc": 1}
    g = qa.Simulation(f"{decks}/linear.in", {**ov, "sweep.groups": groups})
    o = oracle.Sim(f"{decks}/linear.in", ov)
    assert g.groups == groups and g.M == N + 1
    g.step()
    o.step()
    for w in ("fld", "diag"):
        a, b = getattr(g, w), getattr(o, w)
        assert a.shape == b.shape and np.array_equal(a, b), (w, np.argwhere(a != b)[:3])


@pytest.mark.parametrize("N", [769, 1024])
def test_rows_large_m0(qa, oracle, decks, N):
    ov = {"grid.rmax": 8, "grid.dr": 8.0 / N, "xi.min": -0.9, "xi.step": 0.03, "driver.n0": 1.5, "driver.sigma_r": 0.4,
          "driver.sigma_xi": 0.2, "driver.xi0": -0.5, "driver.cut": 3, "driver.nparticles": 4000}
    for groups in (1, 3):
        g = qa.Simulation(f"{decks}/linear.in", {**ov, "sweep.groups": groups})
        o = oracle.Sim(f"{decks}/linear.in", ov)
        g.step()
        o.step()
        assert np.array_equal(g.fld, o.fld) and np.array_equal(g.diag, o.diag), groups
