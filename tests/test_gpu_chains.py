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


@pytest.mark.parametrize("layout", ["rows", "rows padded", "element-major"])
@pytest.mark.parametrize("M,batch", [(1, 5), (2, 1), (7, 3), (8, 4), (9, 5), (127, 6), (128, 4), (129, 9), (257, 2), (1025, 5),
                                     (33, 4097)])
def test_thomas_layouts(qa, oracle, M, batch, layout):
    """thomas_batched and the strided entry point: the last rows' pairs and blocks, batches that leave a wave's DPP rows
    empty, both kernels of element-major systems, and systems whose pivots leave the reciprocal's range."""
    import torch
    rng = np.random.default_rng(M * 7 + batch)
    a, c, d = (rng.uniform(-1, 1, (batch, M)) for _ in range(3))
    b = 2.5 + rng.uniform(-1, 1, (batch, M))
    for s, e in ((0, 1e-310), (1, 1e305), (2, 1e-305)):
        if s < batch:
            a[s], b[s], c[s] = a[s] * e, b[s] * e, c[s] * e
    a[:, 0], c[:, -1] = np.inf, np.nan   # not used
    with np.errstate(all="ignore"):
        n = min(batch, 9)
        ref = [oracle.thomas(np.r_[0.0, a[s, 1:]], b[s].copy(), np.r_[c[s, :-1], 0.0], d[s].copy()) for s in range(n)]
    width = M + 3 if layout == "rows padded" else M
    host = [np.pad(v, ((0, 0), (0, width - M))) for v in (a, b, c, d)]
    if layout == "element-major":
        host = [np.ascontiguousarray(v.T) for v in host]
    dev = [torch.from_numpy(v).cuda() for v in host]
    x = torch.zeros_like(dev[3])
    work = torch.empty(max(1, qa.lib().qz_tridiag_workspace_doubles(M, batch)), dtype=torch.float64, device="cuda")
    ss, es = (1, batch) if layout == "element-major" else (width, 1)
    ptr = [v.data_ptr() for v in dev]
    qa.check(qa.lib().qz_tridiag_thomas_batched(*ptr, x.data_ptr(), M, batch, ss, es, work.data_ptr(), None))
    torch.cuda.synchronize()
    got = x.cpu().numpy()
    got = got.T if layout == "element-major" else got[:, :M]
    for s in range(n):
        r, g = np.asarray(ref[s]), np.ascontiguousarray(got[s])
        nan = np.isnan(r)
        assert np.array_equal(np.isnan(g), nan), s
        assert np.array_equal(g[~nan].view(np.int64), r[~nan].view(np.int64)), s


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


def test_steps_in_flight_of_several_workgroups(qa, tmp_path):
    """Sixteen steps with three in flight, each sweep on eight workgroups beside the others', equal the same steps one at
    a time, bit for bit: a workgroup reads nothing that another has not yet made visible, whatever runs beside it."""
    from quarz_amd import configs
    deck = configs.c3_deck(workdir=str(tmp_path), xi_min=-1.5, steps=30, nd=100000, nw=20000, driver_xi0=-0.6,
                           witness_xi0=-1.2)
    ov = {"driver.sigma_xi": 0.2, "driver.x0": 0.05, "driver.n0": 2, "witness.sigma_xi": 0.05}
    a = qa.Simulation(deck, ov)
    b = qa.Simulation(deck, ov)
    assert a.groups == 8 and b.groups == 8
    for _ in range(16):
        a.step()
    b.step()
    b.run_pipelined(15, chunks=6, depth=3)
    for w in ("fld", "diag", "bsrc"):
        assert np.array_equal(np.array(getattr(b, w)), np.array(getattr(a, w))), w
