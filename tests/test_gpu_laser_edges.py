"""The laser march at the edges of its layout (nodes per thread, blocks of the serial chain, the largest grid in LDS)
and at the ends of the exponent range (where its corrected quotients give way to the division), against the oracle's
restatement, bit for bit."""
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


def _same_bits(a, b):
    return a.shape == b.shape and np.array_equal(a.view(np.int64), b.view(np.int64))


@pytest.mark.parametrize("scheme", ["trapezoid", "bdf2"])
@pytest.mark.parametrize("M", [3, 4, 9, 64, 65, 66, 67, 129, 512, 513, 1024, 1025, 1861])
def test_march_sizes(qa, oracle, M, scheme):
    import torch
    nodes = 12.0 * (np.arange(M) / (M - 1)) ** 1.2
    S = oracle.Solver(nodes)
    rng = np.random.default_rng(M)
    K, dxi, dt, k0 = 9, 0.05, 2.0, 12.0
    a = rng.standard_normal((K, M, 2)) * np.exp(-nodes ** 2 / 8)[None, :, None]
    a[:, M - 1] = 0
    chi = 0.3 * (1 + 0.1 * rng.standard_normal((K, M)))
    L = qa.Laser(nodes, K, 0.0, dxi, dt, k0, scheme=scheme)
    L.set_envelope(a)
    for n in range(2):
        a, pond = S.laser_step(a, dxi, dt, k0, L.SCHEMES[scheme], False, chi)
        L.step(torch.from_numpy(chi).cuda())
        assert _same_bits(L.envelope(), a), n
        assert _same_bits(L.ponderomotive(), pond), n
    L.close()


@pytest.mark.parametrize("scale", [0.0, 5e-324, 1e-310, 1e-300, 1e-290, 1e150, 1e300, np.inf, np.nan])
def test_march_exponent_range(qa, oracle, scale):
    """An envelope that falls through the subnormals (or overflows) along the box: two steps."""
    M, K, dxi, dt, k0 = 131, 24, 0.05, 2.0, 12.0
    nodes = 6.0 * np.arange(M) / (M - 1)
    S = oracle.Solver(nodes)
    rng = np.random.default_rng(5)
    with np.errstate(all="ignore"):
        a = rng.standard_normal((K, M, 2)) * scale * 10.0 ** (-np.arange(K) % 7)[:, None, None]
    a[:, M - 1] = 0
    L = qa.Laser(nodes, K, 0.0, dxi, dt, k0, scheme="trapezoid")
    L.set_envelope(a)
    for _ in range(2):
        a, _ = S.laser_step(a, dxi, dt, k0, 0, False, np.zeros((K, M)))
        L.step()
        got = L.envelope()
        nan = np.isnan(a)
        assert np.array_equal(np.isnan(got), nan)
        assert np.array_equal(got[~nan].view(np.int64), a[~nan].view(np.int64))
    L.close()
