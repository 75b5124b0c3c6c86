"""Batched Thomas on both sides of its dispatch rule (systems and rows), in every layout that the strides allow: every
system against the serial operations of every row, and short systems no slower than their memory traffic asks for."""
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


def _reference(a, b, c, d):
    """The rows of every system (batch, M) in the oracle's order of operations (src/Tridiag.cpp:111-126)."""
    M = d.shape[1]
    cp, dp = np.empty_like(d), np.empty_like(d)
    cp[:, 0], dp[:, 0] = c[:, 0] / b[:, 0], d[:, 0] / b[:, 0]
    for i in range(1, M):
        m = 1.0 / (b[:, i] - a[:, i] * cp[:, i - 1])
        cp[:, i] = c[:, i] * m
        dp[:, i] = (d[:, i] - a[:, i] * dp[:, i - 1]) * m
    x = dp.copy()
    for i in range(M - 2, -1, -1):
        x[:, i] = dp[:, i] - cp[:, i] * x[:, i + 1]
    return x


@pytest.mark.parametrize("layout", ["rows", "rows padded", "element-major", "interleaved"])
@pytest.mark.parametrize("batch", [4096, 4097, 4225])
@pytest.mark.parametrize("M", [1, 2, 3, 4, 8, 9, 10, 16, 17, 18, 34])
def test_every_system(qa, oracle, M, batch, layout):
    import torch
    rng = np.random.default_rng(1000 * M + batch)
    a, c, d = (rng.uniform(-1, 1, (batch, M)) for _ in range(3))
    b = 2.5 + rng.uniform(-1, 1, (batch, M))
    ref = _reference(a, b, c, d)
    for s in (0, batch - 1):   # the vectorised rows are the oracle's
        assert np.array_equal(ref[s], oracle.thomas(np.r_[0.0, a[s, 1:]], b[s].copy(), np.r_[c[s, :-1], 0.0], d[s].copy()))
    # the strides of system and element, and the doubles they span
    ss, es = {"rows": (M, 1), "rows padded": (M + 3, 1), "element-major": (1, batch), "interleaved": (3 * M + 1, 3)}[layout]
    at = np.arange(batch)[:, None] * ss + np.arange(M)[None, :] * es
    size = int(at.max()) + 8

    def dev(v):
        h = np.full(size, 7.0)
        h[at] = v
        return torch.from_numpy(h).cuda()

    ptr = [dev(v) for v in (a, b, c, d)]
    x = dev(np.zeros((batch, M)))
    work = torch.empty(max(1, qa.lib().qz_tridiag_workspace_doubles(M, batch)), dtype=torch.float64, device="cuda")
    qa.check(qa.lib().qz_tridiag_thomas_batched(*[v.data_ptr() for v in ptr], x.data_ptr(), M, batch, ss, es,
                                                work.data_ptr(), None))
    torch.cuda.synchronize()
    got = x.cpu().numpy()
    assert np.array_equal(got[at].view(np.int64), ref.view(np.int64))
    rest = np.ones(size, bool)
    rest[at] = False
    assert (got[rest] == 7.0).all()   # nothing beside the systems is written


@pytest.mark.parametrize("M", [2, 5, 9])
def test_short_systems_cost_their_traffic(qa, M):
    """262144 short systems stored row after row: within 6 times a copy of the same bytes (a wave's whole blocks of 8
    rows per lane took 9 to 45 times it, a thread per system takes 2 to 3)."""
    import torch
    batch = 262144
    a, c, d = (torch.rand(batch, M, dtype=torch.float64, device="cuda") for _ in range(3))
    b = 3.0 + torch.rand(batch, M, dtype=torch.float64, device="cuda")
    x, work = torch.empty_like(d), torch.empty(M * batch, dtype=torch.float64, device="cuda")
    src, dst = torch.empty(3 * M * batch, dtype=torch.float64, device="cuda"), torch.empty(3 * M * batch, dtype=torch.float64,
                                                                                         device="cuda")
    stream = torch.cuda.current_stream()

    def best(f):
        times = []
        for _ in range(5):
            e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            e0.record()
            for _ in range(10):
                f()
            e1.record()
            torch.cuda.synchronize()
            times.append(e0.elapsed_time(e1))
        return min(times)

    ptr = [v.data_ptr() for v in (a, b, c, d, x)]
    solve = best(lambda: qa.check(qa.lib().qz_tridiag_thomas_batched(*ptr, M, batch, M, 1, work.data_ptr(),
                                                                     stream.cuda_stream)))
    copy = best(lambda: dst.copy_(src))
    assert solve < 6 * max(copy, 0.06), (solve, copy)
