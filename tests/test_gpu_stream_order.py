"""Runs on a stream of the caller's: the order of the streams is what the caller made it.  The stream that an
object is made on is kept busy (50 ms), so that work left on it comes too late to go unnoticed."""
import numpy as np
import pytest
import torch

from jax_powspec_amd import batch, correlations, serve

pytestmark = pytest.mark.gpu

N, BOX, NP = 64, 500.0, 50_000
EDGES = 2 * np.pi / BOX * (0.5 + np.arange(N // 2 + 1))


def busy():
    """about 50 ms on the current stream"""
    a = torch.ones((4096, 4096), device="cuda")
    for _ in range(60):
        a = (a @ a) * (1.0 / 4096)
    return a


def positions(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return torch.rand((NP, 3), device="cuda", generator=g) * (BOX - 0.01)


def cat(p):
    return dict(x=p[:, 0], y=p[:, 1], z=p[:, 2], box_size=BOX, n_bins=N, k_edges=EDGES, mas="CIC")


def plain(p):
    return correlations.estimate(p[:, 0], p[:, 1], p[:, 2], box_size=BOX, n_bins=N, k_edges=EDGES, mas="CIC")


@pytest.fixture(scope="module")
def warm(gpu):
    p = positions(0)
    b = batch.BatchEstimator(N, 2, NP, len(EDGES) - 1)
    b.set([cat(p)] * 2).run()
    busy()
    torch.cuda.synchronize()


def test_a_new_batch_is_filled_before_it_runs(warm):
    ps = [positions(1), positions(2)]
    want = [plain(p) for p in ps]
    torch.cuda.synchronize()
    s = torch.cuda.Stream()
    busy()
    b = batch.BatchEstimator(N, 2, NP, len(EDGES) - 1)
    b.set([cat(p) for p in ps], stream=s).run(stream=s)
    torch.cuda.synchronize()   # whatever was left on the current stream has run as well
    for i, w in enumerate(want):
        assert abs(float(b.stats[i, 0]) - NP) < 1e-3 * NP
        assert torch.equal(b.result(i)[1], w[1])


def late_doubles(s):
    """positions in float64, complete on stream s only after a while"""
    p = positions(3)
    want = plain(p)
    torch.cuda.synchronize()
    with torch.cuda.stream(s):
        d = torch.zeros((NP, 3), dtype=torch.float64, device="cuda")
        torch.cuda.synchronize()
        busy()
        d.copy_(p)
    return d, want


def test_batch_inputs_are_converted_on_the_callers_stream(warm):
    s = torch.cuda.Stream()
    b = batch.BatchEstimator(N, 2, NP, len(EDGES) - 1)
    torch.cuda.synchronize()
    d, want = late_doubles(s)
    b.set([cat(d)], stream=s).run(stream=s)
    torch.cuda.synchronize()
    assert torch.equal(b.result(0)[1], want[1])


def test_estimator_inputs_are_converted_on_the_runs_stream(warm):
    s = torch.cuda.Stream()
    est = correlations.Estimator(box_size=BOX, n_bins=N, max_particles=NP, k_edges=EDGES, mas="CIC")
    torch.cuda.synchronize()
    d, want = late_doubles(s)
    pk = est.run(d[:, 0], d[:, 1], d[:, 2], stream=s)
    torch.cuda.synchronize()
    assert torch.equal(pk, want[1])


def test_served_inputs_are_converted_once_they_are_complete(warm):
    s = torch.cuda.Stream()
    srv = serve.PkServer(max_batch=2, max_particles=NP)
    try:
        srv.submit(cat(positions(4))).result(60)   # the engine exists
        d, want = late_doubles(s)
        with torch.cuda.stream(s):
            f = srv.submit(cat(d))                 # ready: on s
        np.testing.assert_array_equal(f.result(60)[1], want[1].cpu().numpy())
    finally:
        srv.close()
