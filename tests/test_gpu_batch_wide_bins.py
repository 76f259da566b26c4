"""Batches whose jobs differ in what their kernels lay out by themselves: more than 256 bins and unequal numbers of
them (the x pass' histogram takes its LDS from the largest), and sorts of different kinds beside each other.
Each job against the plain call: mode counts exactly, sums to the rounding of the float runs (at most 9
rows each)."""
import numpy as np
import pytest
import torch

from jax_powspec_amd import batch, correlations

pytestmark = pytest.mark.gpu

BOX = 1000.0
# side, rows per tile (None: default), (bins, stencil) of every job.  766 bins are the tall histogram's most at 512 and
# 514 at 1024, 4061 the most of any in LDS at 64; at 512 with 16 rows TSC jobs count x planes and CIC jobs keys
CASES = [(512, None, [(300, "CIC"), (766, "TSC"), (20, "CIC_REF")]), (512, None, [(767, "CIC"), (257, "TSC")]),
         (512, 16, [(300, "TSC"), (700, "CIC")]), (512, 16, [(40, "CIC"), (64, "TSC")]),
         (1024, None, [(514, "CIC"), (300, "CIC_REF"), (30, "CIC")]), (128, None, [(1000, "CIC"), (257, "TSC"), (64, "CIC")]),
         (64, None, [(4061, "CIC"), (300, "CIC")]), (64, None, [(300, "CIC"), (4062, "CIC")])]


@pytest.mark.parametrize("capacity_grids", [False, True])
@pytest.mark.parametrize("case", range(len(CASES)))
def test_every_job_equals_the_plain_call(gpu, case, capacity_grids):
    n, ty, jobs = CASES[case]
    tile = None if ty is None else (1, ty, 0)
    cats, want = [], []
    for i, (nb, stencil) in enumerate(jobs):
        g = torch.Generator(device=gpu)
        g.manual_seed(100 * case + i)
        p = torch.rand((150_000 - 40_000 * i, 3), device=gpu, generator=g) * (BOX - 0.01)
        edges = 2 * np.pi / BOX * (0.5 + np.arange(nb + 1) * ((n / 2 + 0.25) / nb) * (1 + 1e-7 * np.sqrt(2)))
        cats.append(dict(x=p[:, 0], y=p[:, 1], z=p[:, 2], box_size=BOX, n_bins=n, mas=stencil, k_edges=edges))
        want.append(correlations.estimate(p[:, 0], p[:, 1], p[:, 2], box_size=BOX, n_bins=n, mas=stencil, k_edges=edges,
                                          tile=tile, full=True)[3])
    b = batch.BatchEstimator(n, len(cats), 200_000, max(nb for nb, _ in jobs) + 50, tile=tile, device=gpu,
                             capacity_grids=capacity_grids)
    for _ in range(3):   # plain launches, capture, replay
        b.set(cats).run()
    for i, w in enumerate(want):
        got = b.result(i, full=True)[3]
        assert torch.equal(got["counts"], w["counts"])
        bound = 2 * 9 * 2.0 ** -24 * w["sums"][:, :1]
        assert bool(((got["sums"] - w["sums"]).abs() <= bound).all())
