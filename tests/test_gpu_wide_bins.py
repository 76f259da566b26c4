"""The binning x pass keeps its histogram in LDS up to a capacity that depends on the mesh side,
and in HBM beyond it.  Every placement sums the same modes: bins split q ways give, added up
again, the counts of the unsplit bins exactly and their sums to the rounding of the float runs."""
import numpy as np
import pytest
import torch

from jax_powspec_amd import correlations

pytestmark = pytest.mark.gpu

BINS = 64
# 64 q bins: below and above 256 (the usual histogram), around the capacities of the
# dynamic ones (512: 512, 768 | 832; 1024: 512 | 576) and beyond all of them
CASES = [(48, 4), (48, 5), (48, 80), (384, 6), (512, 4), (512, 8), (512, 12), (512, 13), (512, 44), (512, 45),
         (1024, 4), (1024, 8), (1024, 9), (1024, 40)]


@pytest.fixture(scope="module")
def meshes():
    made = {}

    def get(n, dev):
        if n not in made:
            made.clear()
            g = torch.Generator(device=dev)
            g.manual_seed(n)
            d = torch.randn((n, n, n), device=dev, generator=g)
            made[n] = d + 0.5 * torch.roll(d, (1, 2, 3), (0, 1, 2))
        return made[n]
    return get


@pytest.mark.parametrize("n,q", CASES)
def test_split_bins_add_up(meshes, n, q):
    dev = torch.device("cuda", 0)
    delta = meshes(n, dev)
    box = 1000.0
    kf = 2 * np.pi / box
    # irrational splits: no mode lies on an edge of either set
    coarse = 0.5 + np.arange(BINS + 1) * ((n / 2 + 0.25) / BINS) * (1 + 1e-7 * np.sqrt(2))
    fine = np.interp(np.arange(BINS * q + 1) / q, np.arange(BINS + 1), coarse)
    _, _, _, want = correlations.powspec_vec(delta, box, coarse * kf, full=True)
    _, _, _, got = correlations.powspec_vec(delta, box, fine * kf, full=True)
    torch.testing.assert_close(got["counts"].view(BINS, q).sum(1), want["counts"], rtol=0, atol=0)
    s = got["sums"].view(BINS, q, 3).sum(1)
    # a run adds at most 9 rows in float32: 9 2^-24 of its power on each side
    bound = 2 * 9 * 2.0 ** -24 * want["sums"][:, :1]
    assert bool(((s - want["sums"]).abs() <= bound).all()), ((s - want["sums"]).abs() / want["sums"][:, :1]).max()
