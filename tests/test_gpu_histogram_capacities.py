"""The binning x pass on both sides of every capacity of its histograms in LDS: bins that split a few wide ones give,
added up again, their counts exactly and their sums to the rounding of the float runs (at most 9 rows)."""
import numpy as np
import pytest
import torch

from jax_powspec_amd import correlations

pytestmark = pytest.mark.gpu

# side, wide bins, parts of each: 256 | 257 and 4061 | 4062 at 64, 256 | 257 at 256, 766 | 767 and 2816 | 2817 at 512,
# 514 | 515 and 2564 | 2565 at 1024
CASES = [(64, 16, 16), (64, 1, 257), (64, 31, 131), (64, 6, 677), (256, 16, 16), (256, 1, 257), (512, 2, 383), (512, 13, 59), (512, 4, 704), (512, 9, 313),
         (1024, 2, 257), (1024, 5, 103), (1024, 4, 641), (1024, 5, 513)]


@pytest.mark.parametrize("n,wide,parts", CASES)
def test_split_bins_add_up(gpu, n, wide, parts):
    g = torch.Generator(device=gpu)
    g.manual_seed(n)
    delta = torch.randn((n, n, n), device=gpu, generator=g)
    delta += 0.5 * torch.roll(delta, (1, 2, 3), (0, 1, 2))
    kf = 2 * np.pi / 1000.0
    # irrational splits: no mode lies on an edge of either set
    coarse = 0.5 + np.arange(wide + 1) * ((n / 2 + 0.25) / wide) * (1 + 1e-7 * np.sqrt(2))
    fine = np.interp(np.arange(wide * parts + 1) / parts, np.arange(wide + 1), coarse)
    want = correlations.powspec_vec(delta, 1000.0, coarse * kf, full=True)[3]
    got = correlations.powspec_vec(delta, 1000.0, fine * kf, full=True)[3]
    torch.testing.assert_close(got["counts"].view(wide, parts).sum(1), want["counts"], rtol=0, atol=0)
    s = got["sums"].view(wide, parts, 3).sum(1)
    bound = 2 * 9 * 2.0 ** -24 * want["sums"][:, :1]
    assert bool(((s - want["sums"]).abs() <= bound).all()), ((s - want["sums"]).abs() / want["sums"][:, :1]).max()
