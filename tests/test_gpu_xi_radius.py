"""xi_vec transforms only the rows that hold a separation below the last edge.  Bins of a short set
of edges hold the same integer sums as the same bins of a set that reaches the grid's corner."""
import numpy as np
import pytest
import torch

from jax_powspec_amd import correlations

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [8, 24, 64, 96, 256, 512])
def test_short_edges_equal_the_full_set(n):
    dev = torch.device("cuda", 0)
    g = torch.Generator(device=dev)
    g.manual_seed(n)
    d = torch.randn((n, n, n), device=dev, generator=g)
    d += torch.roll(d, (1, 2, 1), (0, 1, 2))
    # half-integer edges in cells (box = n): no separation lies on one
    full = 0.5 + np.arange(int(np.sqrt(3) * n / 2) + 1)
    _, _, _, want = correlations.xi_vec(d, float(n), full, full=True)
    h = n // 2
    for bins in sorted({1, 2, 3, h // 8 + 1, h // 2, h - 2, h - 1, h, h + 1}):
        if not 1 <= bins < full.size:
            continue
        _, _, _, got = correlations.xi_vec(d, float(n), full[:bins + 1], full=True)
        assert torch.equal(got["sums"], want["sums"][:bins]), (n, bins)
        assert torch.equal(got["counts"], want["counts"][:bins])


def test_no_cell_below_the_last_edge():
    dev = torch.device("cuda", 0)
    d = torch.randn((32, 32, 32), device=dev)
    _, xi, modes = correlations.xi_vec(d, 32.0, np.array([0.2, 0.5, 0.7]))
    assert bool((xi == 0).all()) and bool(torch.isinf(modes).all())
