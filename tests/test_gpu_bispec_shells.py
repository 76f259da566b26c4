"""The later shells' sums go by rows of the spectrum, 8 shells per block and 128 per launch: every
triangle's result equals that of a call with it alone (other chunk and launch shapes), to the
rounding of FP64 sums in another order."""
import numpy as np
import pytest
import torch

from jax_powspec_amd import correlations

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,count", [(16, 1), (24, 8), (48, 9), (64, 129), (96, 17), (128, 140)])
@pytest.mark.parametrize("reuse", [False, True])
def test_many_shells_equal_single_ones(n, count, reuse):
    dev = torch.device("cuda", 0)
    g = torch.Generator(device=dev)
    g.manual_seed(n + count)
    d = torch.randn((n, n, n), device=dev, generator=g)
    d = d + 0.5 * torch.roll(d, (1, 1, 1), (0, 1, 2)) + 0.2 * (d * d - 1)
    kf = 2 * np.pi / 1000.0
    k1, k2 = 0.22 * n / 2 * kf, 0.4 * n / 2 * kf
    theta = np.linspace(0.05, np.pi - 0.05, count)
    *_, many = correlations.bispec(d, 1000.0, k1, k2, theta, full=True, reuse_shell_sums=reuse)
    if reuse:   # the second call takes the shells' indicator sums as given
        *_, many = correlations.bispec(d, 1000.0, k1, k2, theta, full=True)
    for i in {0, count // 2, count - 1}:
        *_, one = correlations.bispec(d, 1000.0, k1, k2, theta[i:i + 1], full=True, reuse_shell_sums=False)
        a, b = many["sums"][2 + i], one["sums"][2]
        # sums of squares and of signed products: relative to sqrt(sum delta_i^2 sum delta_1^2) and alike
        assert torch.allclose(a[:2], b[:2], rtol=1e-12, atol=0)
        scale = (b[0] * many["sums"][0, 0]).sqrt() * many["sums"][1, 0].sqrt()
        assert abs(float(a[2] - b[2])) <= 1e-12 * float(scale)
        assert abs(float(a[3] - b[3])) <= 1e-12 * float((b[1] * many["sums"][0, 1] * many["sums"][1, 1]).sqrt())
