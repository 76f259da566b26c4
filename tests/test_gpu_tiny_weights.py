"""Weights far below one: the fixed point's scale stays inside float32, so the mesh is that of weights 2^100 times as
large, scaled.  A weight keeps 26 bits there: 2^-25 of the largest weight for each of up to 100 deposits in a cell."""
import pytest
import torch

from jax_powspec_amd import mas

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("stencil", ["CIC_REF", "CIC", "TSC"])
def test_mesh_scales_with_the_weights(gpu, stencil):
    g = torch.Generator(device=gpu)
    g.manual_seed(4)
    n = 32
    p = torch.rand((30_000, 3), device=gpu, generator=g) * (n - 0.01)
    w = 0.5 + torch.rand(30_000, device=gpu, generator=g)
    want, got = (mas.assign(p[:, 0], p[:, 1], p[:, 2], w * s, box_size=float(n), n_bins=n, mas=stencil).double() / s
                 for s in (1.0, 2.0 ** -100))
    assert float((got - want).abs().max()) <= 100 * 1.5 * 2.0 ** -25
