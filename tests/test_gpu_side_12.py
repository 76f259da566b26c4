"""Mesh side 12, whose tiles hold 144 cells: the fused deposit's blocks are whole waves, so the mass
and the power of the estimate are those of the separate assignment and transform."""
import numpy as np
import pytest
import torch

from jax_powspec_amd import correlations, mas

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scheme", ["CIC_REF", "CIC", "TSC"])
def test_estimate_equals_the_mesh_path(scheme):
    dev = torch.device("cuda", 0)
    g = torch.Generator(device=dev)
    g.manual_seed(12)
    pos = torch.rand((5000, 3), device=dev, generator=g) * 95.9
    edges = 2 * np.pi / 96.0 * (0.5 + np.arange(7))
    _, pk, modes = correlations.estimate(pos[:, 0], pos[:, 1], pos[:, 2], box_size=96.0, n_bins=12, k_edges=edges,
                                         mas=scheme)
    rho = mas.assign(pos[:, 0], pos[:, 1], pos[:, 2], box_size=96.0, n_bins=12, mas=scheme).double()
    window = "TSC" if scheme == "TSC" else "CIC"
    _, want, want_modes = correlations.powspec_vec((rho / rho.mean() - 1).float(), 96.0, edges, mas=window)
    assert torch.equal(modes, want_modes)
    # float32 transforms of the same mesh, up to its rounding: 1e-5 of the monopole's scale
    assert bool(((pk - want).abs() <= 1e-5 * 9 * want[:, :1]).all()), (pk - want).abs().max()
