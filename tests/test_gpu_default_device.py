"""Programs that make their tensors on the GPU by default (torch.set_default_device): every entry point that sends
host tables to the device gives what it gives without."""
import numpy as np
import pytest
import torch

from jax_powspec_amd import autodiff, batch, correlations, gauss_field

pytestmark = pytest.mark.gpu

N, BOX = 32, 500.0
KF = np.geomspace(1e-3, 10.0, 200)


def calls(pos, mesh):
    edges = 2 * np.pi / BOX * (0.5 + np.arange(N // 2 + 1))
    x, y, z = pos[:, 0], pos[:, 1], pos[:, 2]
    cat = dict(x=x, y=y, z=z, box_size=BOX, n_bins=N, k_edges=edges)
    yield "estimate", lambda: correlations.estimate(x, y, z, box_size=BOX, n_bins=N, k_edges=edges)
    yield "powspec_vec", lambda: correlations.powspec_vec(mesh, BOX, edges)
    yield "xi_vec", lambda: correlations.xi_vec(mesh, BOX, np.linspace(0.0, 200.0, 9))
    yield "bispec", lambda: correlations.bispec(mesh, BOX, 0.05, 0.08, np.linspace(0.3, 2.8, 6))
    yield "estimate_ad", lambda: autodiff.estimate_ad(pos, box_size=BOX, n_bins=N, k_edges=edges)
    yield "batch", lambda: batch.powspec_batched([cat, cat], tile=None)[1]
    yield "gaussian_mesh", lambda: (gauss_field.gaussian_mesh(N, KF, 1e3 * KF ** -1.0, 0, 3, BOX),)


def test_results_do_not_depend_on_the_default_device(gpu):
    g = torch.Generator(device=gpu)
    g.manual_seed(2)
    pos = torch.rand((20000, 3), device=gpu, generator=g) * (BOX - 0.01)
    mesh = torch.randn((N, N, N), device=gpu, generator=g)
    want = {name: call() for name, call in calls(pos, mesh)}
    torch.set_default_device(gpu)
    try:
        got = {name: call() for name, call in calls(pos, mesh)}
    finally:
        torch.set_default_device(None)
    for name in want:
        for a, b in zip(got[name], want[name]):
            assert torch.equal(torch.nan_to_num(a), torch.nan_to_num(b)), name
