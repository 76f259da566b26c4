"""Tiles of few rows have more keys than the count kernel's LDS table holds: it then counts x
planes, and the keys are counted per plane afterwards.  Owner-computes deposits sum in fixed
point, so the mesh equals that of the default tiles (whose keys fit) bit for bit."""
import numpy as np
import pytest
import torch

from jax_powspec_amd.mas import assign

pytestmark = pytest.mark.gpu

N = 256   # 2-row tiles: 65537 keys (98305 for TSC) against 36864 that fit


def _catalogue(kind, dev, count=60_001):
    g = torch.Generator(device=dev)
    g.manual_seed(11)
    pos = torch.rand((count, 3), device=dev, generator=g) * (N - 1e-3)
    if kind == "slab":          # every record in one x plane: all other planes are empty
        pos[:, 0] = 7.0 + pos[:, 0] / (2 * N)
    elif kind == "ends":        # first and last planes, rows at both edges of the mesh
        pos[:, 0] = torch.where(pos[:, 0] < N / 2, pos[:, 0] / N, N - 1e-2 - pos[:, 0] / N)
        pos[::3, 1] = N - 1e-2
        pos[1::3, 1] = 1e-2
    elif kind == "one":
        pos = pos[:1]
    return pos


@pytest.mark.parametrize("mas", ["CIC_REF", "CIC", "TSC"])
@pytest.mark.parametrize("kind", ["uniform", "slab", "ends", "one"])
@pytest.mark.parametrize("weighted,aos", [(False, True), (True, False)])
def test_small_tiles_give_the_same_mesh(mas, kind, weighted, aos):
    dev = torch.device("cuda", 0)
    pos = _catalogue(kind, dev)
    x, y, z = (pos[:, a] if aos else pos[:, a].contiguous() for a in range(3))
    w = torch.linspace(-0.5, 2.0, pos.shape[0], device=dev) if weighted else None
    kw = dict(box_size=float(N), n_bins=N, mas=mas)
    assert torch.equal(assign(x, y, z, w, tile=(1, 2, 0), **kw), assign(x, y, z, w, **kw))


def test_particles_outside_the_mesh():
    """Dropped and irregular records keep their place in the order of the planes."""
    dev = torch.device("cuda", 0)
    pos = _catalogue("uniform", dev)
    pos[::7, 0] = -1.5
    pos[1::7, 2] = N + 0.5
    pos[2::7, 1] = float("nan")
    kw = dict(box_size=float(N), n_bins=N, mas="CIC_REF")
    got = assign(pos[:, 0], pos[:, 1], pos[:, 2], tile=(1, 2, 0), **kw)
    want = assign(pos[:, 0], pos[:, 1], pos[:, 2], **kw)
    # the irregular records are added with float atomics, in any order
    np.testing.assert_allclose(got.cpu().numpy(), want.cpu().numpy(), rtol=0, atol=2.0 ** -20)
