"""The reference stencil left of the box: truncation towards zero gives corner weights of up to 2 per axis there
(1 - dd with dd < 0), 8 in a corner.  Mesh and P_l against the FP64 oracle; the box has cells of side 8, so that float32
scaled positions are exact.  Bounds: float32 rounding of a few deposits per cell, and of the transforms."""
import numpy as np
import pytest
import torch

from jax_powspec_amd import batch, correlations, mas
from oracle import ref_fp64 as R

pytestmark = pytest.mark.gpu


def moved(rng, n, how):
    box = 8.0 * n
    p = (rng.random((20_000, 3)) * (box - 0.01)).astype(np.float32)
    k = rng.random(len(p)) < 0.2
    if how == "edge":       # up to a cell to the left: base cell 0 on that axis
        p[k] = -8.0 * rng.random((k.sum(), 3)).astype(np.float32)
        p[k & (rng.random(len(p)) < 0.5), 1] = 5.0
    else:                   # anywhere left of the box: base cells below 0
        p[k] -= np.float32(0.7 * box)
    return p, (0.5 + rng.random(len(p))).astype(np.float32), box


@pytest.mark.parametrize("how", ["edge", "left"])
@pytest.mark.parametrize("n", [24, 64, 128])
def test_mesh_and_spectrum_match_the_oracle(gpu, n, how):
    rng = np.random.default_rng(n)
    p, w, box = moved(rng, n, how)
    t, tw = torch.as_tensor(p, device=gpu), torch.as_tensor(w, device=gpu)
    mesh = mas.assign(t[:, 0], t[:, 1], t[:, 2], tw, box_size=box, n_bins=n).cpu().numpy().astype(np.float64)
    want = np.zeros(n ** 3)
    for flat, valid, W, _ in R.corner_stencil("CIC_REF", [p[:, i].astype(np.float64) / 8.0 for i in range(3)], n):
        want += np.bincount(flat[valid], weights=(w * W)[valid], minlength=n ** 3)
    assert np.abs(mesh.ravel() - want).max() <= 1e-6 * np.abs(want).max()
    edges = 2 * np.pi / box * np.linspace(0.6, n / 2 + 0.3, 9)
    _, pk, _ = correlations.estimate(t[:, 0], t[:, 1], t[:, 2], tw, box_size=box, n_bins=n, k_edges=edges)
    ref = R.estimate(*p.T, w, box, n, edges, stencil="CIC_REF")
    scale = ref[3]["scale"]
    assert np.nanmax(np.abs(pk.cpu().numpy().astype(np.float64) - ref[1]) / scale) <= 1e-5
    cat = dict(x=t[:, 0], y=t[:, 1], z=t[:, 2], w=tw, box_size=box, n_bins=n, k_edges=edges)
    assert torch.equal(batch.powspec_batched([cat], tile=None)[0][1], pk)
