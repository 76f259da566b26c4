"""The adjoint's passes at mesh sides of every radix plan, with bin tables in LDS and in HBM: the
gradient against the FP64 oracle, within 1e-3 in the 2-norm (float32 mesh, transforms and gather).
The box has cells of side 8, so that float32 scaled positions are exact."""
import numpy as np
import pytest
import torch

from jax_powspec_amd import autodiff
from oracle import ref_fp64 as R
from test_gpu_parity import catalogue

pytestmark = pytest.mark.gpu


# (side, bins): more than 256 bins are looked up in HBM; most of those are empty at 24
@pytest.mark.parametrize("n,nb", [(8, 4), (12, 6), (16, 8), (24, 300), (48, 24), (64, 256), (64, 257), (96, 48),
                                  (128, 64)])
@pytest.mark.parametrize("stencil", ["CIC_REF", "TSC"])
def test_gradient_matches_oracle(gpu, n, nb, stencil):
    rng = np.random.default_rng(n + nb)
    box = 8.0 * n
    p = catalogue(rng, 6000, box, edges=False)
    w = (0.5 + rng.random(len(p))).astype(np.float32)
    edges = 2 * np.pi / box * np.linspace(0.6, n / 2 + 0.3, nb + 1)
    tp = torch.as_tensor(p, device=gpu).requires_grad_(True)
    tw = torch.as_tensor(w, device=gpu).requires_grad_(True)
    _, pk, _ = autodiff.estimate_ad(tp, tw, box_size=box, n_bins=n, k_edges=edges, mas=stencil)
    full = ~torch.isnan(pk)
    c = torch.where(full, torch.as_tensor(rng.standard_normal(tuple(pk.shape)), dtype=torch.float32, device=gpu), 0.0)
    torch.where(full, pk * c, 0.0).sum().backward()
    wp, ww = R.estimate_backward(*p.T, w, box, n, edges, c.cpu().numpy().astype(np.float64), stencil=stencil,
                                 p=3 if stencil == "TSC" else 2)
    for got, want in ((tp.grad, wp), (tw.grad, ww)):
        err = np.linalg.norm(got.cpu().numpy().astype(np.float64) - want) / np.linalg.norm(want)
        assert err <= 1e-3, err
