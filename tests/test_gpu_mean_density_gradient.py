"""The gradient's term for the mean density, which comes from a sum over the modes in the adjoint's x pass.

Weights multiplied by a common factor leave P(k) as it is, so sum_i w_i dL/dw_i = 0, where the mean's term
alone is -2 L for L = sum_b P_0(b) (no shot noise subtracted).  Transforms, mesh and gather in float32 leave
about 1e-6 of sum_i |w_i dL/dw_i|; 1e-5 is allowed, and the catalogues are such that the mean's term
a thousandth off would be twice that."""
import numpy as np
import pytest
import torch

from jax_powspec_amd import autodiff
from oracle import ref_fp64 as R

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,nb", [(8, 4), (12, 6), (16, 8), (24, 300), (32, 16), (48, 24), (64, 32), (64, 257), (96, 48), (128, 64),
                                  (192, 96), (256, 128), (384, 64)])
@pytest.mark.parametrize("stencil", ["CIC_REF", "CIC", "TSC"])
def test_a_common_factor_of_the_weights_changes_nothing(gpu, n, nb, stencil):
    rng = np.random.default_rng(n + nb)
    box, np_ = 8.0 * n, min(8 * n ** 3, 400_000)
    p = torch.as_tensor(rng.random((np_, 3), dtype=np.float32) * np.float32(box * 0.999999), device=gpu).requires_grad_(True)
    w = torch.as_tensor((0.5 + rng.random(np_)).astype(np.float32), device=gpu).requires_grad_(True)
    edges = 2 * np.pi / box * np.linspace(0.6, n / 2 + 0.3, nb + 1)
    _, pk, _ = autodiff.estimate_ad(p, w, box_size=box, n_bins=n, k_edges=edges, mas=stencil)
    loss = torch.nan_to_num(pk[:, 0]).sum()
    loss.backward()
    terms = (w.detach() * w.grad).double()
    total = float(terms.abs().sum())
    assert 2 * float(loss) >= 0.02 * total, "the mean's term is too small to be seen"
    assert abs(float(terms.sum())) <= 1e-5 * total, float(terms.sum()) / total


@pytest.mark.parametrize("n,nb,np_", [(16, 8, 6000), (48, 24, 100_000), (64, 257, 200_000), (128, 64, 200_000)])
@pytest.mark.parametrize("stencil", ["CIC_REF", "TSC"])
def test_gradient_to_float32(gpu, n, nb, np_, stencil):
    # box and positions in which float32 scaled positions are exact; 1e-5 in the 2-norm: four float32 stages
    # (mesh, two transforms, gather) of a few 2^-24 each, times log2(n) in the transforms
    rng = np.random.default_rng(2 * n + nb)
    box = 8.0 * n
    p = rng.random((np_, 3), dtype=np.float32) * np.float32(box * 0.999999)
    w = (0.5 + rng.random(np_)).astype(np.float32)
    edges = 2 * np.pi / box * np.linspace(0.6, n / 2 + 0.3, nb + 1)
    tp = torch.as_tensor(p, device=gpu).requires_grad_(True)
    tw = torch.as_tensor(w, device=gpu).requires_grad_(True)
    _, pk, _ = autodiff.estimate_ad(tp, tw, box_size=box, n_bins=n, k_edges=edges, mas=stencil)
    torch.nansum(pk).backward()
    c = np.where(np.isnan(pk.detach().cpu().numpy()), 0.0, 1.0)
    wp, ww = R.estimate_backward(*p.T, w, box, n, edges, c, stencil=stencil, p=3 if stencil == "TSC" else 2)
    for got, want in ((tp.grad, wp), (tw.grad, ww)):
        err = np.linalg.norm(got.cpu().numpy().astype(np.float64) - want) / np.linalg.norm(want)
        assert err <= 1e-5, err
