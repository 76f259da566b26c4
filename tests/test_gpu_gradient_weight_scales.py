"""The gradient does not depend on the unit of the weights: dP/dp stays as it is and dP/dw goes as its inverse,
also where squares of the density's modes leave float32's range (weights of 1e20, of 1e-25)."""
import numpy as np
import pytest
import torch

from jax_powspec_amd import autodiff

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [16, 48, 64, 256])
@pytest.mark.parametrize("stencil", ["CIC_REF", "TSC"])
def test_weight_units_cancel(gpu, n, stencil):
    rng = np.random.default_rng(n)
    box, np_ = 8.0 * n, 20_000
    p = torch.as_tensor(rng.random((np_, 3), dtype=np.float32) * np.float32(box * 0.999999), device=gpu)
    w = torch.as_tensor((0.5 + rng.random(np_)).astype(np.float32), device=gpu)
    edges = 2 * np.pi / box * np.linspace(0.6, n / 2 + 0.3, 9)

    def gradient(unit):
        tp, tw = p.clone().requires_grad_(True), (w * unit).requires_grad_(True)
        _, pk, _ = autodiff.estimate_ad(tp, tw, box_size=box, n_bins=n, k_edges=edges, mas=stencil)
        pk.backward(torch.ones_like(pk))   # whatever the values of P: the sums of squares overflow as well
        return tp.grad.double(), tw.grad.double() * unit

    want = gradient(1.0)
    for unit in (2.0 ** 66, 2.0 ** 40, 2.0 ** -40, 2.0 ** -83):   # powers of two: the density scales exactly
        for got, ref in zip(gradient(unit), want):
            assert float((got - ref).norm() / ref.norm()) <= 1e-6, unit
