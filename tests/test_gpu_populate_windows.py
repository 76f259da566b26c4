"""Dense fields: a block of 4096 cells lists its particles' cells 4096 slots at a time, and cells of 255
particles and more are counted again.  Whole catalogues against the oracle, in order."""
import numpy as np
import pytest
import torch

from jax_powspec_amd import gauss_field
from oracle import mocks

pytestmark = pytest.mark.gpu


# particles per cell: below one window per block, several windows, counts around the stored
# byte's end, all of them beyond it; odd sides end inside a thread's 16 cells
@pytest.mark.parametrize("n,rate", [(16, 0.9), (17, 1.1), (24, 5.0), (18, 40.0), (9, 255.0), (16, 300.0), (33, 0.02)])
def test_catalogue_equals_the_oracle(n, rate):
    rng = np.random.default_rng(n)
    rho = (0.9 + 0.2 * rng.random((n, n, n))).astype(np.float32)
    box = 2.0 * n
    pos = gauss_field.populate_field(torch.as_tensor(rho, device="cuda"), n, box, rate / 8.0, 3).cpu().numpy()
    want, counts = mocks.populate(rho, n, box, rate / 8.0, 3)
    assert pos.shape == want.shape and counts.sum() == pos.shape[0]
    assert np.abs(pos.astype(np.float64) - want).max() <= 1e-6 * box   # float32 positions
