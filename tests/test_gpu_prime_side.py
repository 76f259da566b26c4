"""Prime mesh sides whose single tile of rows does not fit LDS are deposited with global atomics:
every row of the mesh is written."""
import pytest
import torch

from jax_powspec_amd.mas import assign

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [127, 131, 257])
def test_every_row_is_written(n):
    dev = torch.device("cuda", 0)
    g = torch.Generator(device=dev)
    g.manual_seed(n)
    pos = torch.rand((30_000, 3), device=dev, generator=g) * (n - 1e-2)
    base = torch.ones((n, n, n), device=dev)
    got = assign(pos[:, 0], pos[:, 1], pos[:, 2], delta=base, box_size=float(n), n_bins=n, mas="CIC")
    want = assign(pos[:, 0], pos[:, 1], pos[:, 2], delta=base, box_size=float(n), n_bins=n, mas="CIC", tile="direct")
    # cells hold a few deposits of at most 1, added in another order
    torch.testing.assert_close(got, want, rtol=0, atol=2.0 ** -18)
    assert abs(float(got.double().sum()) - n ** 3 - 30_000) < 1.0
