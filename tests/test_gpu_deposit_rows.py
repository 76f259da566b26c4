"""The mesh deposit's flush: 16-byte accesses where the mesh side and both pointers allow them, 4-byte
ones elsewhere, into a separate mesh or in place.  The same integers reach every cell."""
import pytest
import torch

from jax_powspec_amd.mas import assign

pytestmark = pytest.mark.gpu


def _offset(t, by):
    """A copy of t whose data starts `by` floats after a 512-byte boundary."""
    buf = torch.empty(t.numel() + 128, dtype=torch.float32, device=t.device)
    v = buf[by:by + t.numel()].view(t.shape)
    v.copy_(t)
    return v


@pytest.mark.parametrize("n", [6, 30, 32, 96, 127])
@pytest.mark.parametrize("scheme", ["CIC_REF", "TSC"])
@pytest.mark.parametrize("count", [0, 1, 20_000])
def test_alignment_and_aliasing(n, scheme, count):
    dev = torch.device("cuda", 0)
    g = torch.Generator(device=dev)
    g.manual_seed(n + count)
    pos = torch.rand((count, 3), device=dev, generator=g) * (n - 1e-2)
    w = torch.rand(count, device=dev, generator=g)
    base = torch.randn((n, n, n), device=dev, generator=g)
    kw = dict(box_size=float(n), n_bins=n, mas=scheme)
    x, y, z = pos[:, 0], pos[:, 1], pos[:, 2]
    alone = assign(x, y, z, w, **kw)
    want = base + alone   # one float32 addition per cell
    assert torch.equal(assign(x, y, z, w, delta=base, **kw), want)
    out = _offset(torch.zeros_like(base), 1)
    assign(x, y, z, w, delta=base, out=out, **kw)
    assert torch.equal(out, want)
    out = torch.zeros_like(base)
    assign(x, y, z, w, delta=_offset(base, 3), out=out, **kw)
    assert torch.equal(out, want)
    for by in (0, 1):   # in place
        mesh = _offset(base, by)
        assign(x, y, z, w, delta=mesh, out=mesh, **kw)
        assert torch.equal(mesh, want)
