"""Population of dense and of very uneven fields: every way a block of cells is emitted, in one field, whole
catalogues against the oracle in order; and the particles per second that dense fields keep."""
import ctypes as C
import time

import numpy as np
import pytest
import torch

from jax_powspec_amd import _device, _lib, gauss_field
from oracle import mocks

pytestmark = pytest.mark.gpu


def fields():
    rng = np.random.default_rng(5)
    # 16 consecutive cells hold 32 particles on average: blocks on both sides of the limit
    yield "about 32 in 16 cells", (0.95 + 0.1 * rng.random((24, 24, 24))).astype(np.float32), 2.0
    # sparse blocks, dense ones, one with a cell of thousands and one with a cell beyond 16 windows of 4096
    rho = np.full(24 ** 3, 0.2, np.float32)
    rho[4096:6000] = 20.0
    rho[5000] = 9000.0
    rho[8192] = 200.0
    rho[-3] = 100000.0
    yield "uneven", rho.reshape(24, 24, 24), float(rho.mean())
    # one cell holds nearly all, most blocks nothing; odd side, the last block ends inside 16 cells
    rho = np.zeros(17 ** 3, np.float32)
    rho[4500] = 30000.0
    rho[[0, 15, 16, 4095, 4096, 4912]] = [1.0, 254.0, 255.0, 256.0, 31.0, 33.0]
    yield "one cell", rho.reshape(17, 17, 17), float(rho.mean())


@pytest.mark.parametrize("k", range(3))
def test_catalogue_equals_the_oracle(k):
    name, rho, rate = list(fields())[k]
    n = rho.shape[0]
    box = 2.0 * n
    pos = gauss_field.populate_field(torch.as_tensor(rho, device="cuda"), n, box, rate / 8.0, 3).cpu().numpy()
    want, counts = mocks.populate(rho, n, box, rate / 8.0, 3)
    assert pos.shape == want.shape and counts.sum() == pos.shape[0], name
    assert np.abs(pos.astype(np.float64) - want).max() <= 1e-6 * box, name   # float32 positions


def test_capacity_below_the_total_gives_the_first_particles():
    _, rho, rate = list(fields())[1]
    n, dev = rho.shape[0], torch.device("cuda", 0)
    box = 2.0 * n
    field = torch.as_tensor(rho, device=dev)
    whole = gauss_field.populate_field(field, n, box, rate / 8.0, 3)
    lib, nbytes = _lib.load(), C.c_size_t()
    _lib.check("size", lib.pk_populate_workspace_size(n, C.byref(nbytes)))
    ws = _device.workspace(nbytes.value, dev)
    total = torch.zeros(1, dtype=torch.int64, device=dev)
    stream = _device.stream_ptr(dev)
    _lib.check("count", lib.pk_populate_count(_device.ptr(field), n, box, rate / 8.0, 0.0, 3, _device.ptr(ws),
                                              nbytes.value, _device.ptr(total), stream))
    assert int(total) == whole.shape[0]
    for cap in (1, 700, 4096, int(total) // 2, int(total) - 1):
        pos = torch.full((cap + 64, 3), -1.0, device=dev)
        _lib.check("place", lib.pk_populate_place(_device.ptr(field), None, 0.0, n, box, 0.0, 3, _device.ptr(ws),
                                                  nbytes.value, _device.ptr(pos), cap, stream))
        assert torch.equal(pos[:cap], whole[:cap]) and bool((pos[cap:] == -1.0).all()), cap


@pytest.mark.parametrize("rate", [40.0, 300.0])
def test_dense_fields_are_not_emitted_by_single_threads(rate):
    # marking every slot's cell first (one kernel) and emitting a particle per thread (another) gave 26 and 33
    # particles per us here; a thread listing each of its particles gave 8.6 and 2.2
    n = 64
    g = torch.Generator(device="cuda")
    g.manual_seed(1)
    rho = 0.5 + torch.rand((n, n, n), device="cuda", generator=g)
    best = np.inf
    for _ in range(5):
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        pos = gauss_field.populate_field(rho, n, float(n), rate, 3)
        torch.cuda.synchronize()
        best = min(best, time.perf_counter() - t0)
    assert pos.shape[0] / best / 1e6 >= 20.0
