"""The dynamic-LDS limit of a kernel belongs to one device: a process that uses several raises it on each.  The host
code runs against a HIP runtime that runs nothing (fake_hip.cpp), in a process of its own."""
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)

PRELUDE = """
import ctypes as C, sys, types
fake = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
pkg = types.ModuleType("jax_powspec_amd")
pkg.__path__ = [sys.argv[2] + "/jax-powspec_amd"]
sys.modules["jax_powspec_amd"] = pkg
from jax_powspec_amd import _lib
lib = _lib.load()
P = 4096                     # stands for every device pointer; nothing reads it
ok = lambda r: r == 0 or sys.exit(lib.pk_last_error())
"""

PROGRAM = """
def run(device, n, nb, stencil):
    fake.fake_set_device(device)
    plan, need = C.c_void_p(), C.c_size_t()
    ok(lib.pk_plan_create(n, C.byref(plan)))
    ok(lib.pk_powspec_workspace_size(plan, nb, C.byref(need)))
    ok(lib.pk_powspec_mesh(plan, P, None, P, P, P, P, nb, 2, 0, 1.0, 0.0, P, P, P, P, P, None, P, need.value, None))
    ok(lib.pk_estimate_workspace_size(plan, 100000, stencil, None, nb, C.byref(need)))
    ok(lib.pk_estimate(plan, P, 3, P + 4, 3, P + 8, 3, None, 1, 100000, 0.0, 0.0, 0.0, 1.0, stencil, 0, None, P, P, P,
                       P, nb, 2, 0, 0.0, P, P, P, P, None, P, P, need.value, None))
    ok(lib.pk_scatter_workspace_size(n, 100000, stencil, None, C.byref(need)))
    ok(lib.pk_scatter(P, 3, P + 4, 3, P + 8, 3, None, 1, 100000, 0.0, 0.0, 0.0, 1.0, n, stencil, 0, None, None, P, P, P,
                      need.value, None))
    ok(lib.pk_batch_workspace_size(plan, 1, 100000, nb, None, C.byref(need)))
    b, job = C.c_void_p(), _lib.PkJob()
    ok(lib.pk_batch_create(plan, 1, 100000, nb, None, 0, P, need.value, C.byref(b)))
    for f in ("x", "y", "z", "thr", "jstart", "modes", "ksum", "sums", "counts", "pk", "nmodes", "stats"):
        setattr(job, f, P)
    job.sx = job.sy = job.sz = job.sw = 1
    job.np, job.box_size, job.stencil, job.window_p, job.nb = 100000, 1.0, stencil, 2, nb
    ok(lib.pk_batch_set_jobs(b, 1, C.byref(job), None))
    ok(lib.pk_batch_run(b, None))
for device in (0, 1, 0, 1):
    for n, nb in ((512, 300), (512, 1000), (1024, 100), (384, 300), (256, 100)):
        for stencil in (0, 2):
            run(device, n, nb, stencil)
"""




def lines_of(program, folder):
    """what a program prints that runs after PRELUDE"""
    lib = str(folder / "libfake_hip.so")
    subprocess.run(["g++", "-O1", "-shared", "-fPIC", os.path.join(HERE, "fake_hip.cpp"), "-o", lib], check=True)
    r = subprocess.run([sys.executable, "-c", PRELUDE + program, lib, ROOT], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stderr
    return r.stdout.splitlines()


def test_every_device_raises_the_limits(tmp_path):
    limit, launches = {}, 0
    for line in lines_of(PROGRAM, tmp_path):
        what, device, value, kernel = line.split(" ", 3)
        if what == "attribute":
            assert int(value) > limit.get((device, kernel), 0), f"set again: {kernel}"
            limit[device, kernel] = int(value)
        elif int(value) > 65536:
            launches += 1
            assert limit.get((device, kernel), 0) >= int(value), f"device {device}: {kernel}"
    assert launches > 0
    kernels = {d: {k for dev, k in limit if dev == d} for d in "01"}
    assert kernels["0"] == kernels["1"]
    # the binning x pass has most of its LDS in static arrays: below 64 KB of dynamic ones it is raised too
    assert any("k_xpass_binI" in k for k in kernels["1"]) and any("k_xpass_bin_jobsI" in k for k in kernels["1"])
