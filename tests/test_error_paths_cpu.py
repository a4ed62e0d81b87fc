"""The solver's host code when a launch or an allocation fails, on the CPU: its
source linked with a stand-in for the GPU (host_stub.cpp) whose streams run only
when the host waits and whose calls fail on request.  After an error the same
call again gives what a context without the error gives."""
import ctypes
import importlib.util
import os
import subprocess

import pytest

import cases

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG_DIR = os.path.join(ROOT, "simple-ts_amd")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
TOL = (1e-9, 1e-9, 1e-9)


@pytest.fixture(scope="module")
def stub(tmp_path_factory):
    d = tmp_path_factory.mktemp("stub")
    lib = str(d / "libstub.so")
    objs = []
    for src in (os.path.join(PKG_DIR, "csrc", "sts_api.cpp"), os.path.join(ROOT, "tests", "host_stub.cpp")):
        objs.append(str(d / (os.path.basename(src) + ".o")))
        subprocess.run([HIPCC, "--offload-arch=gfx950", "-x", "hip", "-O1", "-std=c++17", "-fPIC", "-I",
                        os.path.join(ROOT, "include"), "-c", src, "-o", objs[-1]], check=True)
    subprocess.run([os.environ.get("CXX", "g++"), "-shared", "-Wl,-Bsymbolic", "-o", lib, *objs, "-lpthread"],
                   check=True)
    spec = importlib.util.spec_from_file_location("simple_ts_stub", os.path.join(PKG_DIR, "__init__.py"))
    pkg = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(pkg)
    pkg.LIB_HIP = lib
    return pkg


@pytest.fixture
def gpu(stub):
    L = ctypes.CDLL(stub.LIB_HIP)
    L.stub_clear()
    L.stub_stop(3)
    yield L
    L.stub_clear()


def context(pkg):
    c = cases.channel_case(40, 16)
    return pkg.Context(pkg.Problem(c.hx, c.hy, c.vol, c.bodies, c.boxes, c.scalars, c.given_xb, c.given_xe, c.kn_local,
                                   c.bc))


@pytest.mark.parametrize("call", ["plain", "mixed"])
def test_loop_after_a_failed_one(stub, gpu, call):
    """A launch fails with iterations of the loop in flight, one of which would end
    it: nothing of it is left when the next loop begins."""
    ctx = context(stub)
    step = (lambda: ctx.time_step(20, 2, *TOL, batch=4, wait=False)[0]) if call == "plain" else \
        (lambda: ctx.time_step_mixed(20, 2, *TOL, 0, TOL, batch=4, wait=False)[1])
    assert step() == 3
    gpu.stub_fail(b"launch_edges", 4)
    with pytest.raises(stub.StsError):
        step()
    gpu.stub_stop(6)
    assert step() == 6


def starts(gpu, step, n):
    """The degrees of the starts of n steps."""
    first = gpu.stub_begins()
    for _ in range(n):
        step()
    assert all(gpu.stub_whole(q) for q in range(first, gpu.stub_begins()))
    return [gpu.stub_order(q) for q in range(first, gpu.stub_begins())]


@pytest.mark.parametrize("call,n", [("launch_begin", 1), ("hipMalloc", 6)])
def test_predicted_start_after_a_failed_one(stub, gpu, call, n):
    """A start that was not made counts for no step of the history, and an
    allocation that failed is made good."""
    ctx = context(stub)

    def step(degree=3):
        ctx.time_step_mixed(20, 2, *TOL, 0, TOL, extrapolate=degree, wait=False)

    step(0)  # the loops' own buffers
    gpu.stub_fail(call.encode(), n)
    with pytest.raises(stub.StsError):
        step()
    assert starts(gpu, step, 5) == [0, 1, 2, 3, 3]


@pytest.mark.parametrize("call,n", [("launch_batch_begin", 1), ("hipMalloc", 26)])
def test_batched_starts_after_a_failed_one(stub, gpu, call, n):
    """As above for two cases; the 26th allocation is one of the second case's."""
    batch = stub.Batch([context(stub) for _ in range(2)])

    def step(degree=3):
        batch.time_step(20, 2, *TOL, mixed=(0, TOL, 0, 0.95, degree))

    step(0)
    gpu.stub_fail(call.encode(), n)
    with pytest.raises(stub.StsError):
        step()
    assert starts(gpu, step, 5) == [0, 0, 1, 1, 2, 2, 3, 3, 3, 3]
