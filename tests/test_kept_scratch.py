"""An allocation that fails while the pattern builders keep idle scratch has it freed and is tried again: plans, batches
and the server get memory that only that scratch holds. Without a GPU: the HIP runtime is the stand-in of hip_stub.cpp,
whose device memory has a limit, in a process of its own."""

import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


def scratch_kept(stub, F, np):
    """Builds a pattern of four million nodes (the stand-in's kernels read nothing); returns the bytes left allocated."""
    before = stub.stub_used()
    rowp, blocks = np.zeros(1, np.int32), F.ctypes.c_int64()
    P = F._ptr(rowp)
    assert F.load().fem_bsr_pattern_device(4000000, 1000000, 9, P, P, P, None, 0, F.ctypes.byref(blocks), None) == 0
    return stub.stub_used() - before


def body(stub_path, pkg, what):
    import ctypes

    stub = ctypes.CDLL(stub_path, mode=ctypes.RTLD_GLOBAL)
    stub.stub_used.restype = ctypes.c_size_t
    stub.stub_limit.argtypes = [ctypes.c_size_t]
    sys.path.insert(0, pkg)
    import fem_amd as F
    import numpy as np

    plans = {"plan-1": (1, 0), "plan-3": (3, 0), "residual": (2, F.FEM_PLAN_RESIDUAL_ONLY), "tuned": (4, F.FEM_PLAN_AUTOTUNE)}
    order, flags = plans.get(what, (3, 0))
    m = F.square_mesh(40, order, jitter=0.2, seed=1)
    pat = F.bsr_pattern(m)
    if what in plans:
        def use():
            F.Plan(m, pat, flags=flags).close()
    elif what == "batch":
        def use():
            F.Batch(max_jobs=4096).close()
    elif what == "arena":
        plan, batch = F.Plan(m, pat), F.Batch(max_jobs=4)
        out = np.zeros(4 * pat.num_blocks)

        def use():
            P = F._ptr
            assert F.load().fem_batch_add(batch.handle, plan.handle, P(m.coords), P(m.coords), 1.0, 0.3, 1.0, None,
                                          P(out)) == 0
            F._check(F.load().fem_batch_assemble(batch.handle, 0, None, None))
    else:
        srv = F.Server(budget_bytes=1 << 30, max_batch_jobs=2, slots=1)

        def use():
            (srv.reserve(8 << 20) if what == "reserve" else srv.add_mesh(m, 1.0, 0.3, 1.0))

    kept = scratch_kept(stub, F, np)
    assert kept > 96 << 20, kept
    stub.stub_limit(stub.stub_used() + 1000)  # no room but the scratch
    use()
    # and without scratch the failure is reported
    stub.stub_limit(0)
    try:
        F.Batch(max_jobs=4096)
    except F.FemError:
        print("ok", flush=True)
    os._exit(0)


@pytest.fixture(scope="module")
def stub(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("hip") / "hip_stub.so")
    subprocess.run(["g++", "-O1", "-shared", "-fPIC", "-o", out, os.path.join(HERE, "hip_stub.cpp")], check=True)
    return out


@pytest.mark.parametrize("what", ["plan-1", "plan-3", "residual", "tuned", "batch", "arena", "reserve", "mesh"])
def test_allocation_with_scratch_kept(stub, what):
    pkg = os.path.join(os.path.dirname(HERE), "gpu-fem-project_amd")
    r = subprocess.run([sys.executable, os.path.abspath(__file__), stub, pkg, what], capture_output=True, text=True,
                       timeout=120)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout + r.stderr


if __name__ == "__main__":
    body(*sys.argv[1:])
