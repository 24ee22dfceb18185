"""Residual-only plans hold the tables that their kernel reads and no others: the device memory that a plan reports, by
kind of plan. Without a GPU, on the stand-in of hip_stub.cpp, in a process of its own."""

import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))


def body(stub_path, pkg):
    import ctypes

    stub = ctypes.CDLL(stub_path, mode=ctypes.RTLD_GLOBAL)
    stub.stub_used.restype = ctypes.c_size_t
    sys.path.insert(0, pkg)
    import fem_amd as F

    for order in (1, 2, 3, 4):
        m = F.square_mesh(60, order, jitter=0.2, seed=1)
        pat = F.bsr_pattern(m)
        before = stub.stub_used()
        line = F.Plan(m, pat, flags=F.FEM_PLAN_RESIDUAL_ONLY)
        i = line.info()
        assert stub.stub_used() - before == i["device_bytes"]
        # a node id and a 16-bit row per visited node, the rows, eight ints per part; a few bytes where a table is empty
        assert i["device_bytes"] <= 6 * m.npe * i["element_visits"] + 4 * m.num_nodes + 32 * i["parts"] + 64, (order, i)
        det = F.Plan(m, pat, flags=F.FEM_PLAN_RESIDUAL_ONLY | F.FEM_PLAN_DETERMINISTIC).info()
        # node and element ids of the visits, ranks, three ints per node, runs of four, descriptors, a few colours
        visits, pad = det["element_visits"], (m.npe + 3) // 4 * 4
        most = (4 * m.npe + 4) * visits + m.npe * pad * m.num_elements + 28 * m.num_nodes + 128 * det["parts"] + 64
        assert det["device_bytes"] <= most, (order, det, most)
        line.close()
        assert stub.stub_used() >= before
    print("ok", flush=True)
    os._exit(0)


def test_residual_only_tables(tmp_path):
    out = str(tmp_path / "hip_stub.so")
    subprocess.run(["g++", "-O1", "-shared", "-fPIC", "-o", out, os.path.join(HERE, "hip_stub.cpp")], check=True)
    pkg = os.path.join(os.path.dirname(HERE), "gpu-fem-project_amd")
    r = subprocess.run([sys.executable, os.path.abspath(__file__), out, pkg], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout + r.stderr


if __name__ == "__main__":
    body(*sys.argv[1:])
