"""Graph batches on the device: every assembly of a composition (launched directly, recorded, replayed, replayed after a
refill with other buffers and states, in turn with another composition) against the oracle, with the caller's own work
and synchronisation in between, on the default and on another stream. FP64 bar 1e-12; mixed 1e-5 (residual 1e-12); jobs
of orders 3-4 bit for bit as the plan assembled alone. Preparing a batch
(fem::batch_prepare, the server's) that holds jobs touches none of them."""

import ctypes

import numpy as np
import pytest

import textbook

pytestmark = pytest.mark.gpu

E, NU, T = 70e9, 0.3, 1.0
MESHES = [(1, 40, 31), (2, 33, 30), (3, 14, 9), (4, 11, 6), (1, 3, 3), (3, 1, 1), (2, 150, 151)]
# (mesh, with residual, with values)
A = [(0, True, True), (1, True, True), (2, True, True), (3, False, True), (4, True, False), (5, True, True)]
B = [(1, False, True), (4, True, True), (3, True, False), (3, True, True)]
C = [(6, True, True), (2, False, True), (2, True, False)]
FULL = [(i, True, vals) for i in range(4) for vals in (True, False)]  # the server's kinds
D = FULL + [(i, False, True) for i in range(4)]


@pytest.fixture(scope="module")
def cases(fem, orc):
    out = []
    for order, nx, ny in MESHES:
        m = fem.square_mesh(nx, order, jitter=0.2, seed=nx, ny=ny)
        pat = fem.bsr_pattern(m)
        u = fem.fill_uniform(2 * m.num_nodes, -1e-3, 1e-3, 5)
        res, vals = orc.jacobian(m, u, E, NU, T, fem.element_bcsr_map(m, pat), pat.num_blocks)
        out.append(dict(mesh=m, pat=pat, u=u, res=res, vals=vals))
    return out


class Filled:
    """Jobs on a batch, with buffers of their own; LINEAR strain: R(s u) = s R(u), K does not depend on u."""

    def __init__(self, torch, batch, cases, plans, which, scale):
        on = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()  # noqa: E731
        nan = lambda n: torch.full((n,), float("nan"), dtype=torch.float64, device="cuda")  # noqa: E731
        self.torch, self.jobs = torch, []
        batch.clear()
        for i, with_res, with_vals in which:
            c = cases[i]
            st, co = on(scale * c["u"]), on(c["mesh"].coords)
            res = nan(2 * c["mesh"].num_nodes) if with_res else None
            vals = nan(4 * c["pat"].num_blocks) if with_vals else None
            batch.add(plans[i], st, co, E, NU, T, res=res, values=vals)
            self.jobs.append((c, plans[i], scale, st, co, res, vals))
        torch.cuda.synchronize()

    def check(self, precision):
        torch = self.torch
        torch.cuda.synchronize()
        for c, plan, scale, st, co, res, vals in self.jobs:
            if res is not None:
                assert textbook.normwise_rel(res.cpu().numpy(), scale * c["res"]) < 1e-12
            if vals is not None:
                assert textbook.normwise_rel(vals.cpu().numpy(), c["vals"]) < (1e-5 if precision else 1e-12)
                if c["mesh"].order >= 3:
                    alone = torch.empty_like(vals)
                    plan.assemble(st, co, E, NU, T, values=alone, precision=precision)
                    torch.cuda.synchronize()
                    assert torch.equal(alone, vals)
            for out in (res, vals):
                if out is not None:
                    out.fill_(float("nan"))
        _ = torch.ones(1024, device="cuda").sum().item()  # the caller's own work between assemblies
        torch.cuda.synchronize()


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("own_stream", [False, True])
def test_replays(fem, torch_gpu, cases, precision, own_stream):
    torch = torch_gpu
    stream = torch.cuda.Stream() if own_stream else None
    plans = [fem.Plan(c["mesh"], c["pat"]) for c in cases]
    batch = fem.Batch(max_jobs=4, graph=True)
    for rnd in range(3):
        for name, which in (("A", A), ("B", B), ("C", C), ("D", D)):
            filled = Filled(torch, batch, cases, plans, which, 1.0 + rnd)
            for rep in range(3):
                print(f"graph batch: {name}, round {rnd}, assembly {rep}, precision {precision}", flush=True)
                batch.assemble(precision=precision, stream=stream)
                filled.check(precision)
    # replays queued behind one another, jobs refilled as soon as the call returns
    for which in (A, D):
        first = Filled(torch, batch, cases, plans, which, 1.0)
        for _ in range(3):
            batch.assemble(precision=precision, stream=stream)
        second = Filled(torch, batch, cases, plans, which, 2.0)
        batch.assemble(precision=precision, stream=stream)
        first.check(precision)
        second.check(precision)
    batch.close()
    for p in plans:
        p.close()


def test_prepare_with_jobs(fem, torch_gpu, cases):
    """On a batch with jobs of every kind; the server calls it on empty ones. Then batches that replay what it recorded."""
    torch = torch_gpu
    prepare = fem.load()["_ZN3fem13batch_prepareEP9fem_batchi"]
    prepare.argtypes, prepare.restype = [ctypes.c_void_p, ctypes.c_int], ctypes.c_int
    plans = [fem.Plan(c["mesh"], c["pat"]) for c in cases]
    batch = fem.Batch(max_jobs=4, graph=True)
    filled = Filled(torch, batch, cases, plans, A, 1.0)
    for precision in (0, 1):
        print(f"prepare with jobs: precision {precision}", flush=True)
        assert prepare(batch.handle, precision) == 0
        torch.cuda.synchronize()
        for job in filled.jobs:
            assert all(bool(torch.isnan(out).all()) for out in job[5:] if out is not None)
    for rep in range(3):
        batch.assemble(precision=0)
        filled.check(0)
    for rnd in range(4):  # the prepared composition, of small jobs and of larger ones
        full = FULL if rnd % 2 else [(6 if i == 1 else i, res, vals) for i, res, vals in FULL]
        filled = Filled(torch, batch, cases, plans, full, 1.0 + rnd)
        for rep in range(2):
            print(f"prepared composition: round {rnd}, assembly {rep}", flush=True)
            batch.assemble(precision=1)
            filled.check(1)
            batch.assemble(precision=0)
            filled.check(0)
    batch.close()
    for p in plans:
        p.close()


@pytest.mark.parametrize("warm", [0, 3])
def test_in_a_capture(fem, torch_gpu, cases, warm):
    """A batch of orders 1-2 assembled under the caller's own capture, before any other assembly or after replays:
    the caller's graph uploads the tables and launches the kernels itself."""
    torch = torch_gpu
    which = [(0, True, True), (1, True, True), (1, True, False)]
    plans = [fem.Plan(c["mesh"], c["pat"]) for c in cases]
    batch = fem.Batch(max_jobs=4, graph=True)
    filled = Filled(torch, batch, cases, plans, which, 1.0)
    stream = torch.cuda.Stream()
    for _ in range(warm):
        batch.assemble(stream=stream)
        filled.check(0)
    graph = torch.cuda.CUDAGraph()
    print(f"captured batch: warm {warm}", flush=True)
    with torch.cuda.graph(graph, stream=stream, capture_error_mode="thread_local"):
        batch.assemble(stream=stream)
    for _ in range(3):
        graph.replay()
        filled.check(0)
    del graph
    batch.close()
    for p in plans:
        p.close()
