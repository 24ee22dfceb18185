"""The one gather launch of a batch's element-once jobs at its edges: meshes without staged outputs (one element), with
fewer lines than a wavefront takes, jobs with and without a residual, two jobs on one plan, groups left empty. A batch
sums in the order of the plan assembled alone, so the outputs are compared bit for bit; each batch is refilled once."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

E, NU, T = 70e9, 0.3, 1.0
# (order, nx, ny, with residual) of each job
BATCHES = {
    "one element": [(3, 1, 1, True), (4, 1, 1, False)],
    "few lines": [(3, 2, 1, True), (3, 1, 1, True), (3, 1, 2, True), (3, 5, 7, True)],
    "order 4 alone": [(4, 17, 3, False), (4, 2, 1, False), (4, 2, 1, True)],
    "all": [(3, 5, 7, False), (4, 5, 7, True), (3, 40, 31, True), (4, 1, 1, True), (3, 2, 2, False), (4, 23, 30, False),
            (1, 9, 8, True), (2, 9, 8, True), (4, 2, 2, True), (3, 40, 31, True)],
}


@pytest.mark.parametrize("name", list(BATCHES))
@pytest.mark.parametrize("graph", [False, True])
@pytest.mark.parametrize("precision", [0, 1])
def test_batch_gather(fem, torch_gpu, name, graph, precision):
    torch = torch_gpu
    on = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()  # noqa: E731
    plans = {}
    batch = fem.Batch(max_jobs=8, graph=graph)
    for refill in range(2):
        batch.clear()
        jobs = []
        for k, (order, nx, ny, with_res) in enumerate(BATCHES[name][::1 - 2 * refill]):
            if (order, nx, ny) not in plans:
                m = fem.square_mesh(nx, order, jitter=0.2, seed=nx, ny=ny)
                pat = fem.bsr_pattern(m)
                plans[order, nx, ny] = (m, pat, fem.Plan(m, pat))
            m, pat, plan = plans[order, nx, ny]
            st, co = on(fem.fill_uniform(2 * m.num_nodes, -1e-3, 1e-3, 5 + k)), on(m.coords)
            out = lambda n: torch.full((n,), float("nan"), dtype=torch.float64, device="cuda")  # noqa: E731
            res, vals = out(2 * m.num_nodes) if with_res else None, out(4 * pat.num_blocks)
            batch.add(plan, st, co, E, NU, T, res=res, values=vals)
            jobs.append((plan, order, st, co, res, vals))
        print(f"batch gather: {name}, graph {graph}, precision {precision}, refill {refill}", flush=True)
        batch.assemble(precision=precision)
        torch.cuda.synchronize()
        for plan, order, st, co, res, vals in jobs:
            r, v = None if res is None else torch.empty_like(res), torch.empty_like(vals)
            plan.assemble(st, co, E, NU, T, res=r, values=v, precision=precision)
            torch.cuda.synchronize()
            if order <= 2:  # sums in LDS, in no fixed order
                assert bool(torch.isfinite(vals).all()) and bool(torch.isfinite(res).all())
                continue
            assert torch.equal(v, vals) and (res is None or torch.equal(r, res))
    batch.close()
    for _, _, plan in plans.values():
        plan.close()
