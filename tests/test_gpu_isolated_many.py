"""Meshes with more nodes of no element than the parts of the usual cut have room for: the plan is cut with smaller parts
and takes them. Every route against the oracle (FP64 bar 1e-12); the rows of those nodes are stored as zeros."""

import numpy as np
import pytest

import textbook

pytestmark = pytest.mark.gpu

E, NU, T = 70e9, 0.3, 1.0
# (order, elements along an edge, such nodes, flag): the usual cut's room is 4273 and 3703 in the first two
CASES = [(2, 40, 4600, "default"), (4, 20, 4300, "owner"), (1, 3, 4000, "default"), (2, 5, 30000, "deterministic"),
         (3, 12, 40000, "default"), (2, 7, 40000, "residual")]


@pytest.mark.parametrize("order,n,extra,kind", CASES)
def test_many_isolated_nodes(fem, orc, torch_gpu, order, n, extra, kind):
    torch = torch_gpu
    on = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()  # noqa: E731
    base = fem.square_mesh(n, order, jitter=0.2, seed=n, ny=n + 1 if order == 4 else n)
    rng = np.random.default_rng(extra)
    nodes = base.num_nodes + extra
    perm = rng.permutation(nodes).astype(np.int32)
    coords = rng.random((nodes, 2))
    coords[perm[:base.num_nodes]] = base.coords
    m = fem.Mesh(order, coords, np.ascontiguousarray(perm[base.conn]))
    pat = fem.bsr_pattern(m)
    u = fem.fill_uniform(2 * nodes, -1e-3, 1e-3, 5)
    rref, vref = orc.jacobian(m, u, E, NU, T, fem.element_bcsr_map(m, pat), pat.num_blocks)
    flags = {"default": 0, "deterministic": fem.FEM_PLAN_DETERMINISTIC, "residual": fem.FEM_PLAN_RESIDUAL_ONLY,
             "owner": fem.FEM_PLAN_OWNER_ONLY}[kind]
    print(f"many isolated nodes: order {order}, {n}, {extra}, {kind}", flush=True)
    plan = fem.Plan(m, pat, flags=flags)
    res = torch.full((2 * nodes,), float("nan"), dtype=torch.float64, device="cuda")
    vals = None if kind == "residual" else torch.full((4 * pat.num_blocks,), float("nan"), dtype=torch.float64, device="cuda")
    plan.assemble(on(u), on(m.coords), E, NU, T, res=res, values=vals)
    torch.cuda.synchronize()
    assert textbook.normwise_rel(res.cpu().numpy(), rref) < 1e-12
    assert np.all(res.cpu().numpy().reshape(-1, 2)[perm[base.num_nodes:]] == 0)
    if vals is not None:
        assert textbook.normwise_rel(vals.cpu().numpy(), vref) < 1e-12
    plan.close()
