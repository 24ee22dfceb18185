"""The coordinates given to a plan only order its parts (a Hilbert curve through the elements): the outputs are the same
whatever they are. True coordinates, other ones (one point, one line, far away, mirrored) and none, on shuffled meshes of
one part and of many, with nodes of no element; FP64 bar 1e-12, mixed 1e-5 (values; the residual is FP64 in both)."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

E, NU, T = 70e9, 0.3, 1.0
ORDERINGS = {
    "true": lambda x: x,
    "one point": lambda x: np.full_like(x, 0.25),
    "one line": lambda x: x * [1.0, 0.0],
    "far away": lambda x: x * 1e-9 + 1e6,
    "mirrored": lambda x: -1e12 * x[:, ::-1],
    "none": None,
}


def rel(x, ref):
    return float(np.linalg.norm(x.cpu().numpy() - ref) / np.linalg.norm(ref))


@pytest.mark.parametrize("order,nx,ny", [(1, 1, 1), (1, 41, 37), (2, 3, 2), (2, 29, 31), (3, 12, 13)])
@pytest.mark.parametrize("kind", ["default", "deterministic", "residual", "owner"])
def test_ordering_coordinates(fem, orc, torch_gpu, order, nx, ny, kind):
    torch = torch_gpu
    on = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()  # noqa: E731
    m = fem.square_mesh(nx, order, jitter=0.2, seed=nx, ny=ny)
    rng = np.random.default_rng(nx)
    nodes = m.num_nodes + 3  # three of no element
    perm = rng.permutation(nodes).astype(np.int32)
    coords = np.full((nodes, 2), 0.5)
    coords[perm[:m.num_nodes]] = m.coords
    m = fem.Mesh(order, coords, rng.permutation(perm[m.conn]))
    pat = fem.bsr_pattern(m)
    u = fem.fill_uniform(2 * nodes, -1e-3, 1e-3, 5)
    rref, vref = orc.jacobian(m, u, E, NU, T, fem.element_bcsr_map(m, pat), pat.num_blocks)
    co, st = on(m.coords), on(u)
    flags = {"default": 0, "deterministic": fem.FEM_PLAN_DETERMINISTIC, "residual": fem.FEM_PLAN_RESIDUAL_ONLY,
             "owner": fem.FEM_PLAN_OWNER_ONLY}[kind]
    for name, place in ORDERINGS.items():
        print(f"plan order: {name}, order {order}, {nx}x{ny}, {kind}", flush=True)
        placed = m if place is None else fem.Mesh(order, np.ascontiguousarray(place(m.coords)), m.conn)
        plan = fem.Plan(placed, pat, flags=flags, morton=place is not None)
        for precision, bar in ((fem.FEM_PREC_FP64, 1e-12), (fem.FEM_PREC_MIXED, 1e-5)):
            res = torch.full((2 * nodes,), float("nan"), dtype=torch.float64, device="cuda")
            vals = None if kind == "residual" else torch.full((4 * pat.num_blocks,), float("nan"), dtype=torch.float64,
                                                              device="cuda")
            plan.assemble(st, co, E, NU, T, res=res, values=vals, precision=precision)
            torch.cuda.synchronize()
            assert rel(res, rref) < 1e-12 and (vals is None or rel(vals, vref) < bar)
        plan.close()
