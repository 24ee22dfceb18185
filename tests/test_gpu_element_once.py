"""Element-once Jacobians of orders 3-4: matrix-core tiles, row emission, staging and the 64-byte-line gather.

Meshes at the edges: fewer elements than a wavefront takes (4 at order 3, 2 at order 4), one more than a workgroup's,
odd block counts (the last line of the values holds one block), shuffled elements and nodes (few contributions of an
element are neighbours in the matrix), outputs that start half a line into a 64-byte line, accumulation onto old
values. FP64 bar 1e-12, mixed 1e-5 (values; the residual is FP64 in both), as for every plan route.
"""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

E, NU, T = 70e9, 0.3, 1.0


def on(torch, a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def rel(x, ref):
    return float(np.abs(x.cpu().numpy() - ref).max() / np.abs(ref).max())


@pytest.mark.parametrize("order", [3, 4])
@pytest.mark.parametrize("nx,ny", [(1, 1), (3, 1), (5, 1), (17, 1), (2, 2), (5, 7)])
@pytest.mark.parametrize("shuffle", [False, True])
def test_edges(fem, orc, torch_gpu, order, nx, ny, shuffle):
    torch = torch_gpu
    m = fem.square_mesh(nx, order, jitter=0.2, seed=nx, ny=ny)
    if shuffle:
        rng = np.random.default_rng(nx * 10 + ny)
        perm = rng.permutation(m.num_nodes).astype(np.int32)
        coords = np.empty_like(m.coords)
        coords[perm] = m.coords
        m = fem.Mesh(order, coords, rng.permutation(perm[m.conn]))
    pat = fem.bsr_pattern(m)
    u = fem.fill_uniform(2 * m.num_nodes, -1e-3, 1e-3, 5)
    r_ref, v_ref = orc.jacobian(m, u, E, NU, T, fem.element_bcsr_map(m, pat), pat.num_blocks)
    st, co = on(torch, u), on(torch, m.coords)
    plan = fem.Plan(m, pat)
    for precision, bar in ((fem.FEM_PREC_FP64, 1e-12), (fem.FEM_PREC_MIXED, 1e-5)):
        for offset in (0, 4, 1):  # doubles into the allocation: line-aligned, half a line, 8-byte aligned only
            print(f"element-once: order {order}, {nx}x{ny}, shuffle {shuffle}, offset {offset}", flush=True)
            vals = torch.full((4 * pat.num_blocks + 8,), float("nan"), dtype=torch.float64, device="cuda")
            res = torch.full((2 * m.num_nodes,), float("nan"), dtype=torch.float64, device="cuda")
            v = vals[offset:offset + 4 * pat.num_blocks]
            plan.assemble(st, co, E, NU, T, res=res, values=v, precision=precision)
            assert rel(res, r_ref) <= 1e-12 and rel(v, v_ref) <= bar
            first = v.clone()
            plan.assemble(st, co, E, NU, T, values=v, precision=precision)
            assert torch.equal(first, v)  # fixed order of sums
            plan.assemble(st, co, E, NU, T, res=res, values=v, precision=precision, accumulate=True)
            assert rel(res, 2 * r_ref) <= 1e-12 and rel(v, 2 * v_ref) <= bar
            rest = torch.cat([vals[:offset], vals[offset + 4 * pat.num_blocks:]])
            assert bool(torch.isnan(rest).all())  # nothing outside the matrix
    plan.close()
