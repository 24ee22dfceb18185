"""NONLINEAR tangent at the edges of its row chunks (5 rows of 9, 8 of 16, 5 of 25) and of its wavefronts (16, 7, 4 and 2
elements at orders 1-4): meshes of one element, of a wavefront's and one more, shuffled; with and without the residual,
added onto what the outputs hold. FP64 bar 1e-12, as for the same kernels elsewhere."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

E, NU, T = 70e9, 0.3, 1.0


def rel(x, ref):
    return float(np.linalg.norm(x.cpu().numpy() - ref) / np.linalg.norm(ref))


@pytest.mark.parametrize("order", [1, 2, 3, 4])
@pytest.mark.parametrize("elements", [1, 2, 3, 4, 5, 7, 8, 16, 17, 57])
def test_row_chunks(fem, orc, torch_gpu, order, elements):
    torch = torch_gpu
    on = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()  # noqa: E731
    m = fem.square_mesh(elements, order, jitter=0.2, seed=elements, ny=1)
    rng = np.random.default_rng(elements)
    perm = rng.permutation(m.num_nodes).astype(np.int32)
    coords = np.empty_like(m.coords)
    coords[perm] = m.coords * [elements, 1.0]
    m = fem.Mesh(order, coords, rng.permutation(perm[m.conn]))
    u = fem.smooth_field(m.coords, 5e-2, phase_seed=order, pert=1e-3, pert_seed=7)
    pat = fem.bsr_pattern(m)
    bmap = fem.element_bcsr_map(m, pat)
    rref, vref = orc.jacobian(m, u, E, NU, T, bmap, pat.num_blocks, nonlinear=True)
    cp, conn, st, xy, mp = on(m.conn_ptr), on(m.conn.reshape(-1)), on(u), on(m.coords), on(bmap.reshape(-1))
    print(f"nonlinear chunks: order {order}, {elements} elements", flush=True)
    res = torch.zeros(2 * m.num_nodes, dtype=torch.float64, device="cuda")
    vals = torch.zeros(4 * pat.num_blocks, dtype=torch.float64, device="cuda")
    for r, calls in ((None, 1), (res, 2)):
        fem.jacobian(order, cp, conn, m.num_elements, st, xy, E, NU, T, mp, r, vals, nonlinear=True)
        torch.cuda.synchronize()
        assert rel(vals, calls * vref) <= 1e-12
    assert rel(res, rref) <= 1e-12
