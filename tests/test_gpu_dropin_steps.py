"""The per-call check of fem_jacobian_dropin at the edges of its launch, and the atomic Jacobian kernels' adds in
ascending column order.

The check reads every node reference, 512 to a workgroup and at most 1024 workgroups at a time: meshes of one element,
of one reference fewer and more than a workgroup takes, and of more than a full grid. Two nodes of the last element
trade ids in place; a plan kept from before would write the old layout. The atomic kernels sort an element's columns by
node: elements numbered at random, wavefronts partly empty, and an element that names one node several times (a quad
collapsed to a triangle). FP64 bar 1e-12, mixed 1e-5 (values), as for the same routes elsewhere."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

E, NU, T = 70e9, 0.3, 1.0


def on(torch, a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def rel(x, ref):
    return float(np.linalg.norm(x.cpu().numpy() - ref) / np.linalg.norm(ref))


@pytest.mark.parametrize("order,nx,ny", [(1, 1, 1), (1, 127, 1), (1, 128, 1), (1, 129, 1), (1, 363, 362), (2, 1, 1),
                                         (2, 56, 1), (2, 57, 1), (2, 114, 1)])
def test_check_sees_the_last_reference(fem, orc, torch_gpu, order, nx, ny):
    torch = torch_gpu
    fem.dropin_cache_clear()
    m = fem.square_mesh(nx, order, jitter=0.2, seed=nx, ny=ny)
    u = fem.fill_uniform(2 * m.num_nodes, -1e-3, 1e-3, 9)
    conn_d, cp_d = on(torch, m.conn), on(torch, m.conn_ptr)
    u_d, x_d = on(torch, u), on(torch, m.coords)
    map_d = on(torch, np.zeros(m.conn.shape[0] * m.conn.shape[1] ** 2, dtype=np.int32))
    last = m.conn[-1]
    a, b = int(last[-1]), int(last[order])  # corners of the last element alone (right edge, last row)
    for swapped in (False, True):
        print(f"check: order {order}, {nx}x{ny}, swapped {swapped}", flush=True)
        coords, conn, uu = m.coords.copy(), m.conn.copy(), u.reshape(-1, 2).copy()
        if swapped:
            coords[[a, b]], uu[[a, b]] = coords[[b, a]], uu[[b, a]]
            conn[m.conn == a], conn[m.conn == b] = b, a
        mm = fem.Mesh(order, coords, conn)
        pat = fem.bsr_pattern(mm)
        bmap = fem.element_bcsr_map(mm, pat)
        rref, vref = orc.jacobian(mm, uu.reshape(-1), E, NU, T, bmap, pat.num_blocks)
        conn_d.copy_(on(torch, conn))
        u_d.copy_(on(torch, uu.reshape(-1)))
        x_d.copy_(on(torch, coords))
        map_d.copy_(on(torch, bmap.reshape(-1)))
        for _ in range(2):  # the first call builds, the second checks
            res = torch.zeros(2 * mm.num_nodes, dtype=torch.float64, device="cuda")
            vals = torch.zeros(4 * pat.num_blocks, dtype=torch.float64, device="cuda")
            fem.jacobian(order, cp_d, conn_d, mm.num_elements, u_d, x_d, E, NU, T, map_d, res, vals, dropin=True)
            torch.cuda.synchronize()
            assert fem.dropin_cache_info(order, cp_d, conn_d, mm.num_elements, map_d) == (True, True)
            assert rel(res, rref) < 1e-12 and rel(vals, vref) < 1e-12
    fem.dropin_cache_clear()


@pytest.mark.parametrize("order", [1, 2, 3, 4])
@pytest.mark.parametrize("collapsed", [False, True])
def test_atomic_adds_in_column_order(fem, orc, torch_gpu, order, collapsed):
    torch = torch_gpu
    m = fem.square_mesh(17, order, jitter=0.2, seed=order, ny=3)
    conn, coords = m.conn.copy(), m.coords.copy()
    n = order + 1
    if collapsed:  # the first element's left edge becomes one node
        first = conn[0].reshape(n, n)
        x, y = coords[first, 0], coords[first, 1]
        mid = y.mean()
        coords[first, 1] = mid + (y - mid) * (x - x.min()) / (x.max() - x.min())
        conn[0] = np.where(np.arange(n * n) % n == 0, first[0, 0], conn[0])
    rng = np.random.default_rng(order)
    perm = rng.permutation(m.num_nodes).astype(np.int32)
    shuffled = np.empty_like(coords)
    shuffled[perm] = coords
    m = fem.Mesh(order, shuffled, perm[conn])
    pat = fem.bsr_pattern(m)
    bmap = fem.element_bcsr_map(m, pat)
    u = fem.fill_uniform(2 * m.num_nodes, -1e-3, 1e-3, 5)
    rref, vref = orc.jacobian(m, u, E, NU, T, bmap, pat.num_blocks)
    for precision, bar in ((fem.FEM_PREC_FP64, 1e-12), (fem.FEM_PREC_MIXED, 1e-5)):
        print(f"atomic adds: order {order}, collapsed {collapsed}, precision {precision}", flush=True)
        res = torch.zeros(2 * m.num_nodes, dtype=torch.float64, device="cuda")
        vals = torch.zeros(4 * pat.num_blocks, dtype=torch.float64, device="cuda")
        fem.jacobian(order, on(torch, m.conn_ptr), on(torch, m.conn), m.num_elements, on(torch, u),
                     on(torch, m.coords), E, NU, T, on(torch, bmap.reshape(-1)), res, vals, precision=precision)
        torch.cuda.synchronize()
        assert rel(res, rref) < 1e-12 and rel(vals, vref) < bar
