"""Residual-only routes that work by lines of nodes: fem_residual, fem_residual_nonlinear and residual-only plans.

Sizes at the edges of the kernels: below, at and above the elements of one wavefront (32, 21, 16, 12 for orders
1..4) and of one workgroup (four times as many); parts of one and of several batches; element orders in which an
element's last nodes are and are not the next one's first; more nodes of no element than the parts have room for at
their default size. Bar 1e-12 against the oracle, as for every FP64 path.
"""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

E, NU, T = 70e9, 0.3, 1.0
EPW = {1: 32, 2: 21, 3: 16, 4: 12}


def rel(x, ref):
    return float(np.abs(x.cpu().numpy() - ref).max() / np.abs(ref).max())


def on(torch, a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def strip(fem, order, elements, shuffle):
    m = fem.square_mesh(elements, order, jitter=0.2, seed=elements, ny=1) if elements > 0 else None
    if shuffle:
        m = fem.Mesh(order, m.coords, np.random.default_rng(elements).permutation(m.conn))
    return m


@pytest.mark.parametrize("order", [1, 2, 3, 4])
@pytest.mark.parametrize("shuffle", [False, True])
@pytest.mark.parametrize("waves", [1, 4])
def test_wavefront_edges(fem, orc, torch_gpu, order, shuffle, waves):
    torch = torch_gpu
    for elements in (1, waves * EPW[order] - 1, waves * EPW[order], waves * EPW[order] + 1):
        m = strip(fem, order, max(elements, 1), shuffle)
        print(f"residual lines: order {order}, {m.num_elements} elements, shuffle {shuffle}", flush=True)
        u = fem.fill_uniform(2 * m.num_nodes, -1e-3, 1e-3, 5)
        cp, cn, st, co = (on(torch, a) for a in (m.conn_ptr, m.conn, u, m.coords))
        for nonlinear in (False, True):
            ref = orc.residual(m, u, E, NU, T, nonlinear=nonlinear)
            out = torch.ones(2 * m.num_nodes, dtype=torch.float64, device="cuda")
            fem.residual(order, cp, cn, m.num_elements, st, co, E, NU, T, out, nonlinear=nonlinear)
            out -= 1.0
            # the ones add an absolute rounding error of 1e-16 per sum
            assert rel(out, ref) <= 1e-12 + 1e-14 / np.abs(ref).max()
        plan = fem.Plan(m, fem.bsr_pattern(m), flags=fem.FEM_PLAN_RESIDUAL_ONLY)
        out = torch.full((2 * m.num_nodes,), float("nan"), dtype=torch.float64, device="cuda")
        ref = orc.residual(m, u, E, NU, T)
        plan.assemble(st, co, E, NU, T, res=out)
        assert rel(out, ref) <= 1e-12
        plan.assemble(st, co, E, NU, T, res=out, precision=fem.FEM_PREC_MIXED, accumulate=True)
        assert rel(out, 2 * ref) <= 1e-12
        plan.close()


@pytest.mark.parametrize("order,n", [(1, 90), (2, 60), (3, 41), (4, 37)])
@pytest.mark.parametrize("extra", [0, 900])
def test_parts(fem, orc, torch_gpu, order, n, extra):
    """Several batches per part; `extra` nodes of no element (stored as zeros), in a mesh of few parts when there are
    any, so that they only fit parts of the largest size."""
    torch = torch_gpu
    m = fem.square_mesh(n if extra == 0 else 3, order, jitter=0.2, seed=3)
    used = m.num_nodes
    if extra:
        m = fem.Mesh(order, np.concatenate([m.coords, np.full((extra, 2), 0.5)]), m.conn)
    print(f"residual lines: order {order}, {m.num_elements} elements, {extra} nodes of no element", flush=True)
    u = fem.fill_uniform(2 * m.num_nodes, -1e-3, 1e-3, 7)
    ref = orc.residual(m, u, E, NU, T)
    plan = fem.Plan(m, fem.bsr_pattern(m), flags=fem.FEM_PLAN_RESIDUAL_ONLY)
    out = torch.full((2 * m.num_nodes,), float("nan"), dtype=torch.float64, device="cuda")
    plan.assemble(on(torch, u), on(torch, m.coords), E, NU, T, res=out)
    assert rel(out, ref) <= 1e-12
    assert float(out[2 * used:].abs().sum()) == 0.0
    plan.close()
