"""One plan called with other buffers, outputs and modes on every call and without a wait between them: each launch
carries its own job. Orders 1-4 on the routes that share the job record (streaming parts, deterministic parts, residual
parts), one part and many; FP64 bar 1e-12, mixed 1e-5 (values; the residual is FP64 in both)."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

E, NU, T = 70e9, 0.3, 1.0


def rel(x, ref):
    return float(np.linalg.norm(x.cpu().numpy() - ref) / np.linalg.norm(ref))


@pytest.mark.parametrize("order,nx,ny", [(1, 2, 3), (1, 70, 61), (2, 1, 1), (2, 45, 37), (3, 21, 20), (4, 13, 12)])
@pytest.mark.parametrize("kind", ["default", "deterministic", "residual"])
def test_every_call_its_own_buffers(fem, orc, torch_gpu, order, nx, ny, kind):
    torch = torch_gpu
    on = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()  # noqa: E731
    m = fem.square_mesh(nx, order, jitter=0.2, seed=nx, ny=ny)
    pat = fem.bsr_pattern(m)
    us = [fem.fill_uniform(2 * m.num_nodes, -1e-3, 1e-3, 5 + k) for k in range(3)]
    refs = [orc.jacobian(m, u, E, NU, T, fem.element_bcsr_map(m, pat), pat.num_blocks) for u in us]
    flags = {"default": 0, "deterministic": fem.FEM_PLAN_DETERMINISTIC, "residual": fem.FEM_PLAN_RESIDUAL_ONLY}[kind]
    plan = fem.Plan(m, pat, flags=flags)
    co, states = on(m.coords), [on(u) for u in us]
    for precision, bar in ((fem.FEM_PREC_FP64, 1e-12), (fem.FEM_PREC_MIXED, 1e-5)):
        print(f"plan jobs: order {order}, {nx}x{ny}, {kind}, precision {precision}", flush=True)
        done = []
        for k in range(9):
            u, t = k % 3, T * (1 + k)  # the outputs are linear in the thickness
            res = torch.zeros(2 * m.num_nodes, dtype=torch.float64, device="cuda") if k % 4 != 3 or kind == "residual" else None
            vals = torch.zeros(4 * pat.num_blocks, dtype=torch.float64, device="cuda") if k % 4 != 1 and kind != "residual" else None
            plan.assemble(states[u], co, E, NU, t, res=res, values=vals, precision=precision, accumulate=k % 2 == 1)
            done.append((u, 1 + k, res, vals))
        torch.cuda.synchronize()
        for u, scale, res, vals in done:
            assert res is None or rel(res, scale * refs[u][0]) < 1e-12
            assert vals is None or rel(vals, scale * refs[u][1]) < bar
    plan.close()
