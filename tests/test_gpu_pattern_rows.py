"""Edges of the device pattern's row merge and of the staged map, bit for bit against the host builders: workgroups of
128 rows (one below, at and above), rows of exactly four and of five elements, a workgroup with rows too long for its
LDS, elements that name a node twice, elements of more nodes than the merge takes, and the kept scratch under growing
and shrinking meshes and after its release."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def check(fem, torch, conn, nodes):
    ne, npe = conn.shape
    cp = (np.arange(ne) * npe).astype(np.int32)
    rowp_h = np.zeros(nodes + 1, np.int32)
    lib, P = fem.load(), fem._ptr
    conn = np.ascontiguousarray(conn, dtype=np.int32)
    assert lib.fem_bsr_pattern_rowp(nodes, ne, npe, P(cp), P(conn), P(rowp_h)) == 0
    cols_h = np.zeros(int(rowp_h[-1]), np.int32)
    assert lib.fem_bsr_pattern_cols(nodes, ne, npe, P(cp), P(conn), P(rowp_h), P(cols_h)) == 0
    map_h = np.zeros(ne * npe * npe, np.int32)
    assert lib.fem_element_bcsr_map(P(cp), P(conn), ne, npe, nodes, P(rowp_h), P(cols_h), 2, P(map_h)) == 0
    d = lambda a: torch.from_numpy(a).cuda()  # noqa: E731
    print(f"pattern rows: {nodes} nodes, {ne} elements of {npe}", flush=True)
    for noalloc in (False, True):
        rowp, cols = fem.bsr_pattern_device(nodes, ne, npe, d(cp), d(conn), noalloc=noalloc)
        assert np.array_equal(rowp.cpu().numpy(), rowp_h) and np.array_equal(cols.cpu().numpy(), cols_h)
    m = fem.element_bcsr_map_device(d(cp), d(conn), ne, npe, nodes, rowp, cols)
    assert np.array_equal(m.cpu().numpy(), map_h)


@pytest.mark.parametrize("nodes", [127, 128, 129, 385])
def test_workgroup_edges(fem, torch_gpu, nodes):
    rng = np.random.default_rng(nodes)
    conn = np.stack([rng.permutation(nodes)[:4] for _ in range(nodes)])  # rows of 0 to a dozen elements
    check(fem, torch_gpu, conn, nodes)


@pytest.mark.parametrize("fan", [4, 5, 40])
@pytest.mark.parametrize("npe", [4, 9, 25, 33])
def test_fans_and_wide_elements(fem, torch_gpu, fan, npe):
    """`fan` elements share node 0: a merged row, a sorted one, and one longer than the workgroup's LDS; 33 nodes per
    element leave the merge. The first element names its second node twice."""
    conn = np.concatenate([np.zeros((fan, 1), int), 1 + np.arange(fan * (npe - 1)).reshape(fan, npe - 1)], axis=1)
    conn[0, 2] = conn[0, 1]
    nodes = int(conn.max()) + 3
    if fan * npe > 1024:
        pytest.skip("beyond the device builder's node references per row")
    check(fem, torch_gpu, conn, nodes)


def test_kept_scratch(fem, torch_gpu):
    for n in (40, 90, 20, 90):
        m = fem.square_mesh(n, 2)
        check(fem, torch_gpu, m.conn, m.num_nodes)
    fem.dropin_cache_clear()
    m = fem.square_mesh(30, 4)
    check(fem, torch_gpu, m.conn, m.num_nodes)
