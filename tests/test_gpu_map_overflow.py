"""Element maps on the device whose 32-bit offsets overflow are refused, also where the entries of one block no longer
fit 32 bits; the largest block that a pattern's blocks leave room for is mapped as on the host."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("npe", [4, 5])  # the map in tiles, and one thread per entry
def test_map_offsets(fem, torch_gpu, npe):
    torch = torch_gpu
    conn = np.arange(npe, dtype=np.int32).reshape(1, npe)
    rowp, cols = np.arange(npe + 1, dtype=np.int32) * npe, np.tile(conn[0], npe)
    d = lambda a: torch.from_numpy(a).cuda()  # noqa: E731
    args = d(np.zeros(1, np.int32)), d(conn), 1, npe, npe, d(rowp), d(cols)
    fits = int(np.sqrt((2**31 - 1) // (npe * npe)))
    got = fem.element_bcsr_map_device(*args, bsize=fits)
    assert np.array_equal(got.cpu().numpy(), np.arange(npe * npe) * fits * fits)
    for bsize in (fits + 1, 46340, 46341, 65536, 1 << 20, 2**31 - 1):
        with pytest.raises(fem.FemError) as e:
            fem.element_bcsr_map_device(*args, bsize=bsize)
        assert e.value.status == -7, bsize
