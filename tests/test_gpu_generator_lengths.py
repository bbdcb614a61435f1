"""Graph generation on the GPU where a connection's length changes how its rows are drawn (waves per
row, draws kept in LDS or made twice), against the host build, bit for bit: degrees around 256 KB NW
draws (2,048, 8,192 and 32,768), one target and none, whole rows, many short connections (more
than 64 per row)."""
import numpy as np
import pytest

from oracle import oracle as O
from spice_amd.snn import generate_graph

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("layout", [
    ([2047], [(0, 0, 1.0)]), ([2048], [(0, 0, 1.0)]), ([4090], [(0, 0, 0.5)]),
    ([8191], [(0, 0, 1.0)]), ([40, 8192], [(0, 1, 1.0)]), ([30, 16400], [(0, 1, 0.5)]),
    ([20, 32767], [(0, 1, 1.0)]), ([20, 32768], [(0, 1, 1.0)]), ([10, 70000], [(0, 1, 0.9)]),
    ([500], [(0, 0, 0.002)]), ([64, 1], [(0, 1, 1.0)]), ([300], [(0, 0, 0.0)]),
    ([7] * 70, [(0, d, 0.5) for d in range(70)]), ([50, 60], [(0, 1, 0.3), (1, 0, 0.2), (0, 0, 0.1), (1, 1, 0.9)]),
], ids=lambda x: f"{sum(x[0])}x{len(x[1])}")
def test_generated_graph_equals_host(gpu, layout):
    import torch
    rp_h, col_h, w_h = O.generate_csr(layout, 21)
    rp = torch.full((sum(layout[0]) + 1,), -1, dtype=torch.int64, device="cuda")
    col = torch.full((max(int(rp_h[-1]), 1) + 3,), -7, dtype=torch.int32, device="cuda")
    nnz, w = generate_graph(layout, 21, rp.data_ptr(), col.data_ptr(), max(int(rp_h[-1]), 1))
    torch.cuda.synchronize()
    assert (nnz, w) == (int(rp_h[-1]), w_h)
    np.testing.assert_array_equal(rp.cpu().numpy(), rp_h)
    np.testing.assert_array_equal(col.cpu().numpy()[:nnz], col_h)
    assert (col[max(nnz, 1):].cpu().numpy() == -7).all()  # nothing is written past the graph
