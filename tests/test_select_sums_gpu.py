"""The column sums as doubles with the count of zeros (snapgpu_col_sums_f64) against numpy."""
import numpy as np
import pytest

from snapatac2_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m", [1, 255, 256, 257, 600001])
def test_column_sums_as_doubles(torch_gpu, m):
    torch = torch_gpu
    rng = np.random.default_rng(m)
    sums = rng.integers(0, 3, m) * rng.integers(1, 2**60, m)
    d = torch.from_numpy(sums).cuda()
    out = torch.empty(m, dtype=torch.float64, device="cuda")
    zeros = torch.full((1,), 7, dtype=torch.int64, device="cuda")
    _lib.check(_lib.lib().snapgpu_col_sums_f64(d.data_ptr(), m, out.data_ptr(), zeros.data_ptr(), _lib.stream_ptr()))
    assert np.array_equal(out.cpu().numpy(), sums.astype(np.float64))
    assert int(zeros.item()) == int((sums == 0).sum())


def test_replayed_from_a_graph(torch_gpu):
    """The count starts at zero on every replay, with eager work between them."""
    torch = torch_gpu
    L, m = _lib.lib(), 70_000
    d = torch.zeros(m, dtype=torch.int64, device="cuda")
    out = torch.empty(m, dtype=torch.float64, device="cuda")
    zeros = torch.zeros(1, dtype=torch.int64, device="cuda")
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        rc = L.snapgpu_col_sums_f64(d.data_ptr(), m, out.data_ptr(), zeros.data_ptr(), _lib.stream_ptr())
    assert rc == _lib.OK
    for k in range(1, 6):
        sums = np.random.default_rng(k).integers(0, k + 1, m)
        d.copy_(torch.from_numpy(sums))
        graph.replay()
        torch.cuda.synchronize()
        assert int(zeros.item()) == int((sums == 0).sum())
        assert np.array_equal(out.cpu().numpy(), sums.astype(np.float64))
