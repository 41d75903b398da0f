"""The device-wide inclusive scan (snapgpu_scan_inclusive_i64) against numpy at the edges of
its runs of 16, tiles of 4096 and levels of 4096 tiles."""
import numpy as np
import pytest

from snapatac2_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 15, 16, 17, 255, 4095, 4096, 4097, 100_003, 4096 * 4096, 4096 * 4096 + 5])
def test_scan(torch_gpu, n):
    torch = torch_gpu
    L = _lib.lib()
    x = np.random.default_rng(n).integers(-2**40, 2**40, n)
    d = torch.from_numpy(x).cuda()
    wsb = int(L.snapgpu_scan_workspace_bytes(n))
    ws = torch.empty(wsb, dtype=torch.uint8, device="cuda")
    _lib.check(L.snapgpu_scan_inclusive_i64(d.data_ptr(), n, ws.data_ptr(), wsb, _lib.stream_ptr()))
    assert np.array_equal(d.cpu().numpy(), np.cumsum(x))
