"""Results that a user keeps lie in ordinary host memory (page-locked memory is not mapped in
a forked worker), whole whatever the block they pass through."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _page_locked(torch, a: np.ndarray) -> bool:
    return torch.from_numpy(a).is_pinned()


@pytest.mark.parametrize("shape", [(0,), (0, 3), (1,), (255, 1), (257,), (256, 3), (1000, 7)])
@pytest.mark.parametrize("dtype", ["float64", "int32"])
def test_to_host(torch_gpu, monkeypatch, shape, dtype):
    torch = torch_gpu
    from snapatac2_amd import _device
    monkeypatch.setattr(_device, "_STAGE_BYTES", 2048)  # 256 doubles at a time
    monkeypatch.setattr(_device, "_THREADED_BYTES", 1024)  # whole blocks by torch, most remainders by numpy
    a = np.random.default_rng(1).integers(-9, 9, shape).astype(dtype)
    got = _device.to_host(torch.from_numpy(a).cuda())
    assert got.dtype == a.dtype and got.shape == a.shape and np.array_equal(got, a)
    assert not _page_locked(torch, got)


def test_results_are_ordinary_memory(torch_gpu):
    torch = torch_gpu
    from snapatac2_amd.pp._basic import _counted_column_sums
    from snapatac2_amd.tl._embedding import _finished
    import scipy.sparse as sp
    X = sp.random(50, 300, density=0.1, format="csr", random_state=0)
    X.data = np.ceil(X.data * 3).astype(np.uint32)
    sums, zeros = _counted_column_sums(X.astype(np.uint32))
    assert zeros == int((np.asarray(X.sum(axis=0)) == 0).sum()) and not _page_locked(torch, sums)
    U = torch.randn((40, 3), dtype=torch.float64, device="cuda")
    assert not _page_locked(torch, _finished(U, np.arange(3)))
