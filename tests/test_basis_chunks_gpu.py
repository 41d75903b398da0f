"""The row chunks of C = A^T B (snapgpu_gemm_tn_f64) at the edges of their sizes, and the
allocation-free form where its static scratch bounds their number: accepted, and the same bits."""
import pytest

from snapatac2_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,ka,kb", [(1, 3, 2), (255, 16, 16), (256, 100, 16), (257, 100, 16), (513, 33, 32),
                                     (65535, 48, 16), (65537, 48, 16), (150_000, 320, 32), (400_000, 1300, 32)])
def test_row_chunks(torch_gpu, n, ka, kb):
    torch = torch_gpu
    L = _lib.lib()
    gen = torch.Generator(device="cuda").manual_seed(n)
    A = torch.randn((n, ka), dtype=torch.float64, device="cuda", generator=gen)
    B = torch.randn((n, kb), dtype=torch.float64, device="cuda", generator=gen)
    C, D = (torch.empty((ka, kb), dtype=torch.float64, device="cuda") for _ in range(2))
    wsb = int(L.snapgpu_gemm_tn_workspace_bytes(n, ka, kb))
    ws = torch.empty(wsb, dtype=torch.uint8, device="cuda")
    st = _lib.stream_ptr()
    _lib.check(L.snapgpu_gemm_tn_f64(A.data_ptr(), ka, B.data_ptr(), kb, n, ka, kb, C.data_ptr(), ws.data_ptr(), wsb, st))
    _lib.check(L.snapgpu_gemm_tn_f64_noalloc(A.data_ptr(), ka, B.data_ptr(), kb, n, ka, kb, D.data_ptr(), st))
    bound = 1e-13 * (A.abs().T @ B.abs())
    assert bool(((C - A.T @ B).abs() <= bound).all())
    assert torch.equal(C, D)


def test_one_workspace_for_narrower_products(torch_gpu):
    """The block Lanczos solver's use: a workspace of the widest basis, and a narrower product
    that takes more row chunks (70,000 rows: 125 at 1041 x 32, 256 at 1024 x 16)."""
    torch = torch_gpu
    L = _lib.lib()
    n = 70_000
    gen = torch.Generator(device="cuda").manual_seed(n)
    A = torch.randn((n, 1041), dtype=torch.float64, device="cuda", generator=gen)
    wsb = int(L.snapgpu_gemm_tn_workspace_bytes(n, 1041, 32))
    ws = torch.empty(wsb, dtype=torch.uint8, device="cuda")
    for ka, kb in ((1024, 16), (1041, 32), (17, 1)):
        B = torch.randn((n, kb), dtype=torch.float64, device="cuda", generator=gen)
        C = torch.empty((ka, kb), dtype=torch.float64, device="cuda")
        _lib.check(L.snapgpu_gemm_tn_f64(A.data_ptr(), 1041, B.data_ptr(), kb, n, ka, kb, C.data_ptr(), ws.data_ptr(),
                                         wsb, _lib.stream_ptr()))
        bound = 1e-13 * (A[:, :ka].abs().T @ B.abs())
        assert bool(((C - A[:, :ka].T @ B).abs() <= bound).all()), (ka, kb)
