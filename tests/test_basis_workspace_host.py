"""The workspace of C = A^T B (snapgpu_gemm_tn_workspace_bytes, host only): the block Lanczos
solver sizes one for its widest basis, (n, J, 32), and runs every narrower product in it."""
import pytest

from snapatac2_amd import _lib


@pytest.mark.parametrize("n", [1, 257, 40_000, 70_000, 150_000, 500_000, 1_000_000, 3_000_000])
@pytest.mark.parametrize("J", [16, 511, 512, 513, 1023, 1024, 1041, 2113])
def test_holds_every_narrower_product(n, J):
    need = _lib.lib().snapgpu_gemm_tn_workspace_bytes
    have = need(n, J, 32)
    for ka in {*range(1, J + 1, 16), J - 1, J}:
        assert max(need(n, ka, kb) for kb in (1, 15, 16, 17, 31, 32)) <= have, ka


def test_grows_with_the_rows():
    need = _lib.lib().snapgpu_gemm_tn_workspace_bytes
    rows = [0, 1, 255, 256, 257, 4096, 4097, 65_535, 65_537, 200_000, 1_048_576, 2_097_153, 5_000_000]
    for ka, kb in ((1, 1), (16, 16), (320, 32), (1041, 32)):
        sizes = [need(n, ka, kb) for n in rows]
        assert sizes == sorted(sizes)
