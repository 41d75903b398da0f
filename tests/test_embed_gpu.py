"""The eigenvectors' way out of the device (snapgpu_embed_finish) against numpy: sign of the
first entry of largest magnitude, choice of columns, scaling."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _numpy(U, cols, scale):
    U = U[:, cols]
    lead = U[np.argmax(np.abs(U), axis=0), np.arange(U.shape[1])]
    sign = np.where(lead == 0, 1.0, np.sign(lead))
    out = U * sign
    return out if scale is None else out * scale


# 256 rows per slice of the search, 64 slices at a time when their results are joined
@pytest.mark.parametrize("n,k", [(1, 1), (7, 3), (255, 32), (256, 33), (257, 31), (1024, 2), (5000, 70), (16384, 3),
                                 (16385, 2), (40000, 5)])
@pytest.mark.parametrize("case", ["random", "ties", "zero", "nan", "strided"])
def test_finish(torch_gpu, n, k, case):
    torch = torch_gpu
    from snapatac2_amd.tl._embedding import _finished
    rng = np.random.default_rng(n + k)
    U = rng.standard_normal((n, k + 2))
    if case == "ties":  # equal magnitudes of both signs, in many rows
        U = rng.integers(-2, 3, (n, k + 2)).astype(np.float64)
        if n > 64 * 256:  # and the largest in two slices that one lane joins, 64 apart
            U[200], U[64 * 256 + min(200, n - 64 * 256 - 1)] = (-5.0, 5.0) if k % 2 else (5.0, -5.0)
    if case == "zero":
        U[:, 0] = 0.0
    if case == "nan":
        U[n // 2, 0] = np.nan
        U[n // 3, 0] = np.inf
    t = torch.from_numpy(U).cuda()
    if case != "strided":
        U = np.ascontiguousarray(U[:, :k])
        t = torch.from_numpy(U).cuda()
    else:
        t, U = t[:, :k], U[:, :k]
    cols = rng.permutation(k)[:max(1, k - 1)]
    for scale in (None, rng.uniform(0.1, 2.0, cols.size)):
        assert np.array_equal(_finished(t, cols, scale), _numpy(U, cols, scale), equal_nan=True)
