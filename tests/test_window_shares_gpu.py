"""The window product where its last turn of workgroups is cut into shares along the windows
(more than 256 workgroups, and a remainder of at most 224): against the FP64 oracle within the
operator's 1e-5, bitwise reproducible, with one window (most shares empty), a few and many,
and a cut block that holds rows without entries past its 2048 slots."""
import numpy as np
import pytest
import scipy.sparse as sp

from oracle import spectral as osp

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rest,m,empty", [(1, 900, 0), (1, 5000, 0), (3, 5000, 4000), (224, 5000, 0), (225, 5000, 0),
                                          (60, 100_000, 0)])
def test_shares(torch_gpu, rest, m, empty):
    torch = torch_gpu
    from snapatac2_amd.tl._operator import SpectralOperator, _to_device_csr
    rng = np.random.default_rng(rest)
    n = 2048 * (512 + rest) - 5  # one slot per row
    rows = np.repeat(np.arange(n), 3)
    cols = rng.integers(0, m, 3 * n)
    if empty:  # in the last block, none of them the first row of a window of the transpose
        rows = rows + np.where(rows >= n - 100, empty, 0)
    X = sp.csr_matrix((np.ones(3 * n, np.uint32), (rows, cols)), shape=(n + empty, m))
    X.sort_indices()
    Xd = _to_device_csr(X, torch)
    op = SpectralOperator(Xd, layout="window")
    assert op.layout == "window" and op.window_csr.n_blocks == 512 + rest
    full = np.diff(X.indptr) > 0
    V = rng.standard_normal((n + empty, 16))
    V[~full] = 0.0
    if empty:
        op.r32[torch.from_numpy(~full).cuda()] = 0.0  # no degree: kept out of the products
    Xh, dinv, _, _ = osp.operator_parts(X[full])
    ref = Xh @ (Xh.T @ V[full]) - dinv[:, None] * V[full]
    Y = op.matmat(torch.from_numpy(V).cuda())
    assert np.abs(Y.cpu().numpy()[full] - ref).max() < 1e-5 * np.abs(ref).max()
    again = op.matmat(torch.from_numpy(V).cuda())
    ok = torch.from_numpy(full).cuda()
    assert torch.equal(Y[ok], again[ok])
