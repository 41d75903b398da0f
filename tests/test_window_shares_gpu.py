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


@pytest.mark.parametrize("chunk", [13.9, 14.0, 16.0, 17.9, 18.1])
def test_entries_ahead(torch_gpu, chunk):
    """Both sides of the rule for the entries loaded ahead (24 where a quad's chunk holds 14 to 18
    on average), with chunks shorter than 16 and longer than 24 among them."""
    torch = torch_gpu
    from snapatac2_amd.tl._operator import SpectralOperator, _to_device_csr
    rng = np.random.default_rng(int(10 * chunk))
    n, m = 1500, 3000  # one block, three windows: 768 chunks
    nnz = int(np.ceil(chunk * 768))
    length = np.full(n, nnz // n)
    length[rng.choice(n, nnz - length.sum(), replace=False)] += 1
    cols = [np.sort(rng.choice(m, k, replace=False)) for k in length]
    X = sp.csr_matrix((rng.integers(1, 200, nnz).astype(np.uint32), np.concatenate(cols),
                       np.concatenate([[0], np.cumsum(length)])), shape=(n, m))
    op = SpectralOperator(_to_device_csr(X, torch), layout="window")
    w = op.window_csr
    assert op.layout == "window" and w.n_blocks * w.n_windows == 3
    V = rng.standard_normal((n, 16))
    Xh, dinv, _, _ = osp.operator_parts(X)
    ref = Xh @ (Xh.T @ V) - dinv[:, None] * V
    Y = op.matmat(torch.from_numpy(V).cuda()).cpu().numpy()
    assert np.abs(Y - ref).max() < 1e-5 * np.abs(ref).max()
