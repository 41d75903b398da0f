"""Path C on the GPU: neighbour sets and distances vs the FP64 brute-force oracle."""
import numpy as np
import pytest

from oracle import knn as oknn

pytestmark = pytest.mark.gpu


def clustered(n, d=30, n_clusters=10, seed=0):
    rng = np.random.default_rng(seed)
    centres = 3.0 * rng.standard_normal((n_clusters, d))
    lab = rng.integers(0, n_clusters, n)
    X = centres[lab] + rng.standard_normal((n, d))
    return X / np.linalg.norm(X, axis=1, keepdims=True)


def _check(g, X, k):
    o = oknn.knn_graph(X, k)
    assert g.shape == o.shape
    assert np.array_equal(g.indptr, o.indptr)
    assert np.array_equal(g.indices, o.indices)
    # distances: exact FP64 rescoring with the oracle's formula -> identical bits
    assert np.array_equal(g.data, o.data)


@pytest.mark.parametrize("precision", ["bf16", "fp32"])
@pytest.mark.parametrize("n,d,k", [(5000, 30, 50), (3000, 17, 25), (1000, 30, 100), (100, 5, 50)])
def test_clustered_vs_oracle(torch_gpu, precision, n, d, k):
    from snapatac2_amd.pp._knn import nearest_neighbour_graph
    X = clustered(n, d, seed=n + d)
    g, st = nearest_neighbour_graph(X, k, precision=precision, return_stats=True)
    _check(g, X, k)
    if k <= 50:  # 128 candidates leave a wide margin for k <= 50
        assert st["fallback_rows"] <= n // 100 + 1


def test_spectral_scale_embedding(torch_gpu):
    # embeddings like X_spectral: tiny values (eigenvectors * sqrt(eigenvalue))
    from snapatac2_amd.pp._knn import nearest_neighbour_graph
    X = clustered(4000, 30, seed=9) * 1e-3
    X[:, 20:] *= 1e-2
    _check(nearest_neighbour_graph(X, 50), X, 50)


def test_ties_and_duplicates(torch_gpu):
    # integer lattice points: many exactly equal distances, plus duplicate rows
    from snapatac2_amd.pp._knn import nearest_neighbour_graph
    rng = np.random.default_rng(1)
    X = rng.integers(0, 4, (1500, 3)).astype(np.float64)
    for precision in ("bf16", "fp32"):
        _check(nearest_neighbour_graph(X, 30, precision=precision), X, 30)


def test_forced_fallback_is_exact(torch_gpu):
    from snapatac2_amd.pp._knn import nearest_neighbour_graph
    X = clustered(700, 30, seed=3)
    g, st = nearest_neighbour_graph(X, 50, force_fallback=True, return_stats=True)
    assert st["fallback_rows"] == 700
    _check(g, X, 50)


def test_knn_dropin(torch_gpu):
    import snapatac2_amd as snap
    X = clustered(800, 30, seed=5)
    ad = snap.AnnData(n_obs=800, n_vars=1)
    ad.obsm["X_spectral"] = X
    snap.pp.knn(ad, n_neighbors=25)
    _check(ad.obsp["distances"], X, 25)
    g2 = snap.pp.knn(X, n_neighbors=25, use_dims=10)
    _check(g2, X[:, :10], 25)
    # determinism (reference test_reproducibility, test_tools.py:95-122)
    g3 = snap.pp.knn(ad, n_neighbors=25, inplace=False)
    assert (g3 != ad.obsp["distances"]).nnz == 0
    with pytest.raises(ValueError, match="empty"):
        snap.pp.knn(np.zeros((0, 5)))
    with pytest.raises(ValueError, match="method"):
        snap.pp.knn(ad, method="bogus")
    tiny = snap.pp.knn(X[:5], n_neighbors=50)
    assert tiny.nnz == 20


def test_second_tier_on_offset_clusters(torch_gpu):
    # rows far from the origin with small spreads: |q|^2 >> d^2. The uncentred
    # FP32 bound cannot certify them, so the exact FP64 second tier takes over;
    # the BF16 path centres each query block and certifies them directly.
    from snapatac2_amd.pp._knn import nearest_neighbour_graph
    X = 1.0 + 1e-3 * clustered(3000, 20, seed=4)
    g, st = nearest_neighbour_graph(X, 50, precision="fp32", return_stats=True)
    _check(g, X, 50)
    assert st["fallback_rows"] > 0
    assert st["exact_scan_rows"] <= st["fallback_rows"]
    g, st = nearest_neighbour_graph(X, 50, precision="bf16", return_stats=True)
    _check(g, X, 50)
    assert st["fallback_rows"] <= 30


@pytest.mark.parametrize("n,d", [(2999, 7), (1001, 30), (17, 1)])
def test_second_tier_shapes(torch_gpu, n, d):
    """Offset clusters push rows to the exact FP64 tier; point counts that are
    not a multiple of the 16-point tile and odd dimensions exercise its tile
    loads and padding."""
    from snapatac2_amd.pp._knn import nearest_neighbour_graph
    X = 1.0 + 1e-3 * clustered(n, d, seed=n + d)
    k = min(50, n - 1)
    g, st = nearest_neighbour_graph(X, k, precision="fp32", return_stats=True)
    _check(g, X, k)
    assert st["exact_scan_rows"] <= st["fallback_rows"]


@pytest.mark.parametrize("n_clusters,spread", [(10, 3.0), (40, 8.0), (1, 0.0)])
def test_chunk_skipping_is_exact(torch_gpu, n_clusters, spread):
    """The bf16 path skips database chunks whose bounding sphere lies beyond every
    threshold of a workgroup: the result equals the FP64 oracle and the run that
    visits every chunk; chunks of well-separated clusters are skipped."""
    from snapatac2_amd.pp._knn import nearest_neighbour_graph
    rng = np.random.default_rng(n_clusters)
    n, d, k = 20000, 30, 50
    centres = spread * rng.standard_normal((n_clusters, d))
    X = centres[rng.integers(0, n_clusters, n)] + rng.standard_normal((n, d))
    g, st = nearest_neighbour_graph(X, k, return_stats=True)
    g_all, st_all = nearest_neighbour_graph(X, k, return_stats=True, prune=False)
    _check(g, X, k)
    assert np.array_equal(g.indices, g_all.indices) and np.array_equal(g.data, g_all.data)
    assert st_all["chunk_visits"] == st_all["chunk_pairs"]
    assert st["chunk_visits"] <= st["chunk_pairs"]
    if n_clusters == 40:
        assert st["chunk_visits"] < 0.7 * st["chunk_pairs"], st


# --- beyond d = 30 and k = 100: the exact all-pairs path ------------------------

@pytest.mark.parametrize("precision", ["bf16", "fp32"])
@pytest.mark.parametrize("n,d,k", [(4000, 50, 50), (3000, 20, 150), (2500, 64, 150), (300, 31, 101),
                                   (200, 1, 199), (20_000, 31, 101)])
def test_wide_rows_and_many_neighbours(torch_gpu, precision, n, d, k):
    """knn.rs:9-32 has no limit on d or k: n_comps = 50 or n_neighbors = 150 give
    the FP64 brute-force sets and bit-identical distances (20,000 points take
    several query blocks of the scan)."""
    from snapatac2_amd.pp._knn import nearest_neighbour_graph
    X = clustered(n, d, seed=n + d + k)
    g, st = nearest_neighbour_graph(X, k, precision=precision, return_stats=True)
    _check(g, X, k)
    assert st["exact_scan_rows"] == n


def test_wide_ties_and_duplicates(torch_gpu):
    """Integer lattice in 40 dimensions plus repeated rows: exact ties are ordered
    by neighbour index, as in the oracle."""
    from snapatac2_amd.pp._knn import nearest_neighbour_graph
    rng = np.random.default_rng(2)
    X = rng.integers(0, 2, (1200, 40)).astype(np.float64)
    X[600:700] = X[0]
    _check(nearest_neighbour_graph(X, 120), X, 120)


def test_knn_dropin_with_50_components(torch_gpu):
    import snapatac2_amd as snap
    from snapatac2_amd.anndata import AnnData
    X = clustered(3000, 50, seed=4)
    ad = AnnData(n_obs=3000, n_vars=0)
    ad.obsm["X_spectral"] = X
    snap.pp.knn(ad, n_neighbors=150)
    _check(ad.obsp["distances"], X, 150)
    g = snap.pp.knn(ad, n_neighbors=30, use_dims=45, inplace=False)
    _check(g, np.ascontiguousarray(X[:, :45]), 30)


@pytest.mark.parametrize("n,d,k", [(129, 3, 25), (129, 3, 26), (2777, 8, 25), (2777, 8, 26), (640, 29, 1),
                                   (15, 2, 14), (6000, 2, 25)])
def test_candidate_lists(torch_gpu, n, d, k):
    """Both sides of the rule for the candidates per lane (16 up to k = 25, else 32), with chunks
    that are not full; few rows may need the second tier (16 of the nearest in one stripe, 15 in
    the query's own: one query in 2,900 at k = 25; a Poisson count of mean 2 exceeds 12 once in
    a million draws)."""
    from snapatac2_amd.pp._knn import nearest_neighbour_graph
    X = clustered(n, d, n_clusters=3, seed=n + k)
    g, st = nearest_neighbour_graph(X, k, return_stats=True)
    _check(g, X, k)
    assert st["exact_scan_rows"] == 0 or n < 4 * k
    if n > 2000:
        assert st["fallback_rows"] <= 12, st


def test_candidates_far_from_the_centre(torch_gpu):
    """Values from 1e-3 to 1e12 in one matrix: the padding rows' score stays below the real ones'."""
    from snapatac2_amd.pp._knn import nearest_neighbour_graph
    rng = np.random.default_rng(5)
    X = rng.standard_normal((900, 6)) * 10.0 ** rng.integers(-3, 13, 900)[:, None]
    _check(nearest_neighbour_graph(X, 20), X, 20)


@pytest.mark.parametrize("kind,n,d", [("clusters", 16383, 30), ("clusters", 16385, 30), ("clusters", 33001, 7),
                                      ("one cluster", 25000, 30), ("line", 40000, 1), ("duplicates", 20001, 4),
                                      ("constant", 16400, 3), ("scales", 30000, 5), ("dominant", 30001, 6)])
def test_cells(torch_gpu, kind, n, d):
    """From 16,384 rows on (128 leaves) the rows are ordered by cells and chunks are skipped by
    the planes between them: the graph of a run that skips nothing, and the oracle's rows."""
    from snapatac2_amd.pp._knn import nearest_neighbour_graph
    rng = np.random.default_rng(n)
    k = 30
    X = {"clusters": lambda: clustered(n, d, seed=n),
         "one cluster": lambda: rng.standard_normal((n, d)),
         "line": lambda: rng.random((n, 1)),
         "duplicates": lambda: rng.integers(0, 9, (n, d)).astype(np.float64),
         "constant": lambda: np.full((n, d), 0.25),
         "dominant": lambda: rng.standard_normal((n, d)) + 40.0 * rng.integers(0, 4, (n, d)) * (rng.random((n, 1)) < 0.1),
         "scales": lambda: rng.standard_normal((n, d)) * 10.0 ** rng.integers(-4, 5, n)[:, None]}[kind]()
    g = nearest_neighbour_graph(X, k)
    full = nearest_neighbour_graph(X, k, prune=False)
    assert np.array_equal(g.indices, full.indices) and np.array_equal(g.data, full.data)
    rows = rng.choice(n, 300, replace=False)
    d2 = np.zeros((300, n))
    for c in range(d):  # the reference's order and rounding
        d2 += (X[rows, c][:, None] - X[:, c][None]) ** 2
    d2[np.arange(300), rows] = np.inf
    for i, r in enumerate(rows):
        near = np.sort(np.argsort(d2[i], kind="stable")[:k])
        assert np.array_equal(g.indices[r * k:(r + 1) * k], near)
        assert np.array_equal(g.data[r * k:(r + 1) * k], np.sqrt(d2[i, near]))
