"""The region index of the peak kernels (snapgpu_region_index) against a stable sort in numpy."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [0, 1, 2, 255, 256, 257, 300, 20_000])
@pytest.mark.parametrize("n_chrom,top", [(5, 40), (1, 2**40), (300, 2**59)])
def test_region_index_equals_a_stable_sort(torch_gpu, n, n_chrom, top):
    from snapatac2_amd.pp._peaks import RegionArrays, region_index
    rng = np.random.default_rng(n)
    chrom = rng.integers(-1, max(n_chrom - 1, 1), n).astype(np.int32)  # -1: outside the genome; the last one of many stays empty
    start, end = rng.integers(0, top, n), rng.integers(0, 2 * top, n)
    starts, ends, pmax, index, off = (t.cpu().numpy() for t in region_index(RegionArrays(chrom, start, end), n_chrom, torch_gpu))
    order = np.lexsort((np.arange(n), start, chrom))
    order = order[chrom[order] >= 0]
    k = len(order)
    assert np.array_equal(index[:k], order) and np.array_equal(starts[:k], start[order])
    assert np.array_equal(ends[:k], end[order])
    assert np.array_equal(off, np.searchsorted(chrom[order], np.arange(n_chrom + 1)))
    for c in range(n_chrom):
        a, b = off[c], off[c + 1]
        assert np.array_equal(pmax[a:b], np.maximum.accumulate(end[order][a:b]))
