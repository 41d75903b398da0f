"""Path A on the GPU: libsnapgpu tile kernels vs the oracle, bit-exact."""
import json
import os

import numpy as np
import pytest

from oracle import tile as otile

pytestmark = pytest.mark.gpu
GOLD = os.path.join(os.path.dirname(__file__), "golden")


def _frags(torch, cells, paired=True):
    from snapatac2_amd._device import DeviceFragments
    cell_ptr = np.zeros(len(cells) + 1, dtype=np.int64)
    cell_ptr[1:] = np.cumsum([len(c) for c in cells])
    pos = np.asarray([p for c in cells for p, _ in c], dtype=np.uint32)
    ln = np.asarray([l for c in cells for _, l in c], dtype=np.uint32)
    dev = torch.device("cuda")
    t = lambda a: torch.from_numpy(a.view(np.int32)).to(dev)
    vals = t(ln) if paired else torch.from_numpy(ln.astype(np.int32)).to(dev)
    return DeviceFragments(torch.from_numpy(cell_ptr).to(dev), t(pos), vals, 0, paired), \
        cell_ptr, pos, ln


def _tile(torch, cells, cs, bin_size, excl, lo, hi, strategy):
    from snapatac2_amd.pp import make_tile_matrix
    paired = strategy != "single"
    fr, cp, pos, ln = _frags(torch, cells, paired)
    X, names = make_tile_matrix(fr, cs, bin_size, excl, lo, hi,
                                strategy if paired else "paired-insertion")
    return X.to_scipy(), names, (cp, pos, ln)


def _same(a, b):
    assert a.shape == b.shape, (a.shape, b.shape)
    assert np.array_equal(a.indptr, b.indptr)
    assert np.array_equal(a.indices.astype(np.int64), b.indices.astype(np.int64))
    assert np.array_equal(a.data.astype(np.uint32), b.data.astype(np.uint32))


def test_hand_derived_cases(torch_gpu):
    g = json.load(open(os.path.join(GOLD, "tile_cases.json")))
    cs = dict((c, l) for c, l in g["chrom_sizes"])
    cells = [[tuple(f) for f in c] for c in g["cells"]]
    for case in g["cases"]:
        m, _, _ = _tile(torch_gpu, cells, cs, g["bin_size"], case["exclude"], case["min"],
                        case["max"], case["strategy"])
        assert m.shape == (3, case["n_bins"])
        rows = [[[int(j), int(v)] for j, v in zip(m.indices[m.indptr[r]:m.indptr[r + 1]],
                                                  m.data[m.indptr[r]:m.indptr[r + 1]])]
                for r in range(3)]
        assert rows == case["rows"], case


def test_out_of_range_raises(torch_gpu):
    from snapatac2_amd._lib import PanicException
    g = json.load(open(os.path.join(GOLD, "tile_cases.json")))
    cs = dict((c, l) for c, l in g["chrom_sizes"])
    with pytest.raises(PanicException, match="out of range"):
        _tile(torch_gpu, [[tuple(f) for f in g["panic_cell"]]], cs, 100, [], None, None,
              "paired-insertion")


def test_genome_index_vectors_through_kernel(torch_gpu):
    # every base of the genome.rs test genome, one single-end read per cell
    g = json.load(open(os.path.join(GOLD, "genome_index.json")))
    cs = dict((c, l) for c, l in g["chrom_sizes"])
    total = sum(cs.values())
    cells = [[(i, 1)] for i in range(total)]
    for step in (1, 2, 3):
        m, names, _ = _tile(torch_gpu, cells, cs, step, [], None, None, "single")
        cols = m.indices.astype(np.int64)
        assert np.array_equal(m.indptr, np.arange(total + 1))
        exp = [otile.get_position_rev(cs, step, *otile.get_position(cs, i)) for i in range(total)]
        assert cols.tolist() == exp
    for i1, i2 in g["coarsed_step2"]:
        m, _, _ = _tile(torch_gpu, [[(i1, 1)]], cs, 2, [], None, None, "single")
        assert int(m.indices[0]) == i2


@pytest.mark.parametrize("strategy", ["insertion", "fragment", "paired-insertion", "single"])
def test_random_vs_oracle(torch_gpu, strategy):
    from test_tile_oracle import random_cells
    rng = np.random.default_rng(17)
    cs = {"chr1": 50000, "chr10": 12345, "chr2": 30000, "chrM": 3000, "chrX": 25000}
    cells = random_cells(rng, cs, 300, max_frags=400, max_len=1200)
    cells[5] = []
    for bin_size, excl, lo, hi in [(500, ["chrM", "chrY"], None, None), (37, ["chrX"], 10, 300),
                                   (1, [], None, None), (5000, ["chr1", "chr10"], 50, None)]:
        m, names, (cp, pos, ln) = _tile(torch_gpu, cells, cs, bin_size, excl, lo, hi, strategy)
        o = otile.tile_matrix(cp, pos, ln, cs, bin_size, excl, lo, hi, strategy)
        _same(m, o)
        assert len(names) == m.shape[1]


def test_dense_duplicates_and_long_spans(torch_gpu):
    # many fragments in one bin (pending list grows), and spans that need the
    # larger capacity levels (bin 1 with 3 kb fragments)
    cs = {"chr1": 100000}
    hot = [(1000 + (i % 7), 300 + (i % 50)) for i in range(5000)]
    longf = [(i * 10, 3000 + i % 3) for i in range(200)]
    cells = [sorted(hot), sorted(longf), [(5, 2)] * 1000]
    for strategy in ("insertion", "paired-insertion", "fragment"):
        for bin_size in (1, 100, 500):
            m, _, (cp, pos, ln) = _tile(torch_gpu, cells, cs, bin_size, [], None, None, strategy)
            o = otile.tile_matrix(cp, pos, ln, cs, bin_size, [], None, None, strategy)
            _same(m, o)


def _ordered_cells(rng, cs):
    """Rows that exercise the in-order tile path and its hand-over to the
    general merge: runs that span whole 64-fragment tiles, fragments whose last
    bin is the next fragment's first, occasional interleaved pairs (a fragment
    ending beyond the next one's start bin), size-filtered and excluded-chromosome
    fragments inside runs, and tiles that cross chromosome boundaries."""
    starts = np.cumsum([0] + list(cs.values()))
    names = list(cs)
    cells = []
    # one bin for 300 fragments (the pending run carried through whole tiles)
    cells.append([(1000, 40)] * 300)
    # steady walk: each fragment ends in the bin where the next one starts
    cells.append([(100 * i, 101) for i in range(400)])
    # mostly ordered with interleaved pairs every ~70 fragments
    c, x = [], 5000
    for i in range(700):
        x += int(rng.integers(0, 60))
        ln = 900 if i % 70 == 69 else int(rng.integers(20, 120))
        c.append((x, ln))
    cells.append(sorted(c))
    # walk over every chromosome boundary, with short (size-filtered) fragments
    c = []
    for ci, nm in enumerate(names):
        lo, hi = starts[ci], starts[ci + 1]
        for p in range(int(lo), int(hi) - 400, max(1, (int(hi) - int(lo)) // 150)):
            c.append((p, 5 if (p // 7) % 9 == 0 else int(rng.integers(30, 300))))
    cells.append(sorted(c))
    # dense peaks: many fragments per bin, 1-3 bins long
    c = []
    for _ in range(40):
        ci = int(rng.integers(0, len(names)))
        centre = int(rng.integers(starts[ci] + 200, starts[ci + 1] - 1000))
        for _ in range(int(rng.integers(20, 90))):
            c.append((centre + int(rng.integers(-150, 150)), int(rng.integers(40, 700))))
    cells.append(sorted(c))
    # short fragments (both insertions in one bin) in long runs
    cells.append(sorted([(2000 + 3 * (i // 20), 2) for i in range(500)]))
    return cells


@pytest.mark.parametrize("strategy", ["insertion", "paired-insertion"])
def test_ordered_tiles_and_handover(torch_gpu, strategy):
    rng = np.random.default_rng(23)
    cs = {"chr1": 60000, "chr2": 40000, "chrM": 5000, "chr3": 30000}
    cells = _ordered_cells(rng, cs)
    for bin_size, excl, lo, hi in [(500, ["chrM"], None, None), (1, [], None, None), (7, ["chr2"], 10, 650),
                                   (100, [], 30, None), (20000, ["chrM"], None, None)]:
        m, names, (cp, pos, ln) = _tile(torch_gpu, cells, cs, bin_size, excl, lo, hi, strategy)
        o = otile.tile_matrix(cp, pos, ln, cs, bin_size, excl, lo, hi, strategy)
        _same(m, o)


def test_synthetic_2k_cells_all_strategies(torch_gpu):
    from snapatac2_amd import synth
    from snapatac2_amd.genome import synthetic_genome
    fr = synth.generate_chunk(synth.GeneratorTables(0), 0, 2000)
    h = fr.to_scipy()
    cs = synthetic_genome()
    from snapatac2_amd.pp import make_tile_matrix
    for strategy in ("paired-insertion", "insertion", "fragment"):
        X, names = make_tile_matrix(fr, cs, 500, ["chrM", "chrY", "M", "Y"], None, None, strategy)
        o = otile.tile_matrix(h.indptr, h.indices, h.data, cs, 500, ["chrM", "chrY"], None,
                              None, strategy)
        _same(X.to_scipy(), o)
        assert X.shape[1] == 6_062_095 - 0  # chr1-22, X at 500 bp


def test_add_tile_matrix_dropin_and_determinism(torch_gpu):
    import snapatac2_amd as snap
    from snapatac2_amd import synth
    ad = synth.synthetic_anndata(300, seed=3)
    snap.pp.add_tile_matrix(ad)
    X1 = ad.X.to_scipy()
    out = snap.pp.add_tile_matrix(ad, inplace=False, bin_size=1000, exclude_chroms="chrX",
                                  counting_strategy="insertion")
    assert out.shape[0] == 300 and out.shape[1] == len(out.var_names)
    ad2 = synth.synthetic_anndata(300, seed=3)
    snap.pp.add_tile_matrix(ad2)
    _same(X1, ad2.X.to_scipy())
    assert ad.var_names[0] == "chr1:0-500"
    with pytest.raises(RuntimeError, match="Counting strategy"):
        snap.pp.add_tile_matrix(ad, counting_strategy="bogus")
    with pytest.raises(Exception, match="Value type"):
        snap.pp.add_tile_matrix(ad, value_type="bogus")
    empty = snap.AnnData(n_obs=2, n_vars=0)
    with pytest.raises(RuntimeError, match="must be present"):
        snap.pp.add_tile_matrix(empty)


def test_select_features_matches_numpy(torch_gpu):
    import snapatac2_amd as snap
    from snapatac2_amd import synth
    from snapatac2_amd.pp._basic import _find_most_accessible_features
    ad = synth.synthetic_anndata(500, seed=1)
    snap.pp.add_tile_matrix(ad)
    snap.pp.select_features(ad, n_features=20000)
    Xh = ad.X.to_scipy()
    count = np.ravel(Xh.sum(axis=0)).astype(np.float64)
    assert np.array_equal(ad.var["count"].to_numpy(), count)
    sel = np.zeros(Xh.shape[1], dtype=bool)
    sel[_find_most_accessible_features(count, 0.005, 0.005, 20000)] = True
    assert np.array_equal(ad.var["selected"].to_numpy(), sel)
    assert sel.sum() == 20000


def _shuffled(rng, cells):
    out = []
    for c in cells:
        c = list(c)
        rng.shuffle(c)
        out.append(c)
    return out


@pytest.mark.parametrize("strategy", ["insertion", "fragment", "paired-insertion", "single"])
def test_rows_out_of_order_give_the_sorted_result(torch_gpu, strategy):
    """The reference's per-row BTreeMap accepts fragments in any order
    (data_iter.rs:362-411): shuffled rows give the matrix of the sorted rows.
    The tile pass reports them (SNAPGPU_ERR_UNSORTED) and the host sorts a copy;
    the caller's arrays stay as they were."""
    from test_tile_oracle import random_cells
    from snapatac2_amd.pp import make_tile_matrix
    rng = np.random.default_rng(23)
    cs = {"chr1": 50000, "chr10": 12345, "chr2": 30000, "chrM": 3000, "chrX": 25000}
    cells = random_cells(rng, cs, 200, max_frags=300, max_len=1200)
    shuf = _shuffled(rng, cells)
    shuf[3] = cells[3]  # sorted rows among unsorted ones
    paired = strategy != "single"
    fr, cp, pos, ln = _frags(torch_gpu, shuf, paired)
    before = fr.pos.clone()
    X, _ = make_tile_matrix(fr, cs, 500, ["chrM"], None, None, strategy if paired else "paired-insertion")
    o = otile.tile_matrix(cp, pos, ln, cs, 500, ["chrM"], None, None, strategy)
    _same(X.to_scipy(), o)
    assert torch_gpu.equal(fr.pos, before)
    # the oracle itself is order-independent
    sp_, spos, sln = _frags(torch_gpu, cells, paired)[1:]
    _same(o, otile.tile_matrix(sp_, spos, sln, cs, 500, ["chrM"], None, None, strategy))


def test_rows_out_of_order_chunked(torch_gpu):
    from snapatac2_amd import synth
    from snapatac2_amd.genome import synthetic_genome
    from snapatac2_amd.pp._basic import make_tile_matrix_chunked
    cs = synthetic_genome()
    rng = np.random.default_rng(4)
    chunks, hs = [], []
    first = 0
    for k, n in enumerate([300, 200, 250]):
        fr = synth.generate_chunk(synth.GeneratorTables(0), first, n)
        h = fr.to_scipy()
        if k != 1:  # chunk 1 stays sorted
            for r in rng.choice(n, 40, replace=False):
                a, b = h.indptr[r], h.indptr[r + 1]
                perm = rng.permutation(b - a)
                h.indices[a:b] = h.indices[a:b][perm]
                h.data[a:b] = h.data[a:b][perm]
            fr = type(fr).from_scipy(h, paired=True)
        chunks.append((first, fr))
        hs.append(h)
        first += n
    X, _ = make_tile_matrix_chunked(chunks, cs, 500, ["chrM", "chrY"])
    import scipy.sparse as sp
    H = sp.vstack(hs, format="csr")
    o = otile.tile_matrix(H.indptr, H.indices, H.data, cs, 500, ["chrM", "chrY"])
    _same(X.to_scipy(), o)


def test_sort_rows_entry_and_unsorted_status(torch_gpu):
    """snapgpu_frag_sort_rows orders each row by (position, value); the count pass
    returns SNAPGPU_ERR_UNSORTED for a row whose positions go down, also when the
    decrease crosses a 64-fragment tile boundary."""
    import ctypes
    from snapatac2_amd import _lib
    torch = torch_gpu
    L = _lib.lib()
    rng = np.random.default_rng(9)
    cells = [[(int(p), int(l)) for p, l in zip(np.sort(rng.integers(0, 40000, m)), rng.integers(1, 500, m))]
             for m in (0, 1, 64, 65, 130, 500)]
    cells[4][64], cells[4][63] = cells[4][63], cells[4][64]  # swap across the tile boundary
    cells[4][63] = (cells[4][64][0] + 1, 7)
    cs = {"chr1": 50000}
    fr, cp, pos, ln = _frags(torch, cells, True)
    tab_h = np.zeros(L.snapgpu_tile_table_bytes(1), dtype=np.uint8)
    nb = ctypes.c_uint64()
    _lib.check(L.snapgpu_tile_table_pack(np.asarray([50000], np.uint64).ctypes.data,
                                         np.zeros(1, np.uint8).ctypes.data, 1, 500, tab_h.ctypes.data,
                                         ctypes.byref(nb)))
    tab = torch.from_numpy(tab_h).cuda()
    rows = torch.zeros(len(cells), dtype=torch.int64, device="cuda")
    status = torch.zeros(8, dtype=torch.int32, device="cuda")
    level = ctypes.c_int32(0)
    rc = L.snapgpu_tile_count(fr.cell_ptr.data_ptr(), fr.pos.data_ptr(), fr.values.data_ptr(), len(cells),
                              tab.data_ptr(), 1, 500, 2, 0, 0xFFFFFFFF, rows.data_ptr(), 0, status.data_ptr(),
                              ctypes.byref(level), _lib.stream_ptr())
    assert rc == _lib.ERR_UNSORTED and b"cell 4" in L.snapgpu_last_error()
    F = fr.n_fragments
    wsb = int(L.snapgpu_frag_sort_rows_workspace_bytes(len(cells), F))
    ws = torch.empty(wsb, dtype=torch.uint8, device="cuda")
    _lib.check(L.snapgpu_frag_sort_rows(fr.cell_ptr.data_ptr(), len(cells), F, fr.pos.data_ptr(),
                                        fr.values.data_ptr(), ws.data_ptr(), wsb, _lib.stream_ptr()))
    want = [sorted(c) for c in cells]
    gp = fr.pos.cpu().numpy().view(np.uint32)
    gl = fr.values.cpu().numpy().view(np.uint32)
    got = [list(zip(gp[a:b].tolist(), gl[a:b].tolist())) for a, b in zip(cp[:-1], cp[1:])]
    assert got == want
    level.value = 0
    _lib.check(L.snapgpu_tile_count(fr.cell_ptr.data_ptr(), fr.pos.data_ptr(), fr.values.data_ptr(), len(cells),
                                    tab.data_ptr(), 1, 500, 2, 0, 0xFFFFFFFF, rows.data_ptr(), 0,
                                    status.data_ptr(), ctypes.byref(level), _lib.stream_ptr()))


def _segment_cells(rng, cs):
    """Rows around the segment kernel's edges (256 fragments per segment, 4 per lane): lengths on
    both sides of whole segments; piles of one bin longer than a segment; fragments that reach
    over a segment's end by 1 to 31 bins of 100 bases, over filtered and excluded fragments too."""
    starts = dict(zip(cs, np.cumsum([0] + list(cs.values()))))
    cells = []
    for n in (0, 1, 3, 4, 255, 256, 257, 259, 511, 512, 513, 1030):
        pos = np.sort(rng.integers(0, cs["chr1"] - 4000, n))
        cells.append([(int(a), int(b)) for a, b in zip(pos, rng.integers(1, 3100, n))])
    cells.append([(5000 + i // 200, 1 + (i * 37) % 3100) for i in range(900)])      # one pile
    cells.append([(100 * i, 3101 if i % 5 else 20) for i in range(600)])            # spans of 31 bins
    cells.append([(40 * i, 1500) for i in range(254)] + [(254 * 40 + i, 30) for i in range(300)])
    mixed = [(int(a), 200) for a in np.sort(rng.integers(0, cs["chr1"] - 300, 250))]
    mixed += [(starts["chrM"] + 3 * i, 50) for i in range(300)]                     # excluded
    mixed += [(starts["chrX"] + 2 * i, 150 + i % 900) for i in range(700)]
    cells.append(mixed)
    return cells


@pytest.mark.parametrize("n_cells", [16, 1023, 1024, 8191, 8192])
@pytest.mark.parametrize("strategy", ["insertion", "fragment", "paired-insertion", "single"])
def test_segments(torch_gpu, strategy, n_cells):
    """16, 4 and 1 waves per cell (the cell counts lie on both sides of the rule)."""
    rng = np.random.default_rng(n_cells)
    cs = {"chr1": 70000, "chrM": 2000, "chrX": 20000}
    cells = _segment_cells(rng, cs)
    while len(cells) < n_cells:
        pos = np.sort(rng.integers(0, 59000, int(rng.integers(0, 40))))
        cells.append([(int(a), int(rng.integers(1, 900))) for a in pos])
    for lo, hi in ((None, None), (40, 2000)):
        m, _, (cp, pos, ln) = _tile(torch_gpu, cells, cs, 100, ["chrM"], lo, hi, strategy)
        _same(m, otile.tile_matrix(cp, pos, ln, cs, 100, ["chrM"], lo, hi, strategy))


@pytest.mark.parametrize("length", [3101, 3201, 3301])
def test_segments_hand_over_long_fragments(torch_gpu, length):
    """A fragment over more than 32 bins sends the call to the tile kernel; same matrix."""
    cs = {"chr1": 60000}
    cells = [[(50 * i, 120) for i in range(700)], [(90, 300), (99, length), (4000, 10)]]
    for strategy in ("insertion", "paired-insertion", "fragment"):
        m, _, (cp, pos, ln) = _tile(torch_gpu, cells, cs, 100, [], None, None, strategy)
        _same(m, otile.tile_matrix(cp, pos, ln, cs, 100, [], None, None, strategy))


@pytest.mark.parametrize("n_cells", [3, 1024, 8192])
@pytest.mark.parametrize("strategy", ["insertion", "fragment", "paired-insertion", "single"])
def test_segments_crowded_rows(torch_gpu, strategy, n_cells):
    """Rows whose counts are carried through many segments: 20,000 fragments on 16 kb with lengths up
    to 31 bins of 100 bases, one bin that holds many segments, and a chromosome's end amid them."""
    rng = np.random.default_rng(n_cells)
    cs = {"chr1": 16_000, "chr2": 3_000, "chr3": 9_000}
    def row(n, a, b):
        pos = np.sort(rng.integers(a, b, n))
        end = np.where(pos < 16_000, 16_000, np.where(pos < 19_000, 19_000, 28_000))
        return [(int(p), int(min(l, e - p))) for p, l, e in zip(pos, rng.integers(1, 3101, n), end)]
    cells = [row(20_000, 0, 16_000), row(6_000, 12_000, 28_000),
             [(5_000 + i // 2_000, 1 + (i * 37) % 3_050) for i in range(5_000)] + [(8_200, 100)] * 700]
    cells += [row(int(k), 0, 28_000) for k in rng.integers(0, 20, n_cells - 3)]
    m, _, (cp, pos, ln) = _tile(torch_gpu, cells, cs, 100, ["chr2"], None, None, strategy)
    _same(m, otile.tile_matrix(cp, pos, ln, cs, 100, ["chr2"], None, None, strategy))


def test_crowded_rows_take_no_longer(torch_gpu):
    """The work is linear in the fragments, however they crowd (on 16 kb a look back over the
    fragments within reach took ten times as long as the same number spread over 100 Mb)."""
    torch = torch_gpu
    from snapatac2_amd.pp import make_tile_matrix
    rng = np.random.default_rng(1)
    cs = {"chr1": 100_000_000}
    times = {}
    for width in (16_000, 90_000_000):
        pos = np.sort(rng.integers(0, width, 50_000))
        fr = _frags(torch, [[(int(p), int(l)) for p, l in zip(pos, rng.integers(30, 700, pos.size))]])[0]
        for _ in range(6):
            a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            a.record()
            make_tile_matrix(fr, cs)
            b.record()
            b.synchronize()
            times[width] = min(times.get(width, 1e9), a.elapsed_time(b))
    assert times[16_000] <= 3 * times[90_000_000], times
