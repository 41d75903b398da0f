"""Where the fragment import changes its way: lines at the limits of the eight-character
parser (field lengths around 8 and 16 digits, lines around 64 characters, next to either
end of the text, every optional field), and sort keys of just 64 bits and just more (group,
position and value in one key or in two sorts), against the oracle, bit for bit."""
import numpy as np
import pytest

from oracle.fragments import import_text
from test_import_gpu import _check

pytestmark = pytest.mark.gpu

BIG = {"chr1": 2**32 - 1}


def _gpu(text, sizes, **kw):
    from snapatac2_amd.pp import import_fragment_text
    return import_fragment_text(text, sizes, **kw)


FORMS = [b"chr1\t%d\t%d\tAC" % (10**k, 10**k + 7) for k in range(10)]  # 1 to 10 digits
FORMS += [b"chr1\t" + b"%d".rjust(2, b"0") % 3 + b"\t%s\tACGT-1" % (b"0" * z + b"99") for z in (0, 5, 6, 7, 13, 14, 15, 18)]
FORMS += [b"chr1\t1\t9\t" + b"ACGT-" * 14 + b"A" * z for z in range(0, 3)]  # longer than 64
FORMS += [(b"chr1\t1\t9\t" + b"G" * 80)[:n] for n in (12, 13, 61, 62, 63, 64, 65, 66, 72)]  # barcodes up to the line's end
FORMS += [b"chr1\t1\t9\tAC\t%s" % c for c in (b"0", b"1", b".", b"99999999", b"4294967295", b"00000000005")]
FORMS += [b"chr1\t1\t9\tAC\t2\t%s" % c for c in (b".",)] + [b"chr1\t5\t9\tAC\t2\t.\textra\tmore"]
FORMS += [b"nochr\t1\t9\tAC", b"#chr1\t1\t9\tAC", b"", b"chr1\t7\t7\tAC", b"chr1\t1\t9\tA", b"chr1\t1\t9\t", b"\t1\t9\tAC",
          b"chr1\t1\t9\tAC\r", b"chr1\t1\t9\tAC\t3\r", b"chr12345678\t1\t9\tAC"]
STRANDED = [b"chr1\t1\t9\tAC\t2\t%s" % c for c in (b"+", b"-")] + [b"chr1\t1\t9\tAC\t.\t-\tx", b"chr1\t99999999\t100000007\tACGT\t1\t+"]


@pytest.mark.parametrize("sorted_bc", [True, False])
@pytest.mark.parametrize("fill", [0, 1, 40])
def test_line_forms(torch_gpu, fill, sorted_bc):
    """Every form between `fill` ordinary lines on either side: alone, the line is next to
    both ends of the text, where the loads of eight characters don't fit."""
    for forms, other in ((FORMS, b"chr1\t100\t250\tZZZZ\t1"), (STRANDED, b"chr1\t100\t250\tZZZZ\t1\t+")):
        for form in forms:
            for last in (b"\n", b""):
                text = (other + b"\n") * fill + form + b"\n" + (other.replace(b"ZZZZ", b"zzzz") + b"\n") * fill
                text = text[:-1] + last
                print(fill, form, last, flush=True)
                kw = dict(min_num_fragments=0, sorted_by_barcode=sorted_bc)
                _check(_gpu(text, BIG, **kw), import_text(text, BIG, **kw))


def _bits(x):
    return max(int(x).bit_length(), 1)


# (genome length, largest size, barcodes): key bits without the mark of unsorted input
KEYS = [(2**30 - 1, 2**29 - 1, 16), (2**30 - 1, 2**30 - 1, 16), (2**30 - 1, 2**31 - 1, 16), (2**30 - 1, 2**31 - 1, 17),
        (2**32 - 1, 2**32 - 1, 1), (2**32 - 1, 2**32 - 1, 2), (2**32 - 1, 2**31 - 1, 1), (2**20, 600, 1), (2**20, 600, 300)]


@pytest.mark.parametrize("total,size,n_bc", KEYS)
@pytest.mark.parametrize("sorted_bc", [True, False])
@pytest.mark.parametrize("single", [False, True])
def test_key_widths(torch_gpu, total, size, n_bc, sorted_bc, single):
    rng = np.random.default_rng(n_bc + size % 1000)
    if single:
        size = min(size // 2, 2**31 - 1)
    sizes = {"chrM": 1000, "chr1": total - 1000}
    n = 3000
    lines = []
    for i in range(n):
        chrom = ("chr1", "chr1", "chr1", "chrM", "chrU")[int(rng.integers(5))]
        ln = size if i == 7 else int(rng.integers(1, min(size, 500) + 1))
        start = 900 if i == 7 else int(rng.integers(0, 500 if chrom == "chrM" else total - 1000 - 600))
        if i == 7:
            chrom = "chr1"
        # a '-' record is stored by its last base, which has to lie in the chromosome
        strand = "\t" + ("-" if rng.random() < 0.5 and i != 7 else "+") if single else ""
        lines.append((f"bc{int(rng.integers(n_bc)):03d}x", f"{chrom}\t{start}\t{start + ln}\t", f"\t{int(rng.integers(1, 4))}{strand}"))
    if sorted_bc:
        lines.sort(key=lambda t: t[0])
    text = "\n".join(a + b + c for b, a, c in lines).encode()
    kw = dict(min_num_fragments=0, sorted_by_barcode=sorted_bc)
    ref = import_text(text, sizes, **kw)
    assert len(ref["barcodes"]) == min(n_bc, len(ref["barcodes"])) > 0
    _check(_gpu(text, sizes, **kw), ref)


@pytest.mark.parametrize("n", [1, 63, 64, 65, 5000])
@pytest.mark.parametrize("distinct", [True, False])
def test_groups_of_unsorted_lines(torch_gpu, n, distinct):
    """All barcodes different (the table at its fullest), or all records of one."""
    rng = np.random.default_rng(n)
    ids = rng.permutation(n) if distinct else np.zeros(n, int)
    text = b"".join(b"chr1\t%d\t%d\tcell%d\t%d\n" % (s, s + 50, i, 1 + s % 3) for i, s in zip(ids, rng.integers(0, 900, n)))
    kw = dict(min_num_fragments=0, sorted_by_barcode=False)
    _check(_gpu(text, {"chr1": 1000}, **kw), import_text(text, {"chr1": 1000}, **kw))


@pytest.mark.parametrize("width", [2, 8, 17, 100])
@pytest.mark.parametrize("between", [b"", b"# note\n", b"chr1\t5\t5\tdropped\n", b"\n"])
def test_runs_of_sorted_lines(torch_gpu, width, between):
    """Runs that begin and end next to the parser's rounds of 256 lines and blocks of 4096,
    barcodes that differ in their last character alone, and lines that are not kept between
    records of one barcode."""
    rng = np.random.default_rng(width)
    n = 4096 + 700
    cuts = np.zeros(n, int)
    cuts[[1, 2, 63, 64, 65, 255, 256, 257, 511, 513, 1000, 4095, 4096, 4097, 4400]] = 1
    run = np.cumsum(cuts)
    names = [b"A" * (width - 1) + bytes([65 + r]) if r % 3 else b"A" * (width - 2) + bytes([97 + r]) for r in range(run[-1] + 1)]
    text = b"".join((between if rng.random() < 0.02 else b"") + b"chr1\t%d\t%d\t%s\n" % (s, s + 30, names[r])
                    for r, s in zip(run, rng.integers(0, 900, n)))
    kw = dict(min_num_fragments=0)
    _check(_gpu(text, {"chr1": 1000}, **kw), import_text(text, {"chr1": 1000}, **kw))


@pytest.mark.parametrize("last", [b"\n", b""])
def test_lines_counted_again(torch_gpu, monkeypatch, last):
    """The index that counts the lines by itself, and a line count that does not match."""
    from snapatac2_amd import _lib
    text = b"".join(b"chr1\t%d\t%d\tb%d\n" % (s, s + 9, s // 300) for s in range(1, 5000, 3))[:-1] + last
    ref = import_text(text, {"chr1": 6000}, min_num_fragments=0)
    L, off = _lib.lib(), [0]
    monkeypatch.setattr(L, "snapgpu_frag_index_counted",
                        lambda t, nb, nl, c, cb, *rest: L.snapgpu_frag_index(t, nb, nl + off[0], *rest))
    _check(_gpu(text, {"chr1": 6000}, min_num_fragments=0), ref)
    off[0] = -1
    with pytest.raises(Exception, match="n_lines"):
        _gpu(text, {"chr1": 6000}, min_num_fragments=0)


@pytest.mark.parametrize("change", ["fewer", "moved", "more", "zeros", "ones"])
def test_count_workspace_of_another_text(torch_gpu, change):
    """A text that changed since its lines were counted, or a workspace that holds something
    else, is refused before anything reads the line starts."""
    import ctypes as C
    torch = torch_gpu
    from snapatac2_amd import _lib
    L = _lib.lib()
    line = b"chr1\t%05d\t99999\tcell\n"
    text = np.frombuffer(b"".join(line % i for i in range(8000)), np.uint8).copy()
    size = text.size
    assert size > 2 * 65536
    pad = torch.zeros(size + 16, dtype=torch.uint8, device="cuda")
    pad[:size] = torch.from_numpy(text).cuda()
    ws = torch.empty(L.snapgpu_frag_count_workspace_bytes(size), dtype=torch.uint8, device="cuda")
    n = C.c_int64(0)
    st = _lib.stream_ptr()
    _lib.check(L.snapgpu_frag_count_lines(pad.data_ptr(), size, ws.data_ptr(), ws.numel(), C.byref(n), st))
    assert n.value == 8000
    w = len(line % 0)
    if change in ("fewer", "moved"):
        pad[w - 1] = ord("x")  # one newline less in the first block of 64 KiB
    if change in ("more", "moved"):
        pad[size - 5] = 10     # one more in the last
    if change == "zeros":
        ws.zero_()
    if change == "ones":
        ws.fill_(255)
    from snapatac2_amd.pp._import import _name_table
    d_tab = torch.from_numpy(_name_table(["chr1"], [100_000], [0])).cuda()
    iws = torch.zeros(L.snapgpu_frag_workspace_bytes(size, n.value), dtype=torch.uint8, device="cuda")
    opt, summ = _lib.FragOptions(0, 0, 0, 1, 0), _lib.FragSummary()
    rc = L.snapgpu_frag_index_counted(pad.data_ptr(), size, n.value, ws.data_ptr(), ws.numel(), d_tab.data_ptr(), None,
                                      C.byref(opt), iws.data_ptr(), iws.numel(), C.byref(summ), st)
    assert rc == _lib.ERR_ARG
    assert b"count workspace" in L.snapgpu_last_error() or b"n_lines" in L.snapgpu_last_error()
