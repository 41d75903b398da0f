"""Host-side region handling of the peak and gene matrices (no GPU).

The gene path builds its promoter regions as (chrom, start, end) tuples
instead of formatting "chrom:start-end" strings and parsing them back; the
tuples must equal what parse_regions reads from those strings, including the
strip of the whole string, chromosome names holding ':' and duplicates, and
the string path must still raise where the reference's parse fails.
"""
import pytest

from snapatac2_amd import _lib
from snapatac2_amd.pp._genes import _promoter_tuples, promoter_regions
from snapatac2_amd.pp._peaks import parse_regions

TX = [dict(chrom="chr1", left=101, right=200, strand="+", transcript_id="t1"),
      dict(chrom="chr1", left=151, right=400, strand="+", transcript_id="t2"),
      dict(chrom="chr1", left=501, right=600, strand="-", transcript_id="t3"),
      dict(chrom="chr1", left=101, right=200, strand="+", transcript_id="t4"),  # same region as t1
      dict(chrom=" chr2", left=5, right=9, strand="-", transcript_id="t5"),  # leading space
      dict(chrom="HLA:A", left=1, right=1, strand="+", transcript_id="t6")]  # ':' in the name


@pytest.mark.parametrize("up,down,body", [(2000, 0, True), (20, 5, False), (0, 0, True), (0, 300, False)])
def test_promoter_tuples_match_string_parse(up, down, body):
    assert _promoter_tuples(TX, up, down, body) == parse_regions(promoter_regions(TX, up, down, body))[1]


def test_promoter_tuples_known_values():
    regs = _promoter_tuples(TX, 20, 0, True)
    assert regs[:3] == [("chr1", 80, 199), ("chr1", 130, 399), ("chr1", 500, 619)]
    assert len(regs) == 5  # t4 repeats t1


def test_negative_end_falls_back_to_the_string_error():
    tx = [dict(chrom="chr1", left=0, right=0, strand="+", transcript_id="t")]
    assert _promoter_tuples(tx, 0, 0, True) is None
    with pytest.raises(_lib.PanicException):
        parse_regions(promoter_regions(tx, 0, 0, True))


def test_missing_strand_raises():
    tx = [dict(chrom="chr1", left=1, right=5, strand=".", transcript_id="t")]
    with pytest.raises(_lib.PanicException):
        _promoter_tuples(tx, 0, 0, True)


def test_parse_regions_distinct_first_occurrence():
    names, regs = parse_regions(["chr1:5-10", " chr1:5-10 ", "chr1:005-10", "chr2:1-2", "chr1:5-10"])
    assert names == ["chr1:5-10", "chr2:1-2"] and regs == [("chr1", 5, 10), ("chr2", 1, 2)]
    for bad in ["chr1:5", "chr1-5-10", "chr1:-5-10", "chr1:a-b"]:
        with pytest.raises(_lib.PanicException):
            parse_regions([bad])


# --- select_features' whitelist / blacklist (intersect_bed) ----------------

from oracle import peaks as opeaks  # noqa: E402
from snapatac2_amd.pp._regions import parse_range_names, read_bed3  # noqa: E402

BED = [("chr1", 100, 200), ("chr1", 500, 501), ("chr2", 0, 10), ("chrX", 1000, 2000)]


@pytest.mark.parametrize("name,expect", [
    ("chr1:0-100", False),     # ends where the region starts (half-open)
    ("chr1:0-101", True),
    ("chr1:200-300", False),   # starts where the region ends
    ("chr1:199-200", True),
    ("chr1:120-130", True),    # inside
    ("chr1:50-600", True),     # contains both chr1 regions
    ("chr1:501-502", False),
    ("chr1:500-500", False),   # empty query at a region's start
    ("chr1:150-150", True),    # empty query strictly inside
    ("chr2:9-10", True),
    ("chr3:100-200", False),   # chromosome without regions
    ("chrX:1999-5000", True),
])
def test_oracle_intersect_bed_hand_cases(name, expect):
    assert opeaks.intersect_bed([name], BED)[0] == expect


def test_read_bed3_plain_gzip_and_errors(tmp_path):
    import gzip
    text = "chr1\t100\t200\tname\t0\t+\nchr2\t0\t10\n\nchrX\t1000\t2000\n"
    p = tmp_path / "a.bed"
    p.write_text(text)
    g = tmp_path / "a.bed.gz"
    with gzip.open(g, "wt") as f:
        f.write(text)
    want = [("chr1", 100, 200), ("chr2", 0, 10), ("chrX", 1000, 2000)]
    assert read_bed3(p) == want and read_bed3(g) == want
    bad = tmp_path / "b.bed"
    bad.write_text("chr1\t100\n")
    with pytest.raises(_lib.PanicException):
        read_bed3(bad)
    bad.write_text("track name=x\n")
    with pytest.raises(_lib.PanicException):
        read_bed3(bad)


def test_parse_range_names():
    ch, c, s, e = parse_range_names(["chr1:1-500", "HLA:A:5-9", " chr2:0-3 ", "chr1:7-8"])
    assert [ch[k] for k in c] == ["chr1", "HLA:A", "chr2", "chr1"]
    assert list(s) == [1, 5, 0, 7] and list(e) == [500, 9, 3, 8]
    with pytest.raises(_lib.PanicException):
        parse_range_names(["chr1_100_200"])


def test_bin_index_ranges_equal_the_names():
    from snapatac2_amd.genome import BinIndex
    bi = BinIndex({"chr1": 1234, "chr10": 500, "chr2": 1}, 500)
    ch, c, s, e = bi.ranges()
    assert [f"{ch[k]}:{a}-{b}" for k, a, b in zip(c, s, e)] == list(bi.to_numpy())
    assert list(bi.to_numpy()) == ["chr1:0-500", "chr1:500-1000", "chr1:1000-1234", "chr10:0-500", "chr2:0-1"]


# --- the native parse of the peak matrix ---------------------------

import numpy as np  # noqa: E402

from snapatac2_amd.pp._peaks import RegionArrays, parse_region_arrays  # noqa: E402

CHROMS = ["chr1", "chr2", "HLA:A", "é", "chr1\0x"]
PLAIN = ["chr2:1-2", "chr1:5-10", "chr1:0-0", "chr1:5-10", "HLA:A:7-9", ":3-4", "chrU:5-10", "chr1:5-11", "chr1:50-1",
         "chr2:1-2", "chrU:5-10", "chr1:999999999999999999-1000000000000000"]
EXOTIC = [" chr1:5-10 ", "chr1:005-10", "chr1:+5-10", "chr1: 5-10", "é:5-10", "chr1:1_0-20", "chr1:٥-10", "\udc80:1-2",
          "chr1\0x:1-2", "chr1:5-10\t", "chr\n1:5-10", "chr1:9223372036854775807-1"]
BAD = ["", "chr1:5", "chr1-5-10", "chr1:-5-10", "chr1:a-b", "chr1:5-", "chr1:5-6-7", "chr1:5--7", "chr1:-", "\n"]


@pytest.mark.parametrize("items", [[], PLAIN, *([x] for x in PLAIN), *([x] for x in EXOTIC),
                                   *(PLAIN + [x] + PLAIN for x in EXOTIC)])
@pytest.mark.parametrize("chroms", [CHROMS, CHROMS[:3], []])
def test_region_arrays_equal_the_parse(items, chroms):
    names, regs = parse_regions(items)
    got, arr = parse_region_arrays(items, chroms)
    want = RegionArrays.of(regs, chroms)
    assert got == names
    for a in ("chrom", "start", "end"):
        assert np.array_equal(getattr(arr, a), getattr(want, a)), a


@pytest.mark.parametrize("bad", BAD)
def test_region_arrays_refuse_what_the_parse_refuses(bad):
    for items in ([bad], PLAIN + [bad], [bad] + PLAIN):
        with pytest.raises(_lib.PanicException):
            parse_region_arrays(items, CHROMS)
