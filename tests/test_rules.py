"""CPU tests of the rules that pick a kernel's form (``csrc/tms_rules.h``)."""
import itertools

import pytest

import rules


def test_dense_split_bounds():
    """1, 2 or 4 waves a document, at most one a tile, and no more waves than run at once."""
    waves = rules.lib().dense_split_waves
    for tiles, lds, nqb, ks in itertools.product((0, 1, 2, 3, 4, 5, 12, 24, 60), (0, 16, 4096, 65536, 79 * 1024, 80 * 1024),
                                                 (1, 2), (0, 1, 2, 3, 4)):
        last = 4
        for B in (0, 1, 255, 256, 257, 384, 385, 512, 513, 768, 769, 1024, 1025, 1 << 40):
            w = waves(B, tiles, lds, nqb, ks)
            assert w in (1, 2, 4) and w <= max(1, tiles) and w <= last
            last = w
            if w > 1:
                per_cu = 2048 if ks else 1024 * min(2, 160 * 1024 // (lds + 256 + 512 * nqb))
                assert w * B <= per_cu
    assert waves(1, 60, 4096, 1, 0) == 4


@pytest.mark.parametrize("qdt,ddt,d,nq,nd,B,want", [
    # one workgroup a CU: 80 KiB of query fragments and the kernel's own LDS
    ("float16", "float16", 1280, 32, 180, 512, 2), ("float16", "float16", 1280, 32, 180, 600, 1),
    ("float16", "float16", 1280, 64, 33, 1024, 1), ("float32", "float32", 640, 32, 100, 768, 1),
    ("float32", "float32", 640, 32, 100, 300, 2), ("float16", "float16", 512, 32, 180, 1024, 2),
    # the query in registers: one wave a SIMD, more for little work a tile or long documents
    ("float32", "float32", 128, 64, 33, 600, 1), ("float32", "float32", 128, 32, 100, 600, 1),
    ("float32", "float32", 128, 64, 100, 300, 2), ("float32", "float32", 128, 64, 100, 256, 4),
    ("float32", "float32", 96, 64, 100, 768, 1), ("float32", "float32", 96, 64, 1000, 768, 2),
    ("float32", "float32", 64, 32, 400, 768, 2), ("float32", "float32", 128, 64, 1000, 768, 1)])
def test_dense_split_stays_where_it_is_faster(qdt, ddt, d, nq, nd, B, want):
    assert rules.dense_split(qdt, ddt, d, nq, B, nd) == want
