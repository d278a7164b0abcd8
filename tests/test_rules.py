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


def test_topk_groups_fit():
    """k groups fit the selection, the maxima the workspace, the spans their stage."""
    lanes, workspace = rules.lib().topk_group_lanes, rules.lib().topk_workspace
    taken = 0
    for rows, n, k in itertools.product((1, 3, 256, 257, 513, 65535), (8, 4096, 4097, 5000, 24_000, 33_000, 131_073, 1 << 20, 4_200_000,
                                                                      1 << 24, (1 << 24) + 1, (1 << 32) - 1),
                                        (1, 7, 8, 9, 64, 100, 128, 129, 200, 300, 321, 512, 513, 1024)):
        lg = lanes(rows, n, k)
        if lg == 0:
            continue
        taken += 1
        keys, spans, per = (4096 if k <= 128 else 16384), -(-n // 1024), 1024 >> (lg + 2)
        assert 3 <= lg <= 6 and (4 << lg) * k <= keys and n > 4096
        direct = spans * per <= keys
        assert direct or (k <= spans <= 16384 and per * k <= keys)
        assert 4 * rows * spans * (per + (not direct)) <= workspace(rows, n, k)
    assert taken > 100


@pytest.mark.parametrize("rows,n,k,groups", [
    # more rows than run at once: short ones take the tournament
    (4096, 8192, 100, False), (10_000, 5000, 10, False), (4096, 5000, 128, False), (2048, 16_384, 200, False),
    (1000, 8192, 100, False), (257, 8192, 100, False), (256, 8192, 100, True), (2048, 40_000, 100, True), (512, 24_000, 100, True),
    # few groups for their k, and the tournament's slow last chunk
    (1, 5000, 128, False), (1, 6500, 128, True), (1, 4200, 128, True), (1, 5000, 100, True), (1, 16_384, 256, False),
    (1, 24_000, 200, True), (300, 20_000, 200, False),
    # large k needs much to save
    (1, 300_000, 512, False), (16, 100_000, 460, False), (64, 100_000, 512, True), (1, 1_000_000, 512, True),
    (32, 1_000_000, 100, True)])
def test_topk_groups_stay_where_they_are_faster(rows, n, k, groups):
    assert (rules.lib().topk_group_lanes(rows, n, k) > 0) == groups


@pytest.mark.parametrize("M,K,dsub,nQ,nq,tokens,alone", [
    (16, 256, 8, 2, 32, 524_288, True), (16, 256, 8, 2, 32, 524_287, False), (16, 256, 8, 3, 32, 1_179_647, False),
    (16, 256, 8, 3, 32, 1_179_648, True), (16, 64, 4, 3, 32, 1 << 21, False), (16, 64, 4, 3, 32, 3 << 20, True), (16, 256, 8, 6, 32, 10_240_000, True), (16, 256, 8, 7, 32, 25_600_000, False),
    # codebooks whose shared pass costs few queries, or whose own kernel is slow
    (64, 256, 2, 6, 32, 25_600_000, False), (64, 256, 2, 4, 32, 25_600_000, False), (64, 256, 2, 3, 32, 25_600_000, True),
    (4, 256, 32, 6, 32, 25_600_000, False), (4, 256, 32, 4, 32, 25_600_000, True), (32, 64, 2, 6, 32, 25_600_000, False), (16, 64, 4, 6, 32, 10_240_000, False),
    (16, 16, 8, 5, 32, 10_240_000, True), (16, 256, 8, 2, 64, 3_840_000, True), (16, 64, 4, 3, 64, 7_680_000, False)])
def test_pq_queries_go_alone_where_it_is_faster(M, K, dsub, nQ, nq, tokens, alone):
    assert bool(rules.lib().pq_per_query(nQ, -(-nq // 32), tokens, M, dsub, M * dsub * K * 2)) == alone
