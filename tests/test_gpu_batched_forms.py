"""GPU parity of the shared-tile kernel's workgroup forms (``tms_batched_kernel.h``).

A call of n query blocks takes passes of up to 32 blocks (16 for fp32 queries), each in the
smallest form that holds it: 4 waves of 1-4 blocks, or 8 waves of 2-4 (up to 256 documents
also 8 waves of 1 or 2 for 5 to 16 blocks). Cases sit on both
sides of every form's capacity, at queries of one to four blocks, with document counts on
both sides of one workgroup and of a round of them. Dense scores must be the bits of the
one-query kernels (the same products, and the same order of the sums over query tokens);
PQ and fp32 ones must lie within the fp32-accumulation bar of the float64 oracle.
"""
import numpy as np
import pytest

import accum_bar as bar
from oracle import maxsim_oracle as orc

pytestmark = pytest.mark.gpu

# (queries, tokens per query): blocks at each form's edges, and past one pass
FORMS = [(3, 32), (4, 32), (5, 20), (8, 32), (9, 32), (12, 7), (13, 32), (16, 32), (17, 32), (20, 32), (21, 32), (24, 32),
         (25, 32), (28, 32), (29, 32), (32, 32), (33, 32), (45, 32), (2, 64), (3, 40), (5, 64), (9, 64), (11, 64), (2, 96),
         (5, 96), (9, 96), (2, 128), (4, 100), (5, 128), (9, 128)]


def _emb(rng, *shape):
    x = rng.standard_normal(shape, dtype=np.float32)
    return x / np.linalg.norm(x, axis=-1, keepdims=True)


@pytest.mark.parametrize("d,B", [(128, 130), (96, 1), (64, 65), (32, 1100), (128, 300), (96, 257), (64, 400)])
@pytest.mark.parametrize("nQ,nq", FORMS)
def test_dense_bits(cuda, nQ, nq, d, B):
    import torch
    import tilemaxsim_amd as tms
    from tilemaxsim_amd import _lib
    rng = np.random.default_rng(nQ * 131 + nq + d + B)
    dt = torch.float16 if nQ % 2 else torch.bfloat16
    nd = int(rng.integers(1, 70))
    Qs = torch.from_numpy(_emb(rng, nQ, nq, d)).to(dt).cuda()
    D = torch.from_numpy(_emb(rng, B, nd, d)).to(dt).cuda()
    lens = rng.integers(0, nd + 1, B)
    lens[0] = nd
    offsets = torch.from_numpy(np.concatenate([[0], np.cumsum(lens)])).cuda()
    flat = D.view(-1, d)[:int(offsets[-1])]
    with _lib.rerank_limit(0):
        fixed = tms.flash_maxsim_batched_queries(Qs, D)
        varlen = tms.flash_maxsim_multi_doc_batched(Qs, flat, offsets)
        for q in {0, nQ // 2, nQ - 1}:
            if nq > 96:  # one query of four blocks takes the shared-tile kernel itself
                one = tms.flash_maxsim_batched_queries(Qs[q:q + 1], D)[0]
            else:
                one = tms.flash_maxsim_batch(Qs[q], D)
            assert torch.equal(fixed[q].view(torch.int32), one.view(torch.int32)), f"query {q}, fixed lengths"
            if nq <= 96:
                one = tms.flash_maxsim_multi_doc(Qs[q], flat, offsets)
                assert torch.equal(varlen[q].view(torch.int32), one.view(torch.int32)), f"query {q}, offsets"
    Qn, Dn = Qs.float().cpu().numpy(), D.float().cpu().numpy()
    for q in {0, nQ - 1}:
        ref, lim = bar.with_bound(orc.maxsim_f64, Qn[q], Dn)
        bar.assert_scores(fixed[q].cpu().numpy(), ref, lim, f"query {q}")


@pytest.mark.parametrize("qdt,ddt", [("float32", "float32"), ("float32", "float16"), ("float32", "bfloat16")])
@pytest.mark.parametrize("nQ,nq", [(3, 32), (4, 32), (5, 32), (8, 20), (9, 32), (12, 32), (13, 32), (17, 32), (2, 64), (5, 50)])
def test_fp32_queries(cuda, nQ, nq, qdt, ddt):
    import torch
    import tilemaxsim_amd as tms
    rng = np.random.default_rng(nQ * 7 + nq)
    Qs = torch.from_numpy(_emb(rng, nQ, nq, 128)).cuda()
    D = torch.from_numpy(_emb(rng, 70, 37, 128)).to(getattr(torch, ddt)).cuda()
    got = tms.flash_maxsim_batched_queries(Qs, D).cpu().numpy()
    for q in range(nQ):
        Qn, Dn = Qs[q].cpu().numpy(), D.float().cpu().numpy()
        if ddt == "float32":  # three of four bf16 products: 3 * 2^-16 of each term, beside the sums
            ref = orc.maxsim_f64(Qn, Dn)
            lim = (3 * 2.0 ** -16 + (3 * 128 + nq) * 2.0 ** -23) * orc.maxsim_f64(np.abs(Qn), np.abs(Dn))
        else:
            ref, lim = bar.with_bound(orc.maxsim_f64, Qn, Dn, qsplit="fp16" if ddt == "float16" else "bf16")
        bar.assert_scores(got[q], ref, lim, f"query {q}")


@pytest.mark.parametrize("M,K,dsub", [(16, 256, 8), (8, 100, 16), (4, 256, 32), (32, 256, 4), (16, 64, 4), (32, 64, 2)])
@pytest.mark.parametrize("nQ,nq,B", [(2, 32, 65), (4, 32, 300), (7, 32, 20), (9, 30, 130), (16, 32, 64), (20, 32, 40),
                                     (33, 32, 70), (3, 64, 12), (5, 100, 9), (2, 32, 17_000)])
def test_pq(cuda, M, K, dsub, nQ, nq, B):
    import torch
    import tilemaxsim_amd as tms
    rng = np.random.default_rng(M + K + nQ * 5 + B)
    nd = 33  # 17,000 x 33 tokens: two blocks go query by query
    book = torch.from_numpy(rng.standard_normal((M, K, dsub), dtype=np.float32)).half()
    codes = torch.from_numpy(rng.integers(0, K, (B, nd, M)).astype(np.uint8))
    Qs = torch.from_numpy(_emb(rng, nQ, nq, M * dsub)).half()
    got = tms.TileMaxSimPQ(book.cuda()).score_batch_queries(Qs.cuda(), codes.cuda()).cpu().numpy()
    pick = np.unique(np.concatenate([np.arange(min(B, 70)), np.arange(max(0, B - 70), B)]))
    c = codes.numpy()[pick]
    D = book.float().numpy()[np.arange(M), c].reshape(len(pick), nd, M * dsub)
    for q in {0, nQ // 2, nQ - 1}:
        ref, lim = bar.with_bound(orc.maxsim_f64, Qs[q].float().numpy(), D)
        bar.assert_scores(got[q][pick], ref, lim, f"query {q}")


@pytest.mark.parametrize("d,nbits", [(128, 2), (96, 1), (64, 4), (32, 2)])
@pytest.mark.parametrize("nQ,nq", [f for f in FORMS if f[1] <= 96])
def test_residual_bits(cuda, nQ, nq, d, nbits):
    """A query's scores over a residual index are the same bits in every form."""
    import torch
    import tilemaxsim_amd as tms
    rng = np.random.default_rng(nQ * 17 + nq + d)
    lens = rng.integers(0, 60, 140)
    offsets = torch.from_numpy(np.concatenate([[0], np.cumsum(lens)])).cuda()
    T = int(offsets[-1])
    index = (torch.from_numpy(rng.integers(0, 50, T).astype(np.int32)).cuda(),
             torch.from_numpy(rng.integers(0, 256, (T, d * nbits // 8)).astype(np.uint8)).cuda(),
             torch.from_numpy(_emb(rng, 50, d)).half().cuda(),
             torch.linspace(-0.1, 0.1, 1 << nbits).half().cuda(), nbits, offsets)
    Qs = torch.from_numpy(_emb(rng, nQ, nq, d)).half().cuda()
    got = tms.flashmaxsim_score_residual_batched(Qs, *index)
    for q in {0, nQ // 2, nQ - 1}:
        two = tms.flashmaxsim_score_residual_batched(torch.stack([Qs[q], Qs[0]]), *index)[0]
        assert torch.equal(got[q].view(torch.int32), two.view(torch.int32)), f"query {q}"


@pytest.mark.parametrize("qdt,dt", [("float16", "float16"), ("bfloat16", "bfloat16"), ("float32", "float32"),
                                    ("float32", "float16"), ("float32", "bfloat16")])
@pytest.mark.parametrize("d", [128, 96, 64, 32])
def test_few_documents(cuda, d, qdt, dt):
    """Up to 256 documents the blocks go over eight waves: the bits of the call of 257, whose
    blocks go over four, and (16-bit rows) of the one-query kernels."""
    import torch
    import tilemaxsim_amd as tms
    rng = np.random.default_rng(d)
    lens = rng.integers(0, 50, 257)
    lens[0], lens[255] = 49, 0
    offsets = torch.from_numpy(np.concatenate([[0], np.cumsum(lens)])).cuda()
    D = torch.from_numpy(_emb(rng, int(lens.sum()), d)).to(getattr(torch, dt)).cuda()
    for nQ, nq in ((5, 32), (8, 20), (9, 32), (13, 32), (16, 32), (17, 32), (3, 64), (4, 40), (8, 64), (2, 96), (5, 96)):
        Qs = torch.from_numpy(_emb(rng, nQ, nq, d)).to(getattr(torch, qdt)).cuda()
        many = tms.flash_maxsim_multi_doc_batched(Qs, D, offsets)
        for B in (256, 65, 1):
            few = tms.flash_maxsim_multi_doc_batched(Qs, D, offsets[:B + 1])
            assert torch.equal(few.view(torch.int32), many[:, :B].contiguous().view(torch.int32)), (nQ, nq, B)
        if qdt != "float32":
            one = torch.stack([tms.flash_maxsim_multi_doc(q, D, offsets) for q in Qs])
            assert torch.equal(many.view(torch.int32), one.view(torch.int32)), (nQ, nq)
