"""GPU tests of the checked entry points (``csrc/tms_check.hip``): document bounds are
checked, and the zero padding's length found, by a kernel in front of the scoring kernel.

Document counts sit on both sides of one workgroup's share, of the scan's wave, tile and
list limits, and of the most workgroups a check takes; a bad entry is planted at the first,
an inner and the last place and must be refused, as must one only a pid reaches. Accepted
calls must give the bits of the entry points that take the padding length from the host.
Streams and threads run calls at the same time, and a capture is refused.
"""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

COUNTS = [1, 2, 63, 65, 1023, 1024, 1025, 2048, 2049, 16384, 16385, 140_000]


def _docs(B, d=32, hi=5, seed=0):
    import torch
    g = torch.Generator(device="cuda").manual_seed(seed + B)
    lens = torch.randint(0, hi, (B,), generator=g, device="cuda")
    lens[B // 2] = hi + 3  # the longest document: not in the first workgroup of a long list
    T = int(lens.sum())
    D = torch.nn.functional.normalize(torch.randn(T, d, generator=g, device="cuda"), dim=-1).half()
    Q = torch.nn.functional.normalize(torch.randn(32, d, generator=g, device="cuda"), dim=-1).half()
    return Q, D, lens, torch.cat([lens.new_zeros(1), lens.cumsum(0)])


def _padded(Q, D, offsets, pad_len):
    import torch
    from tilemaxsim_amd import _lib
    B = offsets.numel() - 1
    out = torch.empty(B, device="cuda")
    _lib.check(_lib.load().tms_maxsim_varlen_padded(Q.data_ptr(), Q.shape[0], Q.shape[1], D.data_ptr(), D.shape[0],
                                                    offsets.data_ptr(), B, pad_len, _lib.TMS_DTYPE_F16, out.data_ptr(),
                                                    _lib.stream_of(Q)))
    return out


def _same(a, b):
    import torch
    return torch.equal(a.view(torch.int32), b.view(torch.int32))


@pytest.mark.parametrize("B", COUNTS)
def test_packed_and_varlen(cuda, B):
    import torch
    import tilemaxsim_amd as tms
    Q, D, lens, offsets = _docs(B)
    pad = int(lens.max())
    want = _padded(Q, D, offsets, pad)
    assert _same(tms.flashmaxsim_score_packed(Q, D, lens), want)
    assert _same(tms.flashmaxsim_score_packed(Q, D, lens.to(torch.int32).cpu(), padding="zeros"), want)
    # a strided view of the lengths, and rows past the documents
    wide = torch.stack([lens, lens + 1], 1)[:, 0]
    assert _same(tms.flashmaxsim_score_packed(Q, torch.cat([D, D[:1]]), wide), want)
    plain = tms.flash_maxsim_multi_doc(Q, D, offsets, validate=False)
    assert _same(tms.flash_maxsim_multi_doc(Q, D, offsets), plain)
    assert _same(tms.flashmaxsim_score_packed(Q, D, lens, padding="mask"), plain)
    Qs = torch.stack([Q, Q.flip(0), Q, Q])
    many = tms.flash_maxsim_multi_doc_batched(Qs, D, offsets, validate=False)
    assert _same(tms.flash_maxsim_multi_doc_batched(Qs, D, offsets), many)
    zeros = tms.flashmaxsim_score_packed_batched(Qs, D, lens)
    assert torch.equal(zeros[0], want) and torch.equal(zeros[3], want)


@pytest.mark.parametrize("B", COUNTS)
def test_bad_bounds_are_refused(cuda, B):
    import torch
    import tilemaxsim_amd as tms
    Q, D, lens, offsets = _docs(B)
    T = D.shape[0]
    want = tms.flashmaxsim_score_packed(Q, D, lens)
    for at in sorted({0, B // 3, B - 1}):
        bad = lens.clone()
        bad[at] = -1
        with pytest.raises(ValueError, match="D_lengths must be >= 0"):
            tms.flashmaxsim_score_packed(Q, D, bad)
        bad = lens.clone()
        bad[at] += 1  # one token more than there are
        with pytest.raises(ValueError, match="D_lengths must be >= 0"):
            tms.flashmaxsim_score_packed(Q, D, bad)
        bad[at] = torch.iinfo(torch.int64).max  # sums that wrap
        with pytest.raises(ValueError):
            tms.flashmaxsim_score_packed(Q, D, bad)
        bad = offsets.clone()
        bad[at + 1] = T + 1 if at == B - 1 else bad[at + 2] + 1
        for call in (lambda: tms.flash_maxsim_multi_doc(Q, D, bad),
                     lambda: tms.flash_maxsim_multi_doc_batched(torch.stack([Q, Q]), D, bad),
                     lambda: tms.flash_maxsim_multi_doc_batched(Q[None][:0], D, bad)):
            with pytest.raises(ValueError, match="non-decreasing within"):
                call()
    bad = offsets.clone()
    bad[0] = -1
    with pytest.raises(ValueError):
        tms.flash_maxsim_multi_doc(Q, D, bad)
    assert _same(tms.flashmaxsim_score_packed(Q, D, lens), want)  # a refusal leaves nothing behind


@pytest.mark.parametrize("ndocs,B", [(1, 1), (70, 5), (3000, 3000), (140_000, 1100), (500, 20_000)])
def test_residual(cuda, ndocs, B):
    import torch
    import tilemaxsim_amd as tms
    g = torch.Generator(device="cuda").manual_seed(ndocs)
    lens = torch.randint(0, 6, (ndocs,), generator=g, device="cuda")
    lens[ndocs // 2] = 9
    offsets = torch.cat([lens.new_zeros(1), lens.cumsum(0)])
    T = int(offsets[-1])
    cent = torch.nn.functional.normalize(torch.randn(64, 64, generator=g, device="cuda"), dim=-1).half()
    codes = torch.randint(0, 64, (T,), generator=g, device="cuda", dtype=torch.int32)
    res = torch.randint(0, 256, (T, 16), generator=g, device="cuda", dtype=torch.uint8)
    w = torch.tensor([-.05, -.01, .01, .05], device="cuda").half()
    Q = torch.nn.functional.normalize(torch.randn(32, 64, generator=g, device="cuda"), dim=-1).half()
    pids = torch.randint(0, ndocs, (B,), generator=g, device="cuda")
    index = (codes, res, cent, w, 2)
    docs = tms.decompress_residual(*index)
    for p in (pids, None):
        n = B if p is not None else ndocs
        use = lens[p] if p is not None else lens
        for padding in ("zeros", "mask"):
            one = tms.flashmaxsim_score_residual(Q, *index, offsets, p, padding=padding)
            assert _same(one, tms.flashmaxsim_score_residual(Q, *index, offsets, p, padding=padding, validate=False))
            many = tms.flashmaxsim_score_residual_batched(torch.stack([Q, Q]), *index, offsets, p, padding=padding)
            assert one.shape == (n,) and many.shape == (2, n)
            # MaxSim of the decompressed tokens, each document's padding as asked: the decoded
            # values differ by their fp16 rounding, 2^-11 of each term and of the norm
            flat = tms.flash_maxsim_multi_doc(Q, docs, offsets, validate=False)
            flat = flat[p] if p is not None else flat
            if padding == "zeros":
                short = use < use.max()
                assert bool((one[short] >= 0).all()) and bool((many[0][short] >= 0).all())
                keep = ~short
            else:
                keep = use > 0
                assert bool(torch.isneginf(one[~keep]).all())
            assert torch.allclose(one[keep], flat[keep], atol=32 * 2.0 ** -10, rtol=0)
            assert torch.allclose(many[0][keep], flat[keep], atol=32 * 2.0 ** -10, rtol=0)
    bad_off = offsets.clone()
    bad_off[ndocs] = T + 1
    for bad in (-1, ndocs):
        for at in {0, B - 1}:
            q = pids.clone()
            q[at] = bad
            with pytest.raises(ValueError, match="pids within"):
                tms.flashmaxsim_score_residual(Q, *index, offsets, q)
    for p in (pids[:1] * 0, None):  # offsets that no scored document reads are refused too
        with pytest.raises(ValueError, match="pids within"):
            tms.flashmaxsim_score_residual(Q, *index, bad_off, p, padding="mask")
        with pytest.raises(ValueError, match="pids within"):
            tms.flashmaxsim_score_residual_batched(torch.stack([Q, Q]), *index, bad_off, p)


def test_threads_and_streams(cuda):
    import torch
    import tilemaxsim_amd as tms
    sets = [_docs(B, d=128, hi=40, seed=7) for B in (50, 700, 3000, 20_000)]
    want = [tms.flashmaxsim_score_packed(Q, D, lens) for Q, D, lens, _ in sets]
    torch.cuda.synchronize()
    wrong = []

    def work(k):
        st = torch.cuda.Stream()
        with torch.cuda.stream(st):
            for i in range(30):
                Q, D, lens, offsets = sets[(i + k) % 4]
                if not _same(tms.flashmaxsim_score_packed(Q, D, lens), want[(i + k) % 4]):
                    wrong.append((k, i))
                bad = offsets.clone()
                bad[1] = -1
                try:
                    tms.flash_maxsim_multi_doc(Q, D, bad)
                    wrong.append((k, i, "accepted"))
                except ValueError:
                    pass

    threads = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong


def test_default_device(cuda):
    """Checked calls under a default device, in a thread that has made none before."""
    import torch
    import tilemaxsim_amd as tms
    Q, D, lens, offsets = _docs(70, d=64)
    pq = tms.TileMaxSimPQ(torch.randn(8, 16, 8, device="cuda").half())
    codes = torch.randint(0, 16, (30, 20, 8), device="cuda", dtype=torch.int32)
    calls = [lambda: tms.flash_maxsim_multi_doc(Q, D, offsets), lambda: tms.flashmaxsim_score_packed(Q, D, lens),
             lambda: tms.flash_maxsim_multi_doc_batched(torch.stack([Q, Q, Q]), D, offsets),
             lambda: pq.score_batch(Q, codes)]
    want = [c() for c in calls]
    got, bad = [], offsets.clone()
    bad[3] = -1

    def work():
        for dev in ("cuda", "cpu"):
            with torch.device(dev):
                got.append([c() for c in calls])
                with pytest.raises(ValueError):
                    tms.flash_maxsim_multi_doc(Q, D, bad)

    t = threading.Thread(target=work)
    t.start()
    t.join()
    assert len(got) == 2 and all(_same(a, b) for g in got for a, b in zip(g, want))


def test_capture_is_refused(cuda):
    import torch
    import tilemaxsim_amd as tms
    from tilemaxsim_amd._lib import TileMaxSimError
    Q, D, lens, offsets = _docs(100)
    want = tms.flash_maxsim_multi_doc(Q, D, offsets)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        with pytest.raises(TileMaxSimError, match="capture"):
            tms.flash_maxsim_multi_doc(Q, D, offsets)
        with pytest.raises(TileMaxSimError, match="capture"):
            tms.flashmaxsim_score_packed(Q, D, lens)
        got = tms.flash_maxsim_multi_doc(Q, D, offsets, validate=False)
    g.replay()
    assert _same(got, want)


def test_residual_padding_length_under_capture(cuda):
    """Without the check nothing is waited for, and a replay finds the padding's length itself."""
    import torch
    import tilemaxsim_amd as tms
    g = torch.Generator(device="cuda").manual_seed(3)
    lens = torch.randint(1, 9, (300,), generator=g, device="cuda")
    offsets = torch.cat([lens.new_zeros(1), lens.cumsum(0)])
    T = int(offsets[-1])
    cent = torch.nn.functional.normalize(torch.randn(64, 64, generator=g, device="cuda"), dim=-1).half()
    index = (torch.randint(0, 64, (T,), generator=g, device="cuda", dtype=torch.int32),
             torch.randint(0, 256, (T, 16), generator=g, device="cuda", dtype=torch.uint8), cent,
             torch.tensor([-.05, -.01, .01, .05], device="cuda").half(), 2, offsets)
    Q = torch.nn.functional.normalize(torch.randn(32, 64, generator=g, device="cuda"), dim=-1).half()
    order = torch.argsort(lens)
    pids = order[:100].clone()

    def call():
        return tms.flashmaxsim_score_residual(Q, *index, pids, validate=False)

    call()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = call()
    for lo in (0, 100, 200, 50):  # candidates of other longest lengths
        pids.copy_(order[lo:lo + 100])
        graph.replay()
        torch.cuda.synchronize()
        assert _same(out, call())
