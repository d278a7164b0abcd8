"""GPU tests of what a refused ``*_checked`` call leaves behind: its scoring kernels score
nothing (every document NaN), whichever kernel the call's shape takes.

Offsets in random order make every ascending pair of them a document that is in range by
itself; together they are far longer than the corpus. The sizes here stay small enough that
scoring them after all would take milliseconds.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _words(torch, _lib):
    return (torch.zeros(_lib.TMS_CHECK_PARTS, dtype=torch.int64, pin_memory=True),
            torch.empty(_lib.TMS_CHECK_PARTS, dtype=torch.int64, device="cuda"))


def _offsets(torch, B, T, seed):
    rng = np.random.default_rng(seed)
    off = np.sort(rng.integers(0, T + 1, B + 1))
    off[0], off[-1] = 0, T
    while True:
        bad = rng.permutation(off)
        if np.any(np.diff(bad) < 0):
            return torch.from_numpy(off).cuda(), torch.from_numpy(bad).cuda()


# rows' type, query's type, d, queries, tokens per query, documents: the document-split kernel,
# the streaming, general and shared-tile ones, 16-bit and fp32, registers, LDS and memory queries
DENSE = [("float16", "float16", 128, 1, 32, 40), ("bfloat16", "bfloat16", 96, 1, 32, 700),
         ("float16", "float16", 128, 1, 32, 3000), ("float16", "float16", 128, 1, 160, 3000),
         ("float16", "float16", 64, 5, 32, 900), ("float16", "float16", 200, 1, 32, 300),
         ("bfloat16", "bfloat16", 2560, 1, 32, 50), ("float32", "float32", 128, 1, 32, 500),
         ("float32", "float32", 1280, 1, 32, 50), ("float32", "float32", 64, 4, 20, 300),
         ("float16", "float32", 128, 1, 32, 300), ("float16", "float32", 128, 3, 32, 300)]


@pytest.mark.parametrize("zero_pad", [0, 1])
@pytest.mark.parametrize("ddt,qdt,d,nQ,nq,B", DENSE)
def test_dense(cuda, ddt, qdt, d, nQ, nq, B, zero_pad):
    import torch
    from tilemaxsim_amd import _lib
    lib = _lib.load()
    T = 4 * B
    g = torch.Generator(device="cuda").manual_seed(B + d)
    Q = torch.randn(nQ, nq, d, device="cuda", generator=g).to(getattr(torch, qdt))
    D = torch.randn(T, d, device="cuda", generator=g).to(getattr(torch, ddt))
    good, bad = _offsets(torch, B, T, B)
    verdict, parts = _words(torch, _lib)
    code = _lib.dtype_code(D.dtype) | (_lib.TMS_QUERY_F32 if qdt != ddt else 0)
    stream = torch.cuda.current_stream().cuda_stream

    def call(off, out, parts_ptr, verdict_ptr):
        return lib.tms_maxsim_varlen_checked(Q.data_ptr(), nQ, nq, d, D.data_ptr(), T, off.data_ptr(), B, zero_pad, code,
                                             out.data_ptr(), parts_ptr, verdict_ptr, stream)

    out = torch.zeros(nQ, B, device="cuda")
    assert call(bad, out, parts.data_ptr(), verdict.data_ptr()) == _lib.TMS_ERR_BOUNDS
    torch.cuda.synchronize()
    assert bool(torch.isnan(out).all())
    # the same words and parts serve a call that is not refused
    assert call(good, out, parts.data_ptr(), verdict.data_ptr()) == _lib.TMS_OK
    torch.cuda.synchronize()
    assert not bool(torch.isnan(out).any())
    want = out.clone()
    # no verdict: each document is judged by itself
    assert call(good, out.zero_(), parts.data_ptr(), None) == _lib.TMS_OK
    torch.cuda.synchronize()
    assert torch.equal(out, want)
    odd = good.clone()
    odd[0] = -1
    assert call(odd, out, parts.data_ptr(), None) == _lib.TMS_OK
    torch.cuda.synchronize()
    assert bool(torch.isnan(out[:, 0]).all())
    if not zero_pad:
        assert torch.equal(out[:, 1:], want[:, 1:])
        # no room for what the check says: nothing is scored before the verdict
        mark = torch.full_like(out, 7.0)
        assert call(bad, mark, None, verdict.data_ptr()) == _lib.TMS_ERR_BOUNDS
        torch.cuda.synchronize()
        assert bool((mark == 7.0).all())
        assert call(good, out, None, verdict.data_ptr()) == _lib.TMS_OK
        torch.cuda.synchronize()
        assert torch.equal(out, want)


@pytest.mark.parametrize("B", [3, 3000])
def test_packed(cuda, B):
    import torch
    from tilemaxsim_amd import _lib
    lib = _lib.load()
    g = torch.Generator(device="cuda").manual_seed(B)
    lens = torch.randint(1, 6, (B,), device="cuda", generator=g)
    T = int(lens.sum())
    Q = torch.randn(32, 128, device="cuda", generator=g).half()
    D = torch.randn(T, 128, device="cuda", generator=g).half()
    lens[B // 2] = -1
    verdict, parts = _words(torch, _lib)
    out, off = torch.zeros(B, device="cuda"), torch.empty(B + 1, dtype=torch.int64, device="cuda")
    rc = lib.tms_maxsim_packed_checked(Q.data_ptr(), 32, 128, D.data_ptr(), T, lens.data_ptr(), B, 1, _lib.TMS_DTYPE_F16,
                                       out.data_ptr(), off.data_ptr(), parts.data_ptr(), verdict.data_ptr(),
                                       torch.cuda.current_stream().cuda_stream)
    assert rc == _lib.TMS_ERR_BOUNDS
    torch.cuda.synchronize()
    assert bool(torch.isnan(out).all())


@pytest.mark.parametrize("ids", [False, True])
@pytest.mark.parametrize("nQ,ndocs", [(1, 40), (1, 3000), (3, 900), (2, 3000)])
def test_residual(cuda, nQ, ndocs, ids):
    import torch
    from tilemaxsim_amd import _lib
    lib = _lib.load()
    g = torch.Generator(device="cuda").manual_seed(ndocs)
    T, d, nbits, ncent = 4 * ndocs, 128, 2, 16
    Q = torch.randn(nQ, 32, d, device="cuda", generator=g).half()
    cent = torch.randn(ncent, d, device="cuda", generator=g).half()
    weights = torch.randn(4, device="cuda", generator=g).half()
    codes = torch.randint(0, ncent, (T,), device="cuda", generator=g, dtype=torch.int32)
    res = torch.randint(0, 256, (T, d * nbits // 8), device="cuda", generator=g, dtype=torch.int32).to(torch.uint8)
    good, bad = _offsets(torch, ndocs, T, ndocs)
    verdict, parts = _words(torch, _lib)

    def call(off, pids, out, parts_ptr, verdict_ptr):
        return lib.tms_maxsim_residual_checked(
            Q.data_ptr(), nQ, 32, d, cent.data_ptr(), ncent, weights.data_ptr(), nbits, codes.data_ptr(), res.data_ptr(), T,
            off.data_ptr(), ndocs, _lib.ptr(pids), ndocs, 0, int(nQ > 1), out.data_ptr(), parts_ptr, verdict_ptr,
            torch.cuda.current_stream().cuda_stream)

    pids = torch.randperm(ndocs, device="cuda", generator=g) if ids else None
    out = torch.zeros(nQ, ndocs, device="cuda")
    for off in ([bad, good] if ids else [bad]):
        p = pids
        if off is good:  # an id out of range refuses the call, too
            p = pids.clone()
            p[ndocs // 2] = ndocs
        assert call(off, p, out.zero_(), parts.data_ptr(), verdict.data_ptr()) == _lib.TMS_ERR_BOUNDS
        torch.cuda.synchronize()
        assert bool(torch.isnan(out).all())
    assert call(good, pids, out, parts.data_ptr(), verdict.data_ptr()) == _lib.TMS_OK
    torch.cuda.synchronize()
    assert not bool(torch.isnan(out).any())
