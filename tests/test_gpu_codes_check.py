"""GPU tests of the PQ code check (``codes_check_kernel``, ``csrc/tms_check.hip``).

One bad code is planted at the first, last and inner places of code arrays that start and
end at every alignment, for limits on both sides of each form of the comparison (bytes below
and above 128, signed 16- and 32-bit), below and above the size where workgroups stop having
a verdict word each. It must be refused with the values torch finds; the largest valid code
must pass, and score as without the check.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _verdict(t, K):
    from tilemaxsim_amd import _lib
    lib = _lib.load()
    v, st = _lib.verdict_ptr(), _lib.stream_of(t)
    _lib.check(lib.tms_codes_check(t.data_ptr(), t.numel(), t.element_size(), K, v, st))
    return lib.tms_codes_verdict(v, st)


LIMITS = {"uint8": [1, 2, 100, 127, 128, 129, 200, 255], "int16": [1, 256, 32767, 32768, 40_000],
          "int32": [1, 300, 70_000, (1 << 31) - 1, 1 << 31]}


@pytest.mark.parametrize("dt,K", [(d, k) for d, ks in LIMITS.items() for k in ks])
def test_every_place_and_alignment(cuda, dt, K):
    import torch
    from tilemaxsim_amd._lib import TMS_ERR_BOUNDS, TMS_OK
    tdt = getattr(torch, dt)
    top = min(K - 1, torch.iinfo(tdt).max)
    for n in (1, 3, 16, 17, 63, 4099, 300_001):
        base = torch.full((n + 40,), top, dtype=tdt, device="cuda")
        base[::2] = 0
        for shift in (0, 1, 3, 7, 15):
            t = base[shift:shift + n]
            assert _verdict(t, K) == TMS_OK, (n, shift)
            for bad in {top + 1, torch.iinfo(tdt).min, torch.iinfo(tdt).max} - set(range(0, 2)):
                if not torch.iinfo(tdt).min <= bad <= torch.iinfo(tdt).max or 0 <= bad < K:
                    continue
                for at in sorted({0, 1 % n, n // 2, n - 1}):
                    keep = t[at].item()
                    t[at] = bad
                    assert _verdict(t, K) == TMS_ERR_BOUNDS, (n, shift, at, bad)
                    t[at] = keep
            around = base.clone()
            if K <= torch.iinfo(tdt).max:
                around[:] = K  # bad codes just outside the array are not read
                around[shift:shift + n] = 0
                assert _verdict(around[shift:shift + n], K) == TMS_OK, (n, shift)


@pytest.mark.parametrize("dt", ["uint8", "int16", "int32"])
def test_large(cuda, dt):
    import torch
    from tilemaxsim_amd._lib import TMS_ERR_BOUNDS, TMS_OK
    size = torch.iinfo(getattr(torch, dt)).bits // 8
    for extra in (0, 5):
        n = (33 << 20) // size + extra
        t = torch.zeros(n, dtype=getattr(torch, dt), device="cuda")
        assert _verdict(t, 100) == TMS_OK
        for at in (0, n // 3, n - 1):
            t[at] = 100
            assert _verdict(t, 100) == TMS_ERR_BOUNDS
            t[at] = 99
        assert _verdict(t, 100) == TMS_OK


@pytest.mark.parametrize("dt", ["uint8", "int16", "int32", "int64", "int8"])
def test_scores_and_refusals(cuda, dt):
    import torch
    import tilemaxsim_amd as tms
    rng = np.random.default_rng(3)
    book = torch.from_numpy(rng.standard_normal((16, 64, 4), dtype=np.float32)).half().cuda()
    Q = torch.from_numpy(rng.standard_normal((2, 32, 64), dtype=np.float32)).half().cuda()
    codes = torch.from_numpy(rng.integers(0, 64, (130, 21, 16))).to(getattr(torch, dt)).cuda()
    pq = tms.TileMaxSimPQ(book)
    for method in ("auto", "lut"):
        assert torch.equal(pq.score_batch(Q[0], codes, method), pq.score_batch(Q[0], codes, method, validate=False))
    assert torch.equal(pq.score_batch_queries(Q, codes), pq.score_batch_queries(Q, codes, validate=False))
    assert torch.equal(pq.score_single(Q[0], codes[0]), pq.score_batch(Q[0], codes[:1], validate=False)[0])
    for bad in (64, 100, -1):
        if dt == "uint8" and bad < 0:
            continue
        c = codes.clone()
        c[129, 20, 15] = bad
        found = rf"found \[{min(0, bad)}, {max(63, bad)}\]"
        for call in (lambda: pq.score_batch(Q[0], c), lambda: pq.score_batch(Q[0], c, "lut"),
                     lambda: pq.score_batch_queries(Q, c)):
            with pytest.raises(ValueError, match=found):
                call()
    wide = tms.TileMaxSimPQ(book.float())  # no MFMA path: the codes' error still comes first
    with pytest.raises(NotImplementedError):
        wide.score_batch(Q[0], codes, "mfma")
    with pytest.raises(ValueError, match="codes must lie"):
        wide.score_batch(Q[0], c, "mfma")
