"""GPU parity of the masked streaming kernel (``stream_maxsim_kernel``, ``ST_MASKED``).

Masked documents of at most 1,024 tokens are walked by the tiles that hold a real token;
a masked-out row of such a tile reads the tile's first real row. Cases sit where that can
go wrong: documents of one tile and of 64 (a wave's lanes hold one tile's bits each) and
one token past that limit (the general kernel), partial last tiles, tiles without a real
token at the start, inside and at the end, documents without any, masks of every
alignment, waves with several documents and a short last wave. Scores must lie within the
fp32-accumulation bar of the float64 oracle, with -inf exactly where it has it; masked-out
rows hold infinities and NaN, which must not reach a score (the kernel never reads them).
"""
import numpy as np
import pytest

import accum_bar as bar
from oracle import maxsim_oracle as orc

pytestmark = pytest.mark.gpu

CASES = [(32, 1, 128, 5), (32, 16, 64, 9), (32, 17, 128, 70), (32, 33, 96, 33), (20, 180, 128, 67), (33, 181, 128, 13),
         (70, 90, 64, 31), (32, 1023, 128, 3), (32, 1024, 128, 3), (32, 1025, 32, 3), (32, 12, 128, 40_000),
         (32, 180, 32, 20_001)]


def _mask(rng, B, nd, pattern):
    if pattern == "prefix":
        return np.arange(nd) < rng.integers(0, nd + 1, (B, 1))
    if pattern == "random":
        m = rng.random((B, nd)) < 0.5
        m[:: 7] = False
        return m
    # one real token in a few tiles, the others empty
    m = np.zeros((B, nd), bool)
    for b in range(0, B, max(1, B // 500)):
        m[b, rng.integers(0, nd, 1 + b % 3)] = True
    m[0] = False
    m[0, -1] = True
    return m


@pytest.mark.parametrize("pattern", ["prefix", "random", "sparse"])
@pytest.mark.parametrize("nq,nd,d,B", CASES)
def test_masked_stream(cuda, nq, nd, d, B, pattern):
    import torch
    from tilemaxsim_amd import _lib, maxsim_score
    rng = np.random.default_rng(nq + 31 * nd + d + B)
    dt = torch.bfloat16 if (nd + B) % 2 else torch.float16

    def emb(*shape):
        x = rng.standard_normal(shape, dtype=np.float32)
        t = torch.from_numpy(x / np.linalg.norm(x, axis=-1, keepdims=True)).to(dt)
        return t, t.float().numpy()

    (Qt, Q), (Dt, D) = emb(nq, d), emb(B, nd, d)
    mask = _mask(rng, B, nd, pattern)
    if nd <= 1024:  # the general kernel reads masked-out rows
        Dt[torch.from_numpy(~mask)] = float("nan")
        Dt[:, ::2][torch.from_numpy(~mask[:, ::2])] = float("inf")
    pick = np.unique(np.concatenate([np.arange(min(B, 64)), np.arange(max(0, B - 130), B)]))
    ref, lim = bar.with_bound(orc.maxsim_masked, Q, np.where(mask[pick][:, :, None], D[pick], 0), mask[pick], f64=True)
    flat = torch.zeros(B * nd + 3, dtype=torch.uint8, device="cuda")
    for shift in (0, 1):  # a 4-byte aligned mask, and one that is not
        m = flat[shift:shift + B * nd].view(B, nd)
        m.copy_(torch.from_numpy(mask.astype(np.uint8) * 255))
        with _lib.rerank_limit(0):
            got = maxsim_score(Qt.cuda(), Dt.cuda(), m).cpu().numpy()
        got, empty = got[pick].astype(np.float64), ~mask[pick].any(1)
        assert np.array_equal(np.isneginf(got), empty) and not np.isnan(got).any()
        bar.assert_scores(got[~empty], ref[~empty], lim[~empty], f"masked {pattern} shift {shift}")
