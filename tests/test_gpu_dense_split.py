"""GPU parity of the general dense kernel's split documents (``dense_maxsim_kernel``, SPLIT).

Small calls of fixed-length documents split each over two or four waves (``tms_rules.h``, asked
here which calls do): tokens on both sides of a tile and of the tiles two and four waves need,
document counts on both sides of each split and of the last workgroup's share, queries in
registers and in up to the LDS that a split launch may take (80 KiB), and one past it that is
never split. A document must score the same bits as in a call too large to be split, and lie
within the fp32-accumulation bar of the float64 oracle.
"""
import numpy as np
import pytest

import accum_bar as bar
import rules
from oracle import maxsim_oracle as orc

pytestmark = pytest.mark.gpu


def _emb(rng, *shape):
    x = rng.standard_normal(shape, dtype=np.float32)
    return x / np.linalg.norm(x, axis=-1, keepdims=True)


@pytest.mark.parametrize("qdt,ddt,d", [("float16", "float16", 256), ("bfloat16", "bfloat16", 200), ("float16", "float16", 48),
                                       ("float16", "float16", 77), ("float32", "float32", 128), ("float32", "float32", 160),
                                       ("float32", "float16", 128), ("float32", "bfloat16", 384), ("float32", "float32", 512),
                                       ("float32", "float32", 640), ("bfloat16", "bfloat16", 1280), ("float32", "float32", 768)])
@pytest.mark.parametrize("nq,nd", [(32, 1), (32, 33), (40, 64), (32, 65), (7, 128), (70, 129), (32, 200)])
def test_split_bits(cuda, qdt, ddt, d, nq, nd):
    import torch
    import tilemaxsim_amd as tms
    rng = np.random.default_rng(nq + 7 * nd + d)
    Q = torch.from_numpy(_emb(rng, nq, d)).to(getattr(torch, qdt)).cuda()
    D = torch.from_numpy(_emb(rng, 130, nd, d)).to(getattr(torch, ddt)).cuda()
    whole = tms.flash_maxsim_batch(Q, D.repeat(17, 1, 1))  # 2,210 documents: one wave each
    split = {B: rules.dense_split(qdt, ddt, d, nq, B, nd) for B in range(1, 2211)}
    edges = [B for B in range(1, 2210) if split[B] != split[B + 1]]
    assert split[2210] == 1
    if (ddt, d) == ("float32", 768) or nd <= 16:  # LDS for one eight-wave workgroup; one tile
        assert not edges
    elif nd > 32:  # a second tile of 32 tokens
        assert split[1] > 1 and edges
    for B in sorted({1, 3, 130, 512, 513, 1024, 1025}.union(edges, [B + 1 for B in edges])):
        got = tms.flash_maxsim_batch(Q, D.repeat(-(-B // 130), 1, 1)[:B])
        assert torch.equal(got.view(torch.int32), whole[:B].view(torch.int32)), f"B={B}"
    Qn, Dn = Q.float().cpu().numpy(), D.float().cpu().numpy()
    if ddt == "float32":  # three of four bf16 products: 3 * 2^-16 of each term, beside the sums
        ref = orc.maxsim_f64(Qn, Dn)
        lim = (3 * 2.0 ** -16 + (3 * d + nq) * 2.0 ** -23) * orc.maxsim_f64(np.abs(Qn), np.abs(Dn))
    else:
        qsplit = None if qdt == ddt else ("fp16" if ddt == "float16" else "bf16")
        ref, lim = bar.with_bound(orc.maxsim_f64, Qn, Dn, qsplit=qsplit)
    bar.assert_scores(whole[:130].cpu().numpy(), ref, lim, "split")
