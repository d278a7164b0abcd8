"""GPU parity of the general dense kernel's split documents (``dense_maxsim_kernel``, SPLIT).

Calls of up to 1,024 fixed-length documents split each over two or four waves: tokens on both
sides of a tile and of the tiles two and four waves need, document counts on both sides of
each split and of the last workgroup's share. A document must score the same bits as in a
call too large to be split, and lie within the fp32-accumulation bar of the float64 oracle.
"""
import numpy as np
import pytest

import accum_bar as bar
from oracle import maxsim_oracle as orc

pytestmark = pytest.mark.gpu


def _emb(rng, *shape):
    x = rng.standard_normal(shape, dtype=np.float32)
    return x / np.linalg.norm(x, axis=-1, keepdims=True)


@pytest.mark.parametrize("qdt,ddt,d", [("float16", "float16", 256), ("bfloat16", "bfloat16", 200), ("float16", "float16", 48),
                                       ("float16", "float16", 77), ("float32", "float32", 128), ("float32", "float32", 160),
                                       ("float32", "float16", 128), ("float32", "bfloat16", 384), ("float32", "float32", 768)])
@pytest.mark.parametrize("nq,nd", [(32, 1), (32, 33), (40, 64), (32, 65), (7, 128), (70, 129), (32, 200)])
def test_split_bits(cuda, qdt, ddt, d, nq, nd):
    import torch
    import tilemaxsim_amd as tms
    rng = np.random.default_rng(nq + 7 * nd + d)
    Q = torch.from_numpy(_emb(rng, nq, d)).to(getattr(torch, qdt)).cuda()
    D = torch.from_numpy(_emb(rng, 130, nd, d)).to(getattr(torch, ddt)).cuda()
    whole = tms.flash_maxsim_batch(Q, D.repeat(17, 1, 1))  # 2,210 documents: one wave each
    for B in (1, 3, 130):
        got = tms.flash_maxsim_batch(Q, D[:B])
        assert torch.equal(got.view(torch.int32), whole[:B].view(torch.int32)), f"B={B}"
    for B in (512, 513, 1024, 1025):
        got = tms.flash_maxsim_batch(Q, D.repeat(8, 1, 1)[:B])
        assert torch.equal(got.view(torch.int32), whole[:B].view(torch.int32)), f"B={B}"
    Qn, Dn = Q.float().cpu().numpy(), D.float().cpu().numpy()
    if ddt == "float32":  # three of four bf16 products: 3 * 2^-16 of each term, beside the sums
        ref = orc.maxsim_f64(Qn, Dn)
        lim = (3 * 2.0 ** -16 + (3 * d + nq) * 2.0 ** -23) * orc.maxsim_f64(np.abs(Qn), np.abs(Dn))
    else:
        qsplit = None if qdt == ddt else ("fp16" if ddt == "float16" else "bf16")
        ref, lim = bar.with_bound(orc.maxsim_f64, Qn, Dn, qsplit=qsplit)
    bar.assert_scores(whole[:130].cpu().numpy(), ref, lim, "split")
