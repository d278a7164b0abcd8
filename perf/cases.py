"""The calls whose speed is tracked: what a late-interaction search service asks of this
package, from one reranking call to a pass over a corpus.

A case is a dict of plain values. ``prepare`` makes what a program holds before the call
(embeddings, index arrays, a codebook object), ``run`` is one call through the package's
public functions with their default options, ``exact`` the same result from plain torch in
64 bits. Document lengths of variable-length and padded corpora are drawn from
U[lo, hi]; embeddings are L2-normalised Gaussian tokens unless ``raw`` is set.
"""
import math

import torch

import tilemaxsim_amd as tms

DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32}
SIZE = {"fp16": 2, "bf16": 2, "fp32": 4}
CODES = {"u8": torch.uint8, "i16": torch.int16, "i32": torch.int32}
CHUNK = 1 << 20  # tokens made or checked at a time


def listed():
    return [
        # One query against the candidates of a first stage, best 100 returned: the
        # smallest serving call (256 candidates padded to 180 tokens).
        dict(name="rerank_256", kind="rerank", B=256, Nd=180, d=128, nq=32, dtype="fp16", k=100),
        # The last stage of a PLAID search: packed candidate tokens and their lengths.
        dict(name="packed_1024", kind="packed", B=1024, lo=32, hi=300, d=128, nq=32, dtype="fp16"),
        # The same stage straight from a ColBERTv2 index (2 bits a dimension) of 100,000
        # documents: 1,024 candidate ids.
        dict(name="residual_1024", kind="residual", B=1024, docs=100_000, lo=32, hi=300, d=128, nq=32, nbits=2,
             ncent=1 << 16),
        # Padded documents with a token mask (documents shorter than 180 tokens), a medium
        # corpus scored in one call.
        dict(name="masked_20k", kind="masked", B=20_000, Nd=180, lo=32, hi=180, d=128, nq=32, dtype="fp16"),
        # One query against 10,000 documents of 128 tokens: the usual benchmark size.
        dict(name="dense_10k", kind="dense", B=10_000, Nd=128, d=128, nq=32, dtype="fp16"),
        # The same in fp32, unnormalised, as a precision check runs it.
        dict(name="dense_10k_fp32", kind="dense", B=10_000, Nd=128, d=128, nq=32, dtype="fp32", raw=True),
        # Exhaustive scoring of a corpus, one query at a time: the largest call.
        dict(name="dense_400k", kind="dense", B=400_000, Nd=180, d=128, nq=32, dtype="fp16"),
        # Wide embeddings, the d-tiled path, in bf16.
        dict(name="dense_d768", kind="dense", B=50_000, Nd=128, d=768, nq=32, dtype="bf16"),
        # A variable-length corpus as one flat token buffer with offsets.
        dict(name="varlen_200k", kind="varlen", B=200_000, lo=32, hi=300, d=128, nq=32, dtype="fp16"),
        # 64 queries sharing each pass over a corpus (offline evaluation, batch serving).
        dict(name="batched_64q", kind="batched", nQ=64, B=100_000, Nd=180, d=128, nq=32, dtype="fp16"),
        # A product-quantised corpus, 16 codes of one byte a token.
        dict(name="pq_500k", kind="pq", B=500_000, Nd=128, M=16, K=256, dsub=8, nq=32, codes="u8"),
        # Best 100 of a million scores for each of 32 queries.
        dict(name="topk_32x1m", kind="topk", rows=32, n=1_000_000, k=100),
    ]


def _log(rng, lo, hi):
    """An integer of [lo, hi], even over its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.5)))))))


def draw(rng):
    kind = rng.choice(["rerank", "packed", "residual", "masked", "dense", "dense", "dense", "varlen", "batched", "batched",
                       "varlen_batched", "residual_batched", "pq", "pq", "pq_batched", "topk"])
    half = rng.choice(["fp16", "fp16", "bf16"])
    nq = rng.choice([32, 32, 32, rng.randint(8, 64)])
    if kind == "rerank":
        B = _log(rng, 64, 1024)
        return dict(kind=kind, B=B, Nd=rng.randint(32, 300), d=rng.choice([64, 96, 128, 128]), nq=nq, dtype=half,
                    k=min(B, rng.choice([10, 50, 100])))
    if kind == "packed":
        lo = rng.randint(8, 64)
        return dict(kind=kind, B=_log(rng, 128, 8192), lo=lo, hi=rng.randint(lo + 20, 300), d=rng.choice([64, 96, 128, 128]),
                    nq=nq, dtype="fp16")
    if kind == "residual":
        docs = _log(rng, 10_000, 200_000)
        lo = rng.randint(8, 64)
        return dict(kind=kind, B=_log(rng, 128, 8192), docs=docs, lo=lo, hi=rng.randint(lo + 20, 300),
                    d=rng.choice([64, 96, 128, 128]), nq=nq, nbits=rng.choice([1, 2, 2, 4]),
                    ncent=1 << rng.randint(13, 17))
    if kind == "masked":
        nd = rng.choice([180, rng.randint(64, 300)])
        return dict(kind=kind, B=_log(rng, 256, 50_000), Nd=nd, lo=rng.randint(8, 32), hi=nd,
                    d=rng.choice([64, 96, 128, 128]), nq=nq, dtype=half)
    if kind == "dense":
        d = rng.choice([48, 64, 96, 128, 128, 128, 200, 256, 384, 512, 768])
        dtype = rng.choice(["fp16", "fp16", "bf16", "fp32"])
        nd = rng.randint(16, 300)
        most = max(1000, min(400_000, int(9e9 / (nd * d * SIZE[dtype]))))
        return dict(kind=kind, B=_log(rng, 1000, most), Nd=nd, d=d, nq=nq, dtype=dtype)
    if kind == "varlen":
        lo = rng.randint(8, 64)
        return dict(kind=kind, B=_log(rng, 1000, 200_000), lo=lo, hi=rng.randint(lo + 20, 300), d=rng.choice([64, 96, 128, 128]),
                    nq=nq, dtype=half)
    if kind == "batched":
        return dict(kind=kind, nQ=rng.randint(2, 64), B=_log(rng, 1000, 100_000), Nd=rng.randint(32, 180),
                    d=rng.choice([64, 96, 128, 128]), nq=32, dtype=half)
    if kind == "varlen_batched":
        lo = rng.randint(8, 64)
        return dict(kind=kind, nQ=rng.randint(2, 32), B=_log(rng, 1000, 100_000), lo=lo, hi=rng.randint(lo + 20, 300),
                    d=rng.choice([64, 96, 128, 128]), nq=32, dtype=half)
    if kind == "residual_batched":
        lo = rng.randint(8, 64)
        docs = _log(rng, 1000, 100_000)
        return dict(kind=kind, nQ=rng.randint(2, 32), B=docs, docs=docs, lo=lo, hi=rng.randint(lo + 20, 200), d=128, nq=32,
                    nbits=rng.choice([1, 2, 2, 4]), ncent=1 << rng.randint(13, 17))
    if kind in ("pq", "pq_batched"):
        c = dict(kind=kind, B=_log(rng, 1000, 500_000 if kind == "pq" else 200_000), Nd=rng.randint(32, 180),
                 **rng.choice([dict(M=16, K=256, dsub=8), dict(M=16, K=256, dsub=8), dict(M=32, K=256, dsub=4),
                               dict(M=8, K=256, dsub=16), dict(M=16, K=64, dsub=4)]), nq=nq, codes="u8")
        if kind == "pq_batched":
            return dict(c, nQ=rng.randint(2, 32), nq=32)
        wide = rng.choice(["u8", "u8", "i16", "i32"])
        return c if wide == "u8" else dict(c, codes=wide, B=min(c["B"], 100_000))
    return dict(kind="topk", rows=_log(rng, 1, 64), n=_log(rng, 1000, 1_000_000), k=rng.choice([10, 100, rng.randint(1, 1000)]))


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _tokens(shape, dtype, gen, raw=False):
    """Token embeddings of ``shape`` (last dimension d), made CHUNK tokens at a time."""
    d = shape[-1]
    n = math.prod(shape[:-1])
    out = torch.empty(n, d, dtype=dtype, device="cuda")
    for i in range(0, n, CHUNK):
        x = torch.randn(min(CHUNK, n - i), d, generator=gen, device="cuda")
        out[i:i + CHUNK] = x if raw else x / x.norm(dim=-1, keepdim=True)
    return out.view(shape)


def _lengths(n, lo, hi, gen):
    return torch.randint(lo, hi + 1, (n,), generator=gen, device="cuda")


def _offsets(lengths):
    return torch.cat([lengths.new_zeros(1), lengths.cumsum(0)])


def prepare(case, seed):
    gen = _gen(seed)
    kind = case["kind"]
    s = {"case": case}
    if kind == "topk":
        s["scores"] = torch.randn(case["rows"], case["n"], generator=gen, device="cuda") * 1.3 + 12.0
        return s
    dtype = DTYPES[case.get("dtype", "fp16")]
    d = case["M"] * case["dsub"] if "M" in case else case["d"]
    qshape = (case["nQ"], case["nq"], d) if "nQ" in case else (case["nq"], d)
    s["Q"] = _tokens(qshape, dtype, gen, case.get("raw", False))
    if kind in ("rerank", "dense", "batched", "masked"):
        s["D"] = _tokens((case["B"], case["Nd"], d), dtype, gen, case.get("raw", False))
    if kind == "masked":
        lengths = _lengths(case["B"], case["lo"], case["hi"], gen)
        s["mask"] = torch.arange(case["Nd"], device="cuda") < lengths[:, None]
        s["D"].masked_fill_(~s["mask"][:, :, None], 0)  # padded with zero vectors
    elif kind in ("packed", "varlen", "varlen_batched"):
        s["lengths"] = _lengths(case["B"], case["lo"], case["hi"], gen)
        s["offsets"] = _offsets(s["lengths"])
        s["D"] = _tokens((int(s["offsets"][-1]), d), dtype, gen)
    elif kind in ("residual", "residual_batched"):
        s["offsets"] = _offsets(_lengths(case["docs"], case["lo"], case["hi"], gen))
        T = int(s["offsets"][-1])
        nb = case["nbits"]
        s["codes"] = torch.randint(0, case["ncent"], (T,), generator=gen, device="cuda", dtype=torch.int32)
        s["residuals"] = torch.randint(0, 256, (T, d * nb // 8), generator=gen, device="cuda", dtype=torch.uint8)
        s["centroids"] = _tokens((case["ncent"], d), torch.float16, gen)
        s["weights"] = (torch.linspace(-1.5, 1.5, 1 << nb, device="cuda") * 0.4 / math.sqrt(d)).half()
        s["pids"] = None
        if kind == "residual":  # PLAID's candidates: distinct ids of documents all over the index
            s["pids"] = torch.randperm(case["docs"], generator=gen, device="cuda")[:case["B"]].contiguous()
    elif kind in ("pq", "pq_batched"):
        book = torch.randn(case["M"], case["K"], case["dsub"], generator=gen, device="cuda").half()
        s["pq"] = tms.TileMaxSimPQ(book)
        s["codes"] = torch.randint(0, case["K"], (case["B"], case["Nd"], case["M"]), generator=gen, device="cuda",
                                   dtype=CODES[case["codes"]])
    return s


def run(s):
    kind = s["case"]["kind"]
    if kind == "rerank":
        return tms.maxsim_topk(s["Q"], s["D"], s["case"]["k"])
    if kind == "packed":
        return tms.flashmaxsim_score_packed(s["Q"], s["D"], s["lengths"])
    if kind == "residual":
        return tms.flashmaxsim_score_residual(s["Q"], s["codes"], s["residuals"], s["centroids"], s["weights"],
                                              s["case"]["nbits"], s["offsets"], s["pids"])
    if kind == "masked":
        return tms.maxsim_score(s["Q"], s["D"], s["mask"])
    if kind == "dense":
        return tms.flash_maxsim_v2_multiquery(s["Q"], s["D"])
    if kind == "varlen":
        return tms.flash_maxsim_multi_doc(s["Q"], s["D"], s["offsets"])
    if kind == "batched":
        return tms.flash_maxsim_batched_queries(s["Q"], s["D"])
    if kind == "varlen_batched":
        return tms.flash_maxsim_multi_doc_batched(s["Q"], s["D"], s["offsets"])
    if kind == "residual_batched":
        return tms.flashmaxsim_score_residual_batched(s["Q"], s["codes"], s["residuals"], s["centroids"], s["weights"],
                                                      s["case"]["nbits"], s["offsets"])
    if kind == "pq":
        return s["pq"].score_batch(s["Q"], s["codes"])
    if kind == "pq_batched":
        return s["pq"].score_batch_queries(s["Q"], s["codes"])
    return tms.topk(s["scores"], s["case"]["k"])


def work(case):
    """Bytes read and written once, and the multiply-adds of every scored token."""
    kind = case["kind"]
    if kind == "topk":
        return {"bytes": case["rows"] * (4 * case["n"] + 12 * case["k"]), "flops": 0}
    d = case["M"] * case["dsub"] if "M" in case else case["d"]
    size = SIZE[case.get("dtype", "fp16")]
    nQ, B = case.get("nQ", 1), case["B"]
    mean = (case["lo"] + case["hi"]) / 2 if "lo" in case else case["Nd"]
    tokens = B * mean
    total = nQ * case["nq"] * d * size + nQ * B * 4
    if kind in ("residual", "residual_batched"):  # ids, packed buckets, and the centroid rows they name
        rows = case["ncent"] * (1 - math.exp(-tokens / case["ncent"]))
        total += tokens * (4 + d * case["nbits"] / 8) + rows * d * 2 + B * 8
    elif kind in ("pq", "pq_batched"):
        total += tokens * case["M"] * {"u8": 1, "i16": 2, "i32": 4}[case["codes"]] + d * case["K"] * 2
    else:
        total += tokens * d * size
        if kind == "masked":
            total += B * case["Nd"]
        elif kind != "dense" and "lo" in case:
            total += 8 * B
    return {"bytes": total, "flops": 2.0 * nQ * case["nq"] * tokens * d}


def tolerance(case):
    """About four times what another order of the 32-bit sums gives, or, where the format
    asks for more roundings, another correct place for them: the bf16 terms of fp32
    documents, and the fp16 norm and tokens of a residual index."""
    kind = case["kind"]
    if kind == "topk":
        return "exact"
    if kind == "residual" or kind == "residual_batched":
        return {"rel": 2e-5, "max": 3e-4}
    if case.get("dtype") == "fp32":
        return {"rel": 2e-6, "max": 2e-5}
    return {"rel": 5e-7, "max": 5e-6, "differ": 0.01}


def _maxsim64(Q, rows, offsets):
    """sum over query tokens of the max over each document's tokens, in 64 bits: ``Q``
    (n, d), ``rows(i, j)`` the tokens [i, j) in 64 bits, documents at ``offsets``."""
    best = torch.full((offsets.numel() - 1, Q.shape[0]), -math.inf, dtype=torch.float64, device="cuda")
    QT = Q.double().t().contiguous()
    T = int(offsets[-1])
    step = max(1024, min(CHUNK, (1 << 28) // Q.shape[0]))
    for i in range(0, T, step):
        j = min(T, i + step)
        dots = rows(i, j) @ QT
        a = int(torch.searchsorted(offsets, torch.tensor(i, device="cuda"), right=True)) - 1
        b = int(torch.searchsorted(offsets, torch.tensor(j, device="cuda")))
        cut = offsets[a:b + 1].clamp(i, j) - i
        part = torch.segment_reduce(dots, "max", lengths=cut[1:] - cut[:-1], initial=-math.inf, unsafe=True)
        best[a:b] = torch.maximum(best[a:b], part)
    return best


def _residual64(s, i, j):
    """Tokens [i, j) of a residual index: fp16(centroid + weight) over its fp16 norm."""
    nb = s["case"]["nbits"]
    packed = s["residuals"][i:j].int()
    bits = (packed[:, :, None] >> torch.arange(7, -1, -1, device="cuda", dtype=torch.int32)) & 1
    bits = bits.view(j - i, -1, nb)
    bucket = (bits << torch.arange(nb, device="cuda", dtype=torch.int32)).sum(-1)  # least significant bit first
    v = (s["centroids"][s["codes"][i:j].long()].float() + s["weights"].float()[bucket]).half().double()
    return v / v.norm(dim=-1, keepdim=True).half().double()


def exact(case, seed):
    kind = case["kind"]
    s = prepare(case, seed)
    if kind == "topk":
        return torch.topk(s["scores"].double(), case["k"], dim=-1).values, None
    Q = s["Q"].reshape(-1, s["Q"].shape[-1])
    d = Q.shape[1]
    if kind in ("rerank", "dense", "batched", "masked"):
        flat = s["D"].view(-1, d)
        offsets = torch.arange(case["B"] + 1, device="cuda") * case["Nd"]
        if kind == "masked":
            flat = flat[s["mask"].view(-1)]
            offsets = _offsets(s["mask"].sum(1))
        best = _maxsim64(Q, lambda i, j: flat[i:j].double(), offsets)
    elif kind in ("packed", "varlen", "varlen_batched"):
        best = _maxsim64(Q, lambda i, j: s["D"][i:j].double(), s["offsets"])
        if kind == "packed":  # documents zero-padded to the longest one
            best = torch.where((s["lengths"] < s["lengths"].max())[:, None], best.clamp(min=0), best)
    elif kind in ("residual", "residual_batched"):
        lengths = s["offsets"][1:] - s["offsets"][:-1]
        starts = s["offsets"][:-1]
        if s["pids"] is not None:
            lengths, starts = lengths[s["pids"]], starts[s["pids"]]
        offsets = _offsets(lengths)
        if s["pids"] is not None:  # the candidates' rows, back to back
            at = torch.arange(int(offsets[-1]), device="cuda") + (starts - offsets[:-1]).repeat_interleave(lengths)
            s = dict(s, codes=s["codes"][at], residuals=s["residuals"][at])
        best = _maxsim64(Q, lambda i, j: _residual64(s, i, j), offsets)
        best = torch.where((lengths < lengths.max())[:, None], best.clamp(min=0), best)
    else:
        book = s["pq"].codebook.double()
        codes = s["codes"].view(-1, case["M"])
        m = torch.arange(case["M"], device="cuda")
        offsets = torch.arange(case["B"] + 1, device="cuda") * case["Nd"]
        best = _maxsim64(Q, lambda i, j: book[m, codes[i:j].long()].reshape(j - i, d), offsets)
    scores = best.view(best.shape[0], case.get("nQ", 1), case["nq"]).sum(-1).t().contiguous()
    if "nQ" in case:
        return scores
    if kind == "rerank":
        return torch.topk(scores[0], case["k"]).values, None
    return scores[0]
