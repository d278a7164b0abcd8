"""GPU tests of top-k by group maxima (``topk_group_max_kernel``, ``topk_group_last_kernel``).

Rows past one 4,096-score chunk at 8 <= k <= 512 are selected by the maxima of groups of 32
to 256 scores and of spans of 1,024. Row lengths sit on both sides of a span, of the rows
whose groups are selected without spans, and of each span count the selection is built for;
k on both sides of each group size and of the sorting and key limits; rows hold ties, sorted
scores (every winner in one span), NaN of both signs, infinities and zeros of both signs, and
start at every alignment. Values must be the input's bits, indices exact: values descending,
NaN first, equal values by ascending index.
"""
import pytest

pytestmark = pytest.mark.gpu

KS = [8, 9, 16, 17, 32, 33, 64, 65, 66, 67, 100, 127, 128, 129, 200, 256, 257, 511, 512, 513]


def _expected(scores, k):
    """Indices by the order's definition, from a 64-bit integer key per score."""
    import torch
    n = scores.shape[-1]
    b = scores.view(torch.int32).to(torch.int64) & 0xffffffff
    order = torch.where(b >= 1 << 31, (1 << 32) - b, b + (1 << 31)) & 0xffffffff
    order = torch.where(torch.isnan(scores), torch.full_like(order, 0xffffffff), order)
    key = (order << 25) + ((1 << 25) - 1 - torch.arange(n, device=scores.device))
    return (1 << 25) - 1 - (torch.sort(key, dim=-1, descending=True).values[:, :k] & ((1 << 25) - 1))


def _fill(kind, rows, n, seed):
    import torch
    g = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.randn(rows, n, generator=g, device="cuda")
    if kind == "ties":
        x = torch.randint(0, 5, (rows, n), generator=g, device="cuda").float() - 2.0
    elif kind == "equal":
        x = torch.full((rows, n), -3.25, device="cuda")
    elif kind == "rising":
        x = torch.sort(x, dim=-1).values
    elif kind == "falling":
        x = torch.sort(x, dim=-1, descending=True).values
    elif kind == "special":
        at = torch.randint(0, n, (rows, 300), generator=g, device="cuda")
        val = torch.tensor([0.0, -0.0, float("inf"), float("-inf"), float("nan"), 1e-42, -1e-42], device="cuda")
        x.scatter_(1, at, val[torch.arange(300, device="cuda") % 7].expand(rows, 300))
        neg = torch.full((rows, 1), -4194303, dtype=torch.int32, device="cuda").view(torch.float32)  # a negative NaN
        x.scatter_(1, at[:, 5:6], neg)
    elif kind == "lowest":
        x = torch.full((rows, n), float("-inf"), device="cuda")
        x[:, n // 3: n // 3 + 40] = -1.0
    return x


def _check(x, ks):
    import torch
    import tilemaxsim_amd as tms
    n = x.shape[-1]
    want = _expected(x, min(n, max(ks)))
    for k in ks:
        v, i = tms.topk(x, k)
        assert torch.equal(i, want[:, :k]), f"k={k} n={n}"
        assert torch.equal(v.view(torch.int32), torch.gather(x, 1, want[:, :k]).view(torch.int32)), f"k={k} n={n}"


@pytest.mark.parametrize("kind", ["gauss", "ties", "equal", "rising", "falling", "special", "lowest"])
@pytest.mark.parametrize("rows,n", [(1, 4097), (3, 5119), (2, 5121), (5, 16_458), (2, 65_537), (3, 131_072), (2, 131_073),
                                    (33, 70_001), (2, 300_003)])
def test_rows(cuda, rows, n, kind):
    _check(_fill(kind, rows, n, n + rows), KS)


@pytest.mark.parametrize("n", [1024 * 1024, 1024 * 1024 + 1, 4096 * 1024 - 3, 4096 * 1024 + 1, 16384 * 1024,
                               16384 * 1024 + 1])
def test_long_rows(cuda, n):
    _check(_fill("gauss", 1, n, n), [8, 64, 100, 128, 129, 512])
    _check(_fill("rising", 1, n, n), [100, 300])


@pytest.mark.parametrize("n,k,groups,kept", [
    (40_000, 100, 100, c) for c in (100, 767, 768, 769, 3000)] + [
    (100_000, 300, 300, c) for c in (1023, 1024, 1025, 5000)] + [
    # by spans: the groups that reach the bound in one load of the selection, in two, and in too many
    (1_000_000, 100, 100, c) for c in (700, 2000)] + [
    (1_000_000, 100, 200, c) for c in (700, 5000)] + [(1_000_000, 100, 600, 15_000), (1_000_000, 400, 1200, 20_000)])
def test_scores_that_reach_the_bound(cuda, n, k, groups, kept):
    """``kept`` scores reach the k-th largest maximum, in ``groups`` groups of 32 (as many a
    span in the k best spans, where spans come first): on both sides of the count that is
    ordered by rank, and of what the last selection holds."""
    import torch
    import rules
    assert rules.lib().topk_group_lanes(2, n, k) == 3
    g = torch.Generator(device="cuda").manual_seed(n + kept)
    x = torch.randn(2, n, generator=g, device="cuda")
    spans = n > 100_000
    for row in range(2):
        if spans:  # groups // k of each of k spans
            span = torch.randperm(n // 1024, generator=g, device="cuda")[:k]
            first = (span[:, None] * 1024 + 32 * torch.arange(groups // k, device="cuda")).reshape(-1)
        else:
            first = 32 * torch.randperm(n // 32, generator=g, device="cuda")[:groups]
        first = first.cpu()
        # one score of the first group is the bound, and in its span the largest; the others go over the rest
        lead = 1 if not spans else groups // k
        rest = (first[lead:, None] + torch.arange(32)).reshape(-1, 32)
        order = torch.cat([rest[:, 0], rest[:, 1:].reshape(-1)[torch.randperm(rest.numel() - len(rest))]])
        at = order[:kept - lead].cuda()
        x[row, at] = 200.0 + torch.rand(len(at), generator=g, device="cuda")
        x[row, first[:lead].cuda()] = 100.0
    reach = torch.sort(x, dim=1, descending=True).values
    assert bool((reach[:, kept - 1] == 100.0).all()) and bool((reach[:, kept] < 50.0).all())
    _check(x, [k])


def test_alignment_and_rows(cuda):
    """Rows that start at every offset of 16 bytes (odd row lengths), and many rows."""
    import torch
    flat = _fill("gauss", 1, 700 * 4099 + 3, 5)[0]
    for shift in range(4):
        _check(flat[shift:shift + 700 * 4099].view(700, 4099), [10, 100])
    assert flat.data_ptr() % 16 == 0 and torch.isfinite(flat).all()


def test_graph_and_streams(cuda):
    import torch
    import tilemaxsim_amd as tms
    x = _fill("gauss", 4, 200_000, 9)
    for _ in range(2):
        tms.topk(x, 100)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        v, i = tms.topk(x, 100)
    for seed in (1, 2, 3):
        x.copy_(_fill("gauss", 4, 200_000, seed))
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(i, _expected(x, 100))
    other = torch.cuda.Stream()
    other.wait_stream(torch.cuda.current_stream())
    y = _fill("ties", 4, 200_000, 11)
    other.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(other):
        _, j = tms.topk(y, 100)
    _, i = tms.topk(x, 100)
    torch.cuda.synchronize()
    assert torch.equal(i, _expected(x, 100)) and torch.equal(j, _expected(y, 100))
