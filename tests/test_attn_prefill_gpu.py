"""GPU tests of attention over several new tokens per sequence (prompt
chunks): block and tile edges of the MFMA kernel, pages of any size, missing
pages, and infinite or NaN values that causality hides from some rows.

The reference is the definition in float64 on the CPU.  Bound per element:
the result's rounding to bf16 (2^-9 of its size, itself at most the largest
|V|), the fp32 accumulation over the context and the probabilities' 2^-17:
4e-3 of the largest |V| covers them.
"""

import math

import pytest
import torch

from tests._util import BF16, randn

pytestmark = pytest.mark.gpu


def _case(dev, nseq, L, hq, hkv, ctx, page, missing=()):
    """Random q/k/v over shuffled pages (no RoPE); `missing`: (sequence, page
    index) entries of the block table set to -1."""
    per = (max(ctx) + L + page - 1) // page + 1
    nb = nseq * per
    c = {"q": randn((nseq, L, hq, 128), 1), "k": randn((nseq, L, hkv, 128), 2), "v": randn((nseq, L, hkv, 128), 3),
         "kc": randn((nb, page, hkv, 128), 4), "vc": randn((nb, page, hkv, 128), 5),
         "bt": torch.randperm(nb, generator=torch.Generator().manual_seed(6)).reshape(nseq, per).to(torch.int32),
         "len": torch.tensor(ctx, dtype=torch.int32)}
    for s, j in missing:
        c["bt"][s, j] = -1
    return c


def _run(dev, c, scale):
    from swarmlora_amd import ops
    d = {k: v.to(dev) for k, v in c.items()}
    out = ops.paged_attention(d["q"], d["k"], d["v"], d["kc"], d["vc"], d["bt"], d["len"], None, None, scale, rope=False)
    torch.cuda.synchronize()
    return out.cpu().double(), d


def _want(c, scale):
    nseq, L, hq, _ = c["q"].shape
    hkv, page = c["k"].shape[2], c["kc"].shape[1]
    kc, vc = c["kc"].double(), c["vc"].double()
    out = torch.zeros(nseq, L, hq * 128, dtype=torch.float64)
    for s in range(nseq):
        n = int(c["len"][s])
        for i in range(L):
            b = int(c["bt"][s, (n + i) // page])
            if b >= 0:
                kc[b, (n + i) % page], vc[b, (n + i) % page] = c["k"][s, i].double(), c["v"][s, i].double()
        keys = torch.arange(n + L)
        blocks = c["bt"][s][keys // page].long()
        ks, vs = kc[blocks.clamp_min(0), keys % page], vc[blocks.clamp_min(0), keys % page]
        for i in range(L):
            see = (blocks >= 0) & (keys < n + i + 1)
            if not bool(see.any()):
                continue
            for h in range(hq):
                kv = h * hkv // hq
                p = ((ks[see][:, kv] @ c["q"][s, i, h].double()) * scale).softmax(0)
                out[s, i, h * 128:(h + 1) * 128] = p @ vs[see][:, kv]
    return out


def _check(got, want, vmax):
    bad = ~((got - want).abs() <= 4e-3 * vmax)
    assert not bool(bad.any()), f"max error {float((got - want).abs().max()):.3e}"


# rows per (sequence, kv head) = L * hq / hkv around 32 and 64 (row blocks);
# contexts around 64, 128 and 256 keys (tiles); more blocks than CUs (the
# four-wave form) in the last two
@pytest.mark.parametrize("nseq,L,hq,hkv,ctx,page", [
    (1, 2, 4, 4, [0], 16), (1, 31, 4, 4, [33], 16), (1, 33, 4, 4, [0], 16), (2, 8, 16, 4, [224, 3], 16),
    (3, 9, 32, 4, [255, 0, 47], 16), (1, 16, 32, 8, [1000], 16), (2, 65, 8, 2, [63, 129], 32),
    (1, 130, 16, 8, [127], 8), (1, 40, 8, 4, [300], 7), (1, 300, 32, 8, [212], 16),
    (3, 130, 32, 16, [11, 90, 64], 48), (2, 200, 64, 32, [5, 130], 16),
])
def test_prefill_attention_edges(dev, nseq, L, hq, hkv, ctx, page):
    c = _case(dev, nseq, L, hq, hkv, ctx, page)
    got, _ = _run(dev, c, 128 ** -0.5)
    _check(got, _want(c, 128 ** -0.5), 6.0)


@pytest.mark.parametrize("scale", [-0.09, 0.5])
def test_prefill_attention_missing_pages(dev, scale):
    """Block table entries of -1 hide their keys (a whole first page, one in
    the middle, a new token's own page), also with a negative scale."""
    c = _case(dev, 2, 20, 8, 2, [40, 0], 16, missing=((0, 0), (0, 3), (1, 0)))
    got, d = _run(dev, c, scale)
    _check(got, _want(c, scale), 6.0)
    assert bool((got[1, :16] == 0).all())  # no key at all


@pytest.mark.parametrize("value", [math.inf, -math.inf, math.nan])
@pytest.mark.parametrize("L,ctx,at", [(40, 10, 27), (100, 200, 217), (100, 200, 3), (70, 300, 299), (33, 1000, 500)])
def test_prefill_attention_keeps_nonfinite_values_causal(dev, value, L, ctx, at):
    """A non-finite value of key `at` (a new token, or one of the cached context,
    which every row sees) gives the rows that see it what the definition gives
    (inf, -inf or NaN) and reaches no other; with an infinity of the other sign
    beside it, NaN.  Non-finite cache contents past the context reach none."""
    c = _case(dev, 1, L, 8, 2, [ctx], 16)
    clean, _ = _run(dev, {k: v.clone() for k, v in c.items()}, 128 ** -0.5)

    def put(key, x, dim):
        if key < ctx:
            c["vc"][int(c["bt"][0, key // 16]), key % 16, 1, dim] = x
        else:
            c["v"][0, key - ctx, 1, dim] = x
    put(at, value, 5)
    put(at, value, 77)
    put(min(at + 2, ctx + L - 1), -value, 77)
    c["vc"][int(c["bt"][0, -1])] = math.nan   # a page past every context
    c["kc"][int(c["bt"][0, -1])] = math.nan
    got, _ = _run(dev, c, 128 ** -0.5)
    seen = torch.arange(L) + ctx >= at
    both = torch.arange(L) + ctx >= at + 2
    got, clean = got.view(L, 8, 128), clean.view(L, 8, 128)
    hit = torch.zeros(L, 8, 128, dtype=torch.bool)
    hit[:, 4:, 5], hit[:, 4:, 77] = seen[:, None], seen[:, None]  # kv head 1 serves query heads 4..7
    want = torch.full_like(got, value)
    want[both, :, 77] = math.nan
    assert bool(((got == want) | (got.isnan() & want.isnan()))[hit].all())
    # the rest as without it; rows computed key by key round differently
    assert float((got[~hit] - clean[~hit]).abs().max()) <= 4e-3 * 6.0


@pytest.mark.parametrize("at", [280, 301])
def test_prefill_attention_values_near_the_largest_number(dev, at):
    """V of 3e38 at a key whose score is 5 above the others', which come first:
    the weighted sum stays finite (the weights are at most 1)."""
    L, ctx, big = 20, 300, 3e38
    c = _case(dev, 1, L, 8, 2, [ctx], 16)
    c["q"].fill_(1.0)
    c["k"].zero_(), c["kc"].zero_()
    if at < ctx:
        c["kc"][int(c["bt"][0, at // 16]), at % 16] = 1.0
        c["vc"][int(c["bt"][0, at // 16]), at % 16] = big
    else:
        c["k"][0, at - ctx], c["v"][0, at - ctx] = 1.0, big
    got, _ = _run(dev, c, 5.0 / 128)
    _check(got, _want(c, 5.0 / 128), big)


def test_prefill_attention_nan_scores_cost_no_recomputation(dev):
    """A NaN in q, or in a key, makes 0 of the rows it reaches; the others keep
    their bits (the block is not computed again key by key)."""
    c = _case(dev, 1, 50, 8, 2, [300], 16)
    clean, _ = _run(dev, {k: v.clone() for k, v in c.items()}, 128 ** -0.5)
    clean = clean.view(50, 8, 128)
    c["q"][0, 7, 2] = math.nan
    c["k"][0, 20, 1] = math.nan    # kv head 1: query heads 4..7 of tokens 20..
    got, _ = _run(dev, c, 128 ** -0.5)
    got = got.view(50, 8, 128)
    hit = torch.zeros(50, 8, dtype=torch.bool)
    hit[7, 2], hit[20:, 4:] = True, True
    assert bool((got[hit] == 0).all())
    assert torch.equal(got[~hit], clean[~hit])


def test_prefill_attention_under_capture_without_a_first_call(dev):
    """The kernel takes no scratch: a graph can capture the first call ever
    made with a shape, and replays give the eager result each time."""
    from swarmlora_amd import ops
    c = {k: v.to(dev) for k, v in _case(dev, 1, 24, 8, 2, [100], 16).items()}
    out = torch.zeros(1, 24, 1024, dtype=BF16, device=dev)
    args = (c["q"], c["k"], c["v"], c["kc"], c["vc"], c["bt"], c["len"], None, None, 0.1)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        ops.paged_attention(*args, rope=False, out=out)
    for _ in range(3):
        out.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, ops.paged_attention(*args, rope=False))
        torch.cuda.synchronize()
