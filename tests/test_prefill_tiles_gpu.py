"""GPU tests of the prefill round just past the decode regime: 128 x 128 tiles
with and without K splits, their edges and remainders, LoRA carried by the
tiles, by the splits' sum and by the large tiles' epilogue, against float32
products of the same bf16 operands (bound: the result's bf16 rounding, 1e-2 of
the largest output as everywhere)."""

import pytest
import torch

from tests._util import BF16, assert_close, randn

pytestmark = pytest.mark.gpu


def _round(dev, rows, n, k, cols, ranks, bias=False, seed=0):
    """One round over `rows`, segment i with an adapter of ranks[i] (0: none)
    -> (outputs, expected)."""
    from swarmlora_amd import ops
    w = randn((n, k), seed, std=0.02).to(dev)
    b = randn((n,), seed + 1).to(dev) if bias else None
    xs = [randn((r, k), seed + 2 + i).to(dev) for i, r in enumerate(rows)]
    # sentinel rows after each slot's rows
    bufs = [torch.full((r + 1, n), 9.0, dtype=BF16, device=dev) for r in rows]
    table, ids, want = ops.LoraTable(dev), [], []
    for i, (x, r) in enumerate(zip(xs, ranks)):
        y = x.float() @ w.float().t() + (b.float() if bias else 0)
        if r:
            a = randn((r * len(cols), k), 50 + i, std=0.02).to(dev)
            bs = [randn((c, r), 80 + 7 * i + j, std=0.02).to(dev) for j, c in enumerate(cols)]
            u = x.float() @ a.float().t()
            y += 2.0 * torch.cat([u[:, j * r:(j + 1) * r] @ bs[j].float().t() for j in range(len(cols))], 1)
            ids.append(table.add(a, bs, r, 2.0))
        else:
            ids.append(-1)
        want.append(y)
    lora = any(ranks)
    ops.round_fused(xs, bufs, rows, w, b, seg_lora=ids if lora else None, table=table if lora else None,
                    blk_cols=cols if lora else None)
    torch.cuda.synchronize()
    for o in bufs:
        assert bool((o[-1] == 9.0).all())
    return [o[:-1] for o in bufs], want


@pytest.mark.parametrize("rows,n,k,cols,ranks,bias", [
    ([65], 128, 64, [128], [16], True),                              # one tile, one stage
    ([1, 64], 256, 2048, [128, 128], [8, 64], False),                # splits of 4 stages and more
    ([100, 3, 26], 1536, 4096, [1024, 256, 256], [16, 0, 32], True),  # a full row tile and one row
    ([128], 384, 8192, [384], [24], False),
    ([90, 40], 200, 4096, [72, 128], [16, 16], True),                # blocks not on tile bounds: delta in the sum
    ([70], 130, 2048, [130], [12], False),                           # ... rank not a multiple of 8, n % 4
    ([300, 1, 1, 1], 2048, 1024, [2048], [16, 8, 0, 64], False),
    ([66, 62], 1000, 4160, [1000], [0, 0], True),                    # no adapters: no splits
    ([1000, 60], 14336, 512, [7168, 7168], [16, 8], True),           # 1024 rows in large tiles, 36 behind
    ([700, 80, 1], 16400, 512, [8200, 8200], [16, 0, 12], True),     # ... and the delta in both epilogues
])
def test_short_prefill_rounds(dev, rows, n, k, cols, ranks, bias):
    got, want = _round(dev, rows, n, k, cols, ranks, bias)
    for g, w in zip(got, want):
        assert_close(g, w, what=f"{rows} {n} {k}")


@pytest.mark.parametrize("rows,k,cols", [([70], 512, [128, 256]), ([90, 60], 4096, [384, 640, 256])])
def test_short_prefill_delta_off_the_large_grid_in_fp32(dev, rows, k, cols):
    """Column blocks at multiples of 128 that are none of 256: the delta is
    fp32 up to the result's one rounding (half a bf16 step is at most 2^-8 of
    the value; 1e-5 of the largest for the fp32 sums over k)."""
    from swarmlora_amd import ops
    n, r = sum(cols), 8
    w = torch.zeros(n, k, dtype=BF16, device=dev)
    table, ids, xs, want = ops.LoraTable(dev), [], [], []
    for i, m in enumerate(rows):
        x, a = randn((m, k), i), randn((r * len(cols), k), 10 + i, std=0.05)
        bs = [randn((c, r), 20 + 5 * i + j) for j, c in enumerate(cols)]
        u = 1.7 * (x.double() @ a.double().t())
        want.append(torch.cat([u[:, j * r:(j + 1) * r] @ b.double().t() for j, b in enumerate(bs)], 1))
        ids.append(table.add(a.to(dev), [b.to(dev) for b in bs], r, 1.7))
        xs.append(x.to(dev))
    outs = [torch.zeros(m, n, dtype=BF16, device=dev) for m in rows]
    ops.round_fused(xs, outs, rows, w, None, seg_lora=ids, table=table, blk_cols=cols)
    torch.cuda.synchronize()
    for o, y in zip(outs, want):
        err = (o.double().cpu() - y).abs() - 2 ** -8 * y.abs()
        assert float(err.max()) <= 1e-5 * float(y.abs().max())


def test_short_prefill_round_captured_without_room_for_splits(dev):
    """A captured round that would need more scratch for its splits than the
    library holds runs unsplit (its shrink fits what an earlier call sized),
    and replays give the eager result."""
    import subprocess
    import sys
    code = """
import torch
from swarmlora_amd import ops
bf = torch.bfloat16
g = torch.Generator(device="cuda").manual_seed(3)
rn = lambda *s: torch.randn(*s, generator=g, device="cuda").to(bf)
def call(n, k, rows):
    t = ops.LoraTable("cuda")
    t.add(rn(16, k) * 0.05, [rn(n, 16) * 0.05], 16, 2.0)
    x, y, w = rn(rows, k), torch.zeros(rows, n, dtype=bf, device="cuda"), rn(n, k) * 0.05
    t.device_table()
    return y, lambda: ops.round_fused([x], [y], [rows], w, None, [0], t, [n])
_, small = call(256, 512, 70)   # sizes the scratch: its smallest step
small()
torch.cuda.synchronize()
y, big = call(4096, 4096, 128)  # its splits would need 16 MB
gr = torch.cuda.CUDAGraph()
with torch.cuda.graph(gr):
    big()
outs = []
for _ in range(3):
    y.zero_()
    gr.replay()
    torch.cuda.synchronize()
    outs.append(y.clone())
assert all(torch.equal(o, outs[0]) for o in outs)
big()
torch.cuda.synchronize()
d = (y.float() - outs[0].float()).abs().max() / y.float().abs().max()
assert float(d) < 1e-2, float(d)
print("captured ok")
"""
    p = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=100)
    assert p.returncode == 0 and "captured ok" in p.stdout, p.stdout + p.stderr


@pytest.mark.parametrize("rows,n,k,cols,same", [
    ([150, 300, 150], 2048, 4096, [1024, 1024], (0, 2)),       # 128 x 128 tiles, K split
    ([200] + [1] * 40, 4096, 8192, [4096], (1, 20, 40)),       # one-row slots of two row tiles
    ([130, 1, 200, 130], 2304, 4096, None, (0, 3)),            # no adapters: unsplit
    ([90, 40, 90], 456, 4096, [200, 256], (0, 2)),             # the delta in the splits' sum
    ([300] * 9, 6144, 4096, [4096, 1024, 1024], (0, 4, 8)),    # large tiles, then 128 x 128
    ([300] * 9, 6144, 4096, None, (0, 8)),
    ([700, 700, 700], 2048, 1024, [2048], (0, 1, 2)),
])
def test_a_prompt_gives_the_same_bits_wherever_it_is_in_the_round(dev, rows, n, k, cols, same):
    """Segments of the same rows and adapter: every row adds its products in
    the same order, in whichever tile, launch or split it lands."""
    from swarmlora_amd import ops
    w, b = randn((n, k), 0, std=0.02).to(dev), randn((n,), 1).to(dev)
    table, nb = ops.LoraTable(dev), len(cols or [])
    xs, ids = [], []
    for i, r in enumerate(rows):
        j = same[0] if i in same else i
        xs.append(xs[j].clone() if i in same[1:] else randn((r, k), 2 + i).to(dev))
        if cols:
            ids.append(ids[j] if i in same[1:] else table.add(
                randn((16 * nb, k), 100 + i, std=0.02).to(dev), [randn((c, 16), 200 + i, std=0.02).to(dev) for c in cols],
                16, 2.0))
    outs = [torch.zeros(r, n, dtype=BF16, device=dev) for r in rows]
    ops.round_fused(xs, outs, rows, w, b, seg_lora=ids or None, table=table if cols else None, blk_cols=cols)
    torch.cuda.synchronize()
    for i in same[1:]:
        assert torch.equal(outs[i], outs[same[0]]), f"segment {i}"


@pytest.mark.parametrize("m,n,k,bias", [
    (16, 18440, 128, True),    # ragged last tile of 128 columns, two stages
    (17, 14337, 64, False),    # odd row stride (below the line of 17 rows)
    (17, 15361, 64, False),    # ... past it, one stage (fewer than the slots)
    (32, 14336, 192, False),   # a full 32-row tile
    (33, 14340, 320, True),    # the 64-row tile, one valid row past 32
    (64, 28672, 256, False),   # tiles starting at each of four stages
    (1, 18432, 1024, False),
    (15, 18433, 4096, True),
    (15, 18304, 64, False),    # one tile short: the K-sliced kernel
])
def test_wide_decode_products(dev, m, n, k, bias):
    from swarmlora_amd import ops
    x, w = randn((m, k), 1).to(dev), torch.empty((n, k), dtype=BF16, device=dev).normal_(0, 0.02)
    b = randn((n,), 3).to(dev) if bias else None
    out = torch.full((m + 1, n), 9.0, dtype=BF16, device=dev)
    ops.gemm(x, w, b, out=out[:m])
    want = x.float() @ w.float().t() + (b.float() if bias else 0)
    torch.cuda.synchronize()
    assert bool((out[m] == 9.0).all())
    assert_close(out[:m], want, what=f"{m} {n} {k}")
