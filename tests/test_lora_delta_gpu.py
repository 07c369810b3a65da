"""GPU tests of a worker's LoRA delta over a prompt chunk
(swl_lora_delta_bf16): the edges of its row and column tiles, K remainders,
every rank it takes, both layouts of A and of each B, and the modules that
route to it against the products they used.

Reference: the two products in float64 with the two bf16 roundings (shrink,
expand).  A shrink value may round to the neighbouring bf16 (2^-8 of it), so
the bound is the repository's 1e-2 of the largest output.
"""

import pytest
import torch

from tests._util import BF16, assert_close, randn

pytestmark = pytest.mark.gpu


def _want(x, fA, bs, rank, alpha):
    u = (x.double() @ fA.double()).to(BF16).double()
    return torch.cat([(alpha * (u[:, i * rank:(i + 1) * rank] @ b.double())) for i, b in enumerate(bs)], 1).to(BF16)


@pytest.mark.parametrize("m,k,rank,cols,kmajor,rr_major", [
    (5, 512, 16, [64], True, True), (16, 4096, 16, [4096, 1024, 1024], True, True), (17, 40, 8, [72, 8], True, True),
    (33, 1048, 24, [200, 64, 56, 8], True, True), (64, 4096, 64, [512, 256, 64], True, True),
    (65, 520, 40, [136, 320], True, True), (513, 4096, 32, [1536, 1536], True, True), (1, 4096, 32, [256, 64, 64], True, True),
    (6, 14336, 16, [4096], False, False), (31, 8, 8, [100], False, False), (130, 1000, 64, [333], False, False),
    (48, 544, 56, [37, 91], False, False), (300, 2048, 16, [65, 63, 9, 129], False, False),
    (70, 512, 16, [128, 264], True, False), (70, 512, 48, [128, 264], False, True),
    # 64-row expand workgroups: more than 64 KiB of LDS from 192 shrink columns on, just below
    (700, 512, 64, [4096, 1024, 1024], True, True), (641, 264, 48, [2048, 2048, 1032, 1024], True, True),
    (650, 256, 64, [2048, 2048, 1024, 1024], False, False), (641, 256, 56, [4096, 1024, 1024], True, True),
])
def test_lora_delta_matches_two_products(dev, m, k, rank, cols, kmajor, rr_major):
    from swarmlora_amd import ops
    n = len(cols)
    x, fA = randn((m, k), 1), randn((k, n * rank), 2, std=0.05)
    bs = [randn((rank, c), 3 + i, std=0.05) for i, c in enumerate(cols)]
    a = fA.to(dev) if kmajor else fA.t().contiguous().to(dev)
    blocks = [(b.to(dev) if rr_major else b.t().contiguous().to(dev), c, rr_major) for b, c in zip(bs, cols)]
    xd = x.to(dev)
    assert ops.lora_delta_fits(xd, a, kmajor, blocks, rank)
    # rows wider than the delta: what lies beside and below stays
    buf = torch.full((m + 2, sum(cols) + 24), 7.0, dtype=BF16, device=dev)
    got = ops.lora_delta(xd, a, kmajor, blocks, rank, 2.0, out=buf[:m, :sum(cols)])
    torch.cuda.synchronize()
    assert_close(got, _want(x, fA, bs, rank, 2.0), what="lora_delta")
    assert bool((buf[m:] == 7.0).all()) and bool((buf[:, sum(cols):] == 7.0).all())


def test_lora_delta_of_blocks_of_one_matrix_and_a_row_view(dev):
    """B as diagonal blocks of one fused_B, x as columns of a wider buffer."""
    from swarmlora_amd import ops
    wide, fA, fB = randn((40, 1024 + 64), 5), randn((1024, 48), 6, std=0.05), randn((48, 96 + 64 + 64), 7, std=0.05)
    x = wide[:, 64:]
    cols, blocks, c0 = [96, 64, 64], [], 0
    fBd = fB.to(dev)
    for i, c in enumerate(cols):
        blocks.append((fBd[16 * i:16 * i + 16, c0:c0 + c], c, True))
        c0 += c
    got = ops.lora_delta(wide.to(dev)[:, 64:], fA.to(dev), True, blocks, 16)
    torch.cuda.synchronize()
    bs = [fB[:16, :96], fB[16:32, 96:160], fB[32:, 160:]]
    assert_close(got, _want(x, fA, bs, 16, 1.0), what="lora_delta")


def test_lora_delta_refuses_what_it_cannot_take(dev):
    from swarmlora_amd import ops
    x, a = torch.zeros(8, 512, dtype=BF16, device=dev), torch.zeros(512, 16, dtype=BF16, device=dev)
    b = torch.zeros(16, 64, dtype=BF16, device=dev)
    assert ops.lora_delta_fits(x, a, True, [(b, 64, True)], 16)
    odd = torch.zeros(8 * 512 + 1, dtype=BF16, device=dev)[1:].view(8, 512)
    for xx, aa, bb, r in ((odd, a, b, 16), (x, a[:, :12], b, 12), (x[:, :500], a[:500], b, 16),
                          (x, torch.zeros(512, 72, dtype=BF16, device=dev), b, 72), (x, a, b[:, :60], 16)):
        assert not ops.lora_delta_fits(xx, aa, True, [(bb, bb.shape[1], True)], r)
        with pytest.raises(RuntimeError, match="swl_lora_delta_bf16"):
            ops.lora_delta(xx, aa, True, [(bb, bb.shape[1], True)], r)


@pytest.mark.parametrize("t,rank", [(16, 16), (100, 8), (40, 12), (7, 4), (3, 32)])
def test_worker_modules_route_by_rank(dev, t, rank):
    """FusedLoRA and SyncRemoteLoRALinear over a chunk, for ranks the two
    launches take and ranks they do not (the scalar products), against the
    reference's two products."""
    from swarmlora_amd.worker.model_builder import FastLoRAModule, FusedLoRA, SyncRemoteLoRALinear
    dims = [512, 128, 128]
    ab = [(randn((rank, 512), 10 + i, std=0.05), randn((d, rank), 20 + i, std=0.05)) for i, d in enumerate(dims)]
    x = randn((1, t, 512), 30)
    mods = [FastLoRAModule(a.to(dev), b.to(dev), 2.0) for a, b in ab]
    got = FusedLoRA(mods, dims, dev, BF16)(x.to(dev))
    one = SyncRemoteLoRALinear(3, 0, dims[0], mods[0]).delta(x.to(dev))
    torch.cuda.synchronize()
    for g, (a, b) in zip(got, ab):
        assert_close(g[0], _want(x[0], (a * 2).t(), [b.t()], rank, 1.0), what="fused")
    assert_close(one[0], _want(x[0], ab[0][0].t(), [ab[0][1].t()], rank, 2.0), what="remote")


@pytest.mark.parametrize("m,k,rank,cols,kmajor,rr_major", [
    (1, 4096, 16, [4096, 1024, 1024], True, True), (1, 4096, 16, [14336, 14336], True, True),
    (1, 14336, 16, [4096], False, False), (1, 4096, 64, [1000], False, False), (1, 8, 8, [8], True, True),
    (1, 24, 8, [1025], False, False), (1, 16384, 8, [1032, 24], True, True), (1, 16392, 32, [2056, 16], True, True),
    (1, 20000, 64, [1024], False, False), (2, 4096, 8, [1024, 8, 2048], True, True), (3, 4104, 32, [520, 520], True, True),
    (4, 14336, 64, [1023], False, False), (4, 8200, 16, [64, 1024, 16, 8], True, True), (4, 4096, 64, [136], True, False),
    (2, 1000, 16, [264], False, True),
])
def test_lora_rows_wide_matches_two_products(dev, m, k, rank, cols, kmajor, rr_major):
    """The one-launch delta of a few rows in the ranks and layouts of its
    wide kernel: 1024-column workgroups, K staged in pieces, every rank."""
    from swarmlora_amd import ops
    n = len(cols)
    x, fA = randn((m, k), 1), randn((k, n * rank), 2, std=0.05)
    bs = [randn((rank, c), 3 + i, std=0.05) for i, c in enumerate(cols)]
    a = fA.to(dev) if kmajor else fA.t().contiguous().to(dev)
    blocks = [(b.to(dev) if rr_major else b.t().contiguous().to(dev), c, rr_major) for b, c in zip(bs, cols)]
    buf = torch.full((m + 1, sum(cols) + 24), 7.0, dtype=BF16, device=dev)
    ops.lora_rows(x.to(dev), a, kmajor, blocks, rank, 2.0, out=buf[:m, :sum(cols)])
    torch.cuda.synchronize()
    assert_close(buf[:m, :sum(cols)], _want(x, fA, bs, rank, 2.0), what="lora_rows")
    assert bool((buf[m:] == 7.0).all()) and bool((buf[:, sum(cols):] == 7.0).all())
