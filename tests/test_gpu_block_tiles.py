"""The tiled block-granular attention (blocks of 32 keys and more) at the edges of
its tiles: query vectors that fill no tile, a last block of few rows, lists longer
than one 64-entry window, repeated and future blocks, rows with nothing to attend."""

import numpy as np
import pytest
import torch

from tests.helpers import f32, randn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d,g,n,bs,nkb,i64", [
    (128, 1, 97, 32, 2, True),      # one partly filled tile, a last block of one row
    (128, 3, 200, 32, 5, False),    # 96 query vectors: the second tile half used
    (64, 7, 385, 64, 7, True),      # rows split over waves mid-group
    (128, 8, 513, 256, 3, False),   # 2048 query vectors a block, a last block of one row
    (64, 4, 2500, 32, 79, True),    # two list windows
    (128, 2, 130, 128, 1, False)])  # a list without the rows' own block
def test_block_tiles_vs_oracle(dev, orc, d, g, n, bs, nkb, i64):
    from ssa_amd import kernels

    B, h_kv = 1, 2
    q = randn((B, n, h_kv * g, d), 91, torch.bfloat16)
    k = randn((B, n, h_kv, d), 92, torch.bfloat16)
    v = randn((B, n, h_kv, d), 93, torch.bfloat16)
    nb = (n + bs - 1) // bs
    gen = torch.Generator().manual_seed(94)
    blocks = torch.stack([torch.randperm(nb, generator=gen)[:nkb] for _ in range(B * nb * h_kv)])
    blocks = blocks.view(B, nb, h_kv, -1)
    if nkb == 1:
        blocks[:] = nb - 1           # the first block's rows have no key at all: zeros
    elif nkb > 2:
        blocks[..., 0] = blocks[..., 1]  # a block listed twice counts twice
    blocks = blocks if i64 else blocks.to(torch.int32)
    out = torch.empty(B, n, h_kv * g, d, device=dev, dtype=torch.float32)
    flag = torch.zeros(1, dtype=torch.int32, device=dev)
    kernels.block_sparse_attention(q.to(dev), k.to(dev), v.to(dev), blocks.to(dev), bs, out=out, error_flag=flag)
    assert int(flag.item()) == 0
    ref = orc.block_sparse_attention64(f32(q[0]), f32(k[0]), f32(v[0]), blocks[0].numpy(), bs)
    np.testing.assert_allclose(out[0].cpu().numpy(), ref, rtol=1e-3, atol=1e-3)
    bf = kernels.block_sparse_attention(q.to(dev), k.to(dev), v.to(dev), blocks.to(dev), bs)
    assert torch.equal(bf, out.to(torch.bfloat16)), "bf16 output must be the fp32 output rounded"


@pytest.mark.parametrize("d", [64, 128])
def test_block_tiles_non_finite_value_stays_in_its_past(dev, d):
    """A key that is still to come for a row of its own block must not reach that row."""
    from ssa_amd import kernels

    n, g, bs, at = 96, 4, 32, 45
    q, k, v = (randn((1, n, h, d), 95 + h, torch.bfloat16) for h in (g, 1, 2))
    v = v[:, :, :1].contiguous()
    blocks = torch.arange(3).expand(3, 3).contiguous().view(1, 3, 1, 3)
    good = kernels.block_sparse_attention(q.to(dev), k.to(dev), v.to(dev), blocks.to(dev), bs)
    v[0, at, 0, 5] = float("inf")
    got = kernels.block_sparse_attention(q.to(dev), k.to(dev), v.to(dev), blocks.to(dev), bs)
    assert torch.equal(got[0, :32], good[0, :32])
    # the rows before `at` in its block: key by key instead of in the matrix cores
    torch.testing.assert_close(got[0, :at].float(), good[0, :at].float(), rtol=2 ** -7, atol=2 ** -9)
    assert not got[0, at:, :, 5].isfinite().any()
    rest = torch.arange(d) != 5
    torch.testing.assert_close(got[0, at:][..., rest].float(), good[0, at:][..., rest].float(), rtol=2 ** -7, atol=2 ** -9)


def _compare(dev, orc, h_kv, d, g, n, bs, nkb):
    from ssa_amd import kernels

    q = randn((1, n, h_kv * g, d), 91, torch.bfloat16)
    k, v = randn((1, n, h_kv, d), 92, torch.bfloat16), randn((1, n, h_kv, d), 93, torch.bfloat16)
    nb = (n + bs - 1) // bs
    gen = torch.Generator().manual_seed(95)
    blocks = torch.stack([torch.randperm(nb, generator=gen)[:nkb] for _ in range(nb * h_kv)]).view(1, nb, h_kv, -1)
    if nkb == 1:
        blocks[:] = nb - 1               # as above
    elif nkb > 2:
        blocks[..., 0] = blocks[..., 1]
    out = torch.empty(1, n, h_kv * g, d, device=dev, dtype=torch.float32)
    kernels.block_sparse_attention(q.to(dev), k.to(dev), v.to(dev), blocks.to(dev), bs, out=out)
    ref = orc.block_sparse_attention64(f32(q[0]), f32(k[0]), f32(v[0]), blocks[0].numpy(), bs)
    # as test_block_tiles_vs_oracle
    np.testing.assert_allclose(out[0].cpu().numpy(), ref, rtol=1e-3, atol=1e-3)


@pytest.mark.parametrize("h_kv,d,g,n,bs,nkb", [
    (2, 128, 1, 97, 32, 3),      # one partly filled tile, a last block of one row
    (6, 128, 3, 200, 32, 5),     # 96 query vectors: the second tile half used
    (3, 64, 7, 385, 64, 7),      # rows split over waves mid-group
    (9, 128, 2, 130, 128, 1)])   # a list without the rows' own block
def test_block_tiles_of_calls_past_the_small_ones(dev, orc, h_kv, d, g, n, bs, nkb):
    """The tiles' edges again with enough rows or keys that the call does not go row by row."""
    _compare(dev, orc, h_kv, d, g, n, bs, nkb)


@pytest.mark.parametrize("h_kv,n,g,bs,nkb", [(4, 256, 8, 32, 3), (4, 257, 8, 32, 3), (4, 512, 8, 32, 2),
                                             (4, 513, 8, 32, 2), (4, 256, 2, 32, 2), (4, 257, 2, 32, 2)])
def test_block_rule_on_both_sides(dev, orc, h_kv, n, g, bs, nkb):
    _compare(dev, orc, h_kv, 64, g, n, bs, nkb)


@pytest.mark.parametrize("d", [64, 128])
def test_block_tiles_non_finite_value_of_one_head_among_many(dev, d):
    """As above, in a call whose rows share their tiles: the head with the value, and the others."""
    from ssa_amd import kernels

    n, g, h, bs, at, hot = 96, 4, 12, 32, 45, 7
    q, k, v = randn((1, n, h * g, d), 97, torch.bfloat16), randn((1, n, h, d), 98, torch.bfloat16), randn(
        (1, n, h, d), 99, torch.bfloat16)
    blocks = torch.arange(3).expand(3, h, 3).contiguous().view(1, 3, h, 3)
    good = kernels.block_sparse_attention(q.to(dev), k.to(dev), v.to(dev), blocks.to(dev), bs).view(n, h, g, d)
    v[0, at, hot, 5] = float("inf")
    got = kernels.block_sparse_attention(q.to(dev), k.to(dev), v.to(dev), blocks.to(dev), bs).view(n, h, g, d)
    others = torch.arange(h) != hot
    assert torch.equal(got[:, others], good[:, others]) and torch.equal(got[:32, hot], good[:32, hot])
    torch.testing.assert_close(got[:at, hot].float(), good[:at, hot].float(), rtol=2 ** -7, atol=2 ** -9)
    assert not got[at:, hot, :, 5].isfinite().any()
    rest = torch.arange(d) != 5
    torch.testing.assert_close(got[at:, hot][..., rest].float(), good[at:, hot][..., rest].float(),
                               rtol=2 ** -7, atol=2 ** -9)
