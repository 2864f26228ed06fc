"""Score order of bf16 rows on the matrix cores (select_sort_rows_kernel): equal to the
one-block-per-row kernel, whose order the oracle pins, bit for bit."""

import pytest
import torch

from tests.helpers import randn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d,g,k,i64", [
    (64, 1, 64, True),       # one chunk of 64 slots
    (64, 16, 200, False),    # four groups of heads
    (128, 3, 65, True),      # a second chunk of one slot, a head group part filled
    (128, 5, 700, True),     # 11 chunks, two groups
    (128, 8, 1024, False)])  # the longest list the registers hold
def test_sorted_rows_equal_the_exact_kernel(dev, d, g, k, i64):
    from ssa_amd import kernels

    n, h_kv, n_c, a, b = 1500, 2, 16, 8, 4
    q, kk = randn((1, n, h_kv * g, d), 71, torch.bfloat16), randn((1, n, h_kv, d), 72, torch.bfloat16)
    kk[0, 40:80] = kk[0, :40]            # equal scores: ties go to the lower index
    gen = torch.Generator().manual_seed(73)
    kc = torch.stack([torch.randperm(n_c, generator=gen)[:b] for _ in range(h_kv * n)]).view(1, h_kv, n, b).int()
    qc = torch.stack([torch.randperm(n_c, generator=gen)[:a] for _ in range(h_kv * n)]).view(1, h_kv, n, a).int()
    qd, kd, qcd, kcd = (t.to(dev) for t in (q, kk, qc, kc))
    off, post = kernels.build_index(kcd, n_c)
    dt = torch.int64 if i64 else torch.int32
    kw = dict(sorted=True, index_dtype=dt)
    got = kernels.select(qd, kd, qcd, off, post, b, k, **kw)
    ref = kernels.select(qd, kd, qcd, off, post, b, k, use_workspace=False, **kw)
    assert torch.equal(got, ref)
    # [B, heads, n, d] storage: other key and query strides
    qt, kt = (t.transpose(1, 2).contiguous().transpose(1, 2) for t in (qd, kd))
    assert torch.equal(kernels.select(qt, kt, qcd, off, post, b, k, **kw), ref)


@pytest.mark.parametrize("d,g", [(64, 2), (128, 5)])
def test_sorted_rows_with_denormal_scores(dev, d, g):
    """Keys, products and partial sums below the smallest normal number keep their bits.
    (Every row has fewer than k candidates: the order is this kernel's alone.)"""
    from ssa_amd import kernels

    n, h_kv, n_c, a, b, k = 1500, 1, 64, 8, 4, 1024
    q, kk = randn((1, n, h_kv * g, d), 74, torch.bfloat16), randn((1, n, h_kv, d), 75)
    gen = torch.Generator().manual_seed(76)
    scale = torch.tensor([1.0, 1e-38, 3e-39, 2e-40])[torch.randint(0, 4, (1, n, h_kv, 1), generator=gen)]
    kk = (kk * scale).to(torch.bfloat16)
    kc = torch.stack([torch.randperm(n_c, generator=gen)[:b] for _ in range(n)]).view(1, 1, n, b).int()
    qc = torch.stack([torch.randperm(n_c, generator=gen)[:a] for _ in range(n)]).view(1, 1, n, a).int()
    qd, kd, qcd, kcd = (t.to(dev) for t in (q, kk, qc, kc))
    off, post = kernels.build_index(kcd, n_c)
    got, stats = kernels.select(qd, kd, qcd, off, post, b, k, with_stats=True)
    assert int(stats[..., 0].max()) < k
    ref = kernels.select(qd, kd, qcd, off, post, b, k, use_workspace=False)
    assert torch.equal(got, ref)
