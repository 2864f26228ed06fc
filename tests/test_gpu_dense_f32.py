"""fp32 attention over selections that hold a good part of the keys (key tiles with
counts in LDS): several key windows, rows that fill no tile, repeated keys, dropped
slots, a processing order and non-finite values of keys a row did not select."""

import numpy as np
import pytest
import torch

from tests.helpers import f32, randn

pytestmark = pytest.mark.gpu


def _case(n, h_kv, g, d, k, seed):
    q, kk, v = randn((1, n, h_kv * g, d), seed), randn((1, n, h_kv, d), seed + 1), randn((1, n, h_kv, d), seed + 2)
    gen = torch.Generator().manual_seed(seed + 3)
    idx = torch.stack([torch.randperm(n, generator=gen)[:k] for _ in range(n * h_kv)]).view(1, n, h_kv, k)
    return q, kk, v, idx


@pytest.mark.parametrize("d,g,h_kv,n,k,causal,i64", [
    (64, 1, 2, 1999, 300, False, True),    # 16 rows a block, two key windows
    (64, 3, 2, 331, 70, True, False),      # 15 of 16 query vectors used
    (64, 4, 4, 1100, 300, True, True),     # two query tiles a block
    (128, 5, 1, 257, 100, True, True),
    (128, 16, 1, 40, 40, False, False),    # one row a block, all keys
    (64, 8, 1, 17, 30, False, True)])      # k > n: padded with key 0
def test_dense_f32_vs_oracle(dev, orc, d, g, h_kv, n, k, causal, i64):
    from ssa_amd import kernels

    q, kk, v, idx = _case(n, h_kv, g, d, min(k, n), 21)
    if k > n:
        idx = torch.cat((idx, idx.new_zeros(1, n, h_kv, k - n)), dim=-1)
    elif k < n:
        idx[..., 1] = idx[..., 0]  # counts twice
    idx = idx if i64 else idx.to(torch.int32)
    flag = torch.zeros(1, dtype=torch.int32, device=dev)
    order = torch.stack([torch.randperm(n) for _ in range(h_kv)]).to(torch.int32)[None]
    got = kernels.sparse_attention(q.to(dev), kk.to(dev), v.to(dev), idx.to(dev), None, causal, error_flag=flag)
    other = kernels.sparse_attention(q.to(dev), kk.to(dev), v.to(dev), idx.to(dev), None, causal,
                                     row_order=order.to(dev))
    assert int(flag.item()) == 0
    assert torch.equal(got, other), "a row's result must not depend on the rows it shares a block with"
    ref = orc.sparse_attention(f32(q[0]), f32(kk[0]), f32(v[0]), idx[0].to(torch.int64).numpy(), causal=causal)
    # 32-bit sums of at most n terms against 64 bits
    np.testing.assert_allclose(got[0].cpu().numpy(), ref, rtol=1e-5, atol=1e-5)


def test_dense_f32_non_finite_values_reach_their_rows_only(dev, orc):
    from ssa_amd import kernels

    n, h_kv, g, d, k = 96, 2, 4, 64, 48
    q, kk, v, idx = _case(n, h_kv, g, d, k, 31)
    v[0, 7, 0, 3] = float("inf")
    v[0, 50, 1, 60] = float("nan")
    kk[0, 20, 0, 0] = float("inf")
    got = kernels.sparse_attention(q.to(dev), kk.to(dev), v.to(dev), idx.to(dev))[0].cpu()
    has = torch.zeros(n, h_kv, n, dtype=torch.bool).scatter_(2, idx[0], True)
    clean = got.isfinite().view(n, h_kv, g, d)
    assert clean[~has[:, 0, 7] & ~has[:, 0, 20], 0].all() and clean[~has[:, 1, 50], 1].all()
    rows = has[:, 1, 50]
    assert not clean[rows, 1, :, 60].any() and clean[rows, 1, :, :60].all()


def test_dense_f32_flags_and_order(dev):
    from ssa_amd import kernels

    n, h_kv, g, d, k = 64, 1, 4, 64, 32
    q, kk, v, idx = _case(n, h_kv, g, d, k, 41)
    good = kernels.sparse_attention(q.to(dev), kk.to(dev), v.to(dev), idx.to(dev))
    bad = idx.clone()
    bad[0, 5, 0, 9] = n
    flag = torch.zeros(1, dtype=torch.int32, device=dev)
    out = kernels.sparse_attention(q.to(dev), kk.to(dev), v.to(dev), bad.to(dev), error_flag=flag)
    assert int(flag.item()) == 1
    keep = torch.arange(n) != 5
    assert torch.equal(out[0, keep], good[0, keep])
    order = torch.arange(n, dtype=torch.int32)[None, None].clone()
    order[0, 0, 9] = n                       # dropped: row 9 is never listed
    part = torch.full_like(good, 7.0)
    flag.zero_()
    kernels.sparse_attention(q.to(dev), kk.to(dev), v.to(dev), idx.to(dev), out=part, error_flag=flag,
                             row_order=order.to(dev))
    assert int(flag.item()) == 1 and (part[0, 9] == 7.0).all()
    keep = torch.arange(n) != 9
    assert torch.equal(part[0, keep], good[0, keep])


def _backward_oracle(orc, q, kk, v, idx, dout, causal):
    return orc.sparse_attention_backward(f32(q[0]), f32(kk[0]), f32(v[0]), idx[0].to(torch.int64).numpy(),
                                         dout[0].double().numpy(), causal=causal)


@pytest.mark.parametrize("d,g,h_kv,n,k,causal,i64", [
    (64, 1, 2, 1999, 300, False, True),    # several key windows, counted again for the second pass
    (64, 3, 2, 331, 70, True, False),      # 15 of 16 query vectors used
    (64, 4, 4, 700, 130, True, True),      # two query tiles a block
    (128, 5, 1, 257, 100, True, True),
    (128, 16, 1, 40, 40, False, False),
    (64, 8, 1, 17, 30, False, True)])      # k > n: padded with key 0
def test_dense_f32_backward_vs_oracle(dev, orc, d, g, h_kv, n, k, causal, i64):
    from ssa_amd import kernels

    q, kk, v, idx = _case(n, h_kv, g, d, min(k, n), 51)
    dout = randn((1, n, h_kv * g, d), 55)
    if k > n:
        idx = torch.cat((idx, idx.new_zeros(1, n, h_kv, k - n)), dim=-1)
    elif k < n:
        idx[..., 1] = idx[..., 0]
    idx = idx if i64 else idx.to(torch.int32)
    order = torch.stack([torch.randperm(n) for _ in range(h_kv)]).to(torch.int32)[None].to(dev)
    args = [t.to(dev) for t in (q, kk, v, idx)]
    out = kernels.sparse_attention(*args, None, causal)
    flag = torch.zeros(1, dtype=torch.int32, device=dev)
    got = kernels.sparse_attention_backward(*args, out, dout.to(dev), None, causal, error_flag=flag, row_order=order)
    assert int(flag.item()) == 0
    for x, ref in zip(got, _backward_oracle(orc, q, kk, v, idx, dout, causal)):
        # as tests/test_gpu_backward.py: 32-bit sums, atomics in any order
        assert np.abs(x[0].cpu().numpy() - ref).max() <= 2e-5 * np.abs(ref).max()


@pytest.mark.parametrize("what", ["k", "dout"])
def test_dense_f32_backward_keeps_non_finite_values_apart(dev, orc, what):
    """A key's or an output gradient's infinity reaches what its own pairs feed, nothing else."""
    from ssa_amd import kernels

    n, h_kv, g, d, k, at = 80, 1, 4, 64, 24, 11
    q, kk, v, idx = _case(n, h_kv, g, d, k, 61)
    dout = randn((1, n, g, d), 65)
    args = [t.to(dev) for t in (q, kk, v, idx)]
    out = kernels.sparse_attention(*args)
    has = torch.zeros(n, n, dtype=torch.bool).scatter_(1, idx[0, :, 0], True)   # row selects key
    ref = _backward_oracle(orc, q, kk, v, idx, dout, False)
    if what == "k":
        args[1][0, at, 0, 3] = float("inf")
        rows, keys = has[:, at], None
    else:
        dout[0, at, 2, 5] = float("inf")
        rows, keys = torch.arange(n) == at, has[at]
    if keys is None:
        keys = has[rows].any(0)
    got = [x[0].cpu() for x in kernels.sparse_attention_backward(*args, out, dout.to(dev))]
    for x, r, touched in ((got[0], ref[0], rows), (got[1], ref[1], keys), (got[2], ref[2], keys)):
        if bool((~touched).any()):
            np.testing.assert_allclose(x[~touched].numpy(), r[(~touched).numpy()], rtol=0, atol=2e-5 * np.abs(r).max())
    assert not got[0][rows].isfinite().all() and not got[1][keys].isfinite().all()


def _torch64(q, kk, v, idx, causal, dout=None):
    """The reference's gather -> softmax -> V (ssa/attention.py:64-113) in float64 on the
    CPU, NaN scores included; with dout the gradients of q, k and v."""
    q, kk, v = (t[0].double().requires_grad_(dout is not None) for t in (q, kk, v))
    n, h_q, d = q.shape
    h_kv = kk.shape[1]
    head = torch.arange(h_kv)[None, :, None]
    s = torch.einsum("nhgd,nhkd->nhgk", q.view(n, h_kv, -1, d), kk[idx[0], head]) / d**0.5
    if causal:
        s = s.masked_fill((idx[0] > torch.arange(n)[:, None, None])[:, :, None], -float("inf"))
    out = torch.einsum("nhgk,nhkd->nhgd", s.softmax(-1), v[idx[0], head]).reshape(n, h_q, d)
    return out if dout is None else torch.autograd.grad(out, (q, kk, v), dout[0].double())


def _one_key_per_tile(n, h_kv):
    """Row r selects the keys r mod 16 + 16 t, eight times each."""
    keys = torch.arange(n)[:, None] % 16 + 16 * torch.arange(n // 16)[None]
    return keys.repeat(1, 8)[None, :, None].expand(1, n, h_kv, -1).contiguous()


@pytest.mark.parametrize("g", [1, 4])
@pytest.mark.parametrize("what", ["causal", "strided", "query"])
def test_dense_f32_keeps_nan_scores(dev, what, g):
    """A NaN score reaches its row's output also where its wave of the block meets no
    other score of the row: K[16] alone in a causal row's second tile, one key a tile,
    every key (a NaN query)."""
    from ssa_amd import kernels

    n, h_kv, d = 64, 2, 64
    q, kk, v, idx = _case(n, h_kv, g, d, n, 71)
    causal = what == "causal"
    if what == "causal":
        idx = torch.arange(n).expand(1, n, h_kv, n).contiguous()
        kk[0, 16, 0, 5] = float("nan")
        kk[0, 0, 1, 5] = float("nan")       # row 0 selects nothing else
    elif what == "strided":
        idx = _one_key_per_tile(n, h_kv)
        kk[0, 19, 1, 0] = float("nan")
    else:
        q[0, 33, g, 63] = float("nan")
    got = kernels.sparse_attention(q.to(dev), kk.to(dev), v.to(dev), idx.to(dev), None, causal)[0].cpu()
    ref = _torch64(q, kk, v, idx, causal)
    assert ref.isnan().any() and ref.isfinite().any()
    # as test_dense_f32_vs_oracle
    np.testing.assert_allclose(got.numpy(), ref.numpy(), rtol=1e-5, atol=1e-5, equal_nan=True)


@pytest.mark.parametrize("d,g,n,k,n_q,i64", [
    (64, 1, 2500, 320, 1, False),     # few rows: each gathers its own keys
    (64, 1, 2500, 320, 700, True),
    (128, 2, 1300, 600, 40, True),    # tiles, 40 of 1300 positions
    (64, 1, 2500, 2500, 64, False)])  # three windows, every key
def test_dense_f32_rows_at_the_end_vs_oracle(dev, orc, d, g, n, k, n_q, i64):
    """A block of n_q query rows at the last positions, on both sides of the rule that
    weighs the tiles against the rows' gathers."""
    from ssa_amd import kernels

    q, kk, v, idx = _case(n, 1, g, d, k, 101)
    rows = np.arange(n - n_q, n)
    idx = idx[:, n - n_q:] if i64 else idx[:, n - n_q:].to(torch.int32)
    flag = torch.zeros(1, dtype=torch.int32, device=dev)
    got = kernels.sparse_attention(q[:, n - n_q:].to(dev), kk.to(dev), v.to(dev), idx.to(dev), None, True,
                                   error_flag=flag)
    assert int(flag.item()) == 0
    ref = orc.sparse_attention(f32(q[0]), f32(kk[0]), f32(v[0]), idx[0].to(torch.int64).numpy(), causal=True, rows=rows)
    # as test_dense_f32_vs_oracle
    np.testing.assert_allclose(got[0].cpu().numpy(), ref, rtol=1e-5, atol=1e-5)


def _check_backward(dev, q, kk, v, idx, causal):
    from ssa_amd import kernels

    dout = randn(q.shape, 85)
    args = [t.to(dev) for t in (q, kk, v, idx)]
    out = kernels.sparse_attention(*args, None, causal)
    got = kernels.sparse_attention_backward(*args, out, dout.to(dev), None, causal)
    for x, ref in zip(got, _torch64(q, kk, v, idx, causal, dout)):
        # as test_dense_f32_backward_vs_oracle
        atol = 2e-5 * float(ref[ref.isfinite()].abs().max())
        np.testing.assert_allclose(x[0].cpu().numpy(), ref.numpy(), rtol=0, atol=atol, equal_nan=True)


@pytest.mark.parametrize("g", [1, 4])
@pytest.mark.parametrize("what", ["strided", "query"])
def test_dense_f32_backward_keeps_nan_scores(dev, what, g):
    """A NaN score makes its row's whole softmax NaN, and with it dv and dk of every key
    that the row selects, also where its wave meets no other score of the row."""
    n, h_kv, d = 64, 2, 64
    q, kk, v, idx = _case(n, h_kv, g, d, 24, 81)
    if what == "strided":
        idx = _one_key_per_tile(n, h_kv)
        kk[0, 19, 1, 0] = float("nan")
    else:
        q[0, 33, g, 63] = float("nan")
    _check_backward(dev, q, kk, v, idx, False)


def test_dense_f32_backward_unused_query_vectors_add_nothing(dev):
    """g = 3 leaves query vectors of a block without a row: they must not meet a key whose
    infinity (a score of -inf for the rows that select it) would make them NaN."""
    n, h_kv, g, d, at = 80, 2, 3, 64, 11
    q, kk, v, idx = _case(n, h_kv, g, d, 24, 91)
    q[0, :, :, 7] = q[0, :, :, 7].abs() + 0.1
    kk[0, at, 1, 7] = -float("inf")
    _check_backward(dev, q, kk, v, idx, False)


@pytest.mark.parametrize("g", [9, 13])
def test_dense_f32_backward_on_both_sides_of_its_rule(dev, g):
    """d = 128, n / k just under 5, more rows than the rule counts as few: nine heads go
    row by row, thirteen by key tiles."""
    from ssa_amd import kernels

    n, d, k = 2100, 128, 430
    q, kk, v, idx = (t.to(dev) for t in _case(n, 1, g, d, k, 111))
    dout = randn((1, n, g, d), 115).to(dev)
    out = kernels.sparse_attention(q, kk, v, idx)
    got = kernels.sparse_attention_backward(q, kk, v, idx, out, dout)
    q64, k64, v64 = (t[0].double().transpose(0, 1).contiguous().requires_grad_(True) for t in (q, kk, v))
    off = torch.ones(n, n, dtype=torch.bool, device=dev).scatter_(1, idx[0, :, 0], False)
    p = (torch.matmul(q64, k64[0].t().contiguous()) / d**0.5).masked_fill(off, -float("inf")).softmax(-1)
    ref = torch.autograd.grad(torch.matmul(p, v64[0]), (q64, k64, v64), dout[0].double().transpose(0, 1))
    for x, r in zip(got, ref):
        # as test_dense_f32_backward_vs_oracle
        assert float((x[0] - r.transpose(0, 1)).abs().max()) <= 2e-5 * float(r.abs().max())
