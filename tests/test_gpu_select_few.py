"""Index-order selection of a few rows (select_few_kernel, the decoding step's): equal to
the screened path over many rows and to the one-block-per-row kernel."""

import pytest
import torch

from tests.helpers import randn

pytestmark = pytest.mark.gpu


def _routed(n, n_q, h_kv, n_c, a, b, seed):
    gen = torch.Generator().manual_seed(seed)
    kc = torch.stack([torch.randperm(n_c, generator=gen)[:b] for _ in range(h_kv * n)]).view(1, h_kv, n, b).int()
    qc = torch.stack([torch.randperm(n_c, generator=gen)[:a] for _ in range(h_kv * n_q)]).view(1, h_kv, n_q, a).int()
    return qc, kc


@pytest.mark.parametrize("dtype,d,g,n,n_c,k,i64", [
    (torch.bfloat16, 128, 4, 3000, 64, 100, False),   # about 1000 candidates: scored and cut
    (torch.bfloat16, 64, 7, 3000, 512, 500, True),    # fewer than k: filler
    (torch.bfloat16, 128, 16, 2500, 40, 1, False),
    (torch.float32, 64, 3, 2000, 64, 300, True),      # vector-ALU chains
    (torch.bfloat16, 96, 2, 2000, 64, 300, False),    # a head dim without matrix chains
    (torch.bfloat16, 128, 2, 9000, 16, 700, False)])  # over 2048 candidates: the 256-thread kernel's way
def test_few_rows_equal_many_rows(dev, dtype, d, g, n, n_c, k, i64):
    from ssa_amd import kernels

    h_kv, a, b, m = 2, 8, 4, 5
    q, kk = randn((1, n, h_kv * g, d), 81, dtype), randn((1, n, h_kv, d), 82, dtype)
    kk[0, 100:160] = kk[0, :60]          # equal scores: ties go to the lower index
    qc, kc = _routed(n, n, h_kv, n_c, a, b, 83)
    qd, kd, qcd, kcd = (t.to(dev) for t in (q, kk, qc, kc))
    off, post = kernels.build_index(kcd, n_c)
    kw = dict(sorted=False, index_dtype=torch.int64 if i64 else torch.int32)
    ref = kernels.select(qd, kd, qcd, off, post, b, k, **kw)[:, n - m:]
    pfx = torch.empty(1, h_kv, m, device=dev, dtype=torch.int32)
    got = kernels.select(qd[:, n - m:], kd, qcd[:, :, n - m:], off, post, b, k, use_workspace=False,
                         row_prefix=pfx, **kw)
    assert torch.equal(got, ref)
    pref = torch.empty_like(pfx)
    kernels.select(qd[:, n - m:], kd, qcd[:, :, n - m:], off, post, b, k, row_prefix=pref, **kw)
    assert torch.equal(pfx, pref)
    # an explicit mask instead of the causal window
    mask = (torch.rand(n, n, generator=torch.Generator().manual_seed(84)) < 0.5).to(dev)
    from ssa_amd import _lib
    kw.update(mask_mode=_lib.MASK_DENSE, mask=mask)
    ref = kernels.select(qd, kd, qcd, off, post, b, k, **kw)[:, n - m:]
    got = kernels.select(qd[:, n - m:], kd, qcd[:, :, n - m:], off, post, b, k, use_workspace=False, **kw)
    assert torch.equal(got, ref)


def _tiny(t, seed):
    """t with rows whose products and partial sums with rows of order 1 are denormal, and rows
    that are denormal themselves."""
    gen = torch.Generator().manual_seed(seed)
    scale = torch.tensor([1.0, 1e-38, 3e-39, 2e-40])[torch.randint(0, 4, t.shape[:2], generator=gen)]
    return (t.float() * scale[..., None, None]).to(t.dtype)


@pytest.mark.parametrize("dtype,d,g,n,n_c,a,k,m,tiny", [
    (torch.bfloat16, 128, 4, 2000, 64, 8, 200, 256, False),     # as many rows as one kernel takes
    (torch.bfloat16, 128, 4, 2000, 64, 8, 200, 257, False),     # the other on both sides
    (torch.float32, 64, 2, 2000, 64, 8, 200, 60, False),
    (torch.bfloat16, 64, 3, 9000, 16, 8, 300, 100, False),      # past the list's cap
    (torch.bfloat16, 128, 16, 344000, 4096, 8, 1024, 3, False),  # over 64 KB of LDS, part of it static
    (torch.bfloat16, 128, 4, 2000, 64, 8, 200, 40, True),
    (torch.bfloat16, 64, 7, 2000, 64, 8, 200, 40, True)])
def test_few_rows_equal_one_block_per_row(dev, dtype, d, g, n, n_c, a, k, m, tiny):
    from ssa_amd import kernels

    b = 4
    q, kk = randn((1, m, g, d), 85, dtype), randn((1, n, 1, d), 86, dtype)
    if tiny:
        kk = _tiny(kk, 87)
    base = torch.randint(0, n_c, (1, 1, n, 1), generator=torch.Generator().manual_seed(88))
    kc = ((base + torch.arange(b) * (n_c // b)) % n_c).int()
    qc = ((base[:, :, :m] + torch.arange(a) * (n_c // a)) % n_c).int()
    qd, kd, qcd, kcd = (t.to(dev) for t in (q, kk, qc, kc))
    off, post = kernels.build_index(kcd, n_c)
    kw = dict(sorted=False, index_dtype=torch.int32, use_workspace=False)
    got = kernels.select(qd, kd, qcd, off, post, b, k, **kw)
    ref, _ = kernels.select(qd, kd, qcd, off, post, b, k, with_stats=True, **kw)   # statistics: select_kernel
    assert torch.equal(got, ref)
