"""The index and the query order of heads small enough for one block: a stable sort by
code at the edges of its waves and chunks, with codes out of range left out."""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _codes(rng, shape, n_c, kind):
    if kind == "one":
        return np.full(shape, n_c - 1, np.int32)
    c = rng.integers(0, n_c, shape).astype(np.int32)
    if kind == "few":
        c = np.where(rng.random(shape) < 0.9, c % 3, c).astype(np.int32)
    if kind == "outside":
        c = np.where(rng.random(shape) < 0.3, rng.choice([-1, n_c, 1 << 20], shape), c).astype(np.int32)
    return c


@pytest.mark.parametrize("n,b,n_c,kind", [
    (1, 1, 1, "any"), (63, 1, 31, "any"), (64, 4, 32, "few"), (341, 3, 1023, "any"), (256, 4, 1024, "one"),
    (1025, 1, 1024, "outside"), (1171, 7, 4096, "any"), (2048, 4, 2048, "few"), (8192, 1, 16384, "any"),
    (8191, 1, 16384, "outside"), (2049, 4, 512, "any")])
def test_index_of_small_heads(dev, n, b, n_c, kind):
    from ssa_amd import kernels

    rng = np.random.default_rng(n * b)
    B, h = 2, 3
    codes = _codes(rng, (B, h, n, b), n_c, kind)
    off, post = (t.cpu().numpy() for t in kernels.build_index(torch.from_numpy(codes).to(dev), n_c))
    for i in np.ndindex(B, h):
        flat = codes[i].reshape(-1)
        keys = np.arange(n * b) // b
        ok = (flat >= 0) & (flat < n_c)
        ref = keys[ok][np.argsort(flat[ok], kind="stable")]
        np.testing.assert_array_equal(off[i], np.searchsorted(np.sort(flat[ok]), np.arange(n_c + 1)))
        np.testing.assert_array_equal(post[i][: len(ref)], ref)


@pytest.mark.parametrize("n,a,n_c,shift", [(1, 1, 2, 0), (203, 8, 512, 0), (1000, 5, 97, 0), (8192, 16, 4096, 0),
                                           (8192, 4, 4096, 1), (8193, 4, 4096, 0)])
def test_query_order_of_small_heads(dev, n, a, n_c, shift):
    from ssa_amd import kernels

    rng = np.random.default_rng(n + a)
    codes = _codes(rng, (2, 2, n, a), n_c, "any")
    flat = torch.empty(codes.size + shift, dtype=torch.int32, device=dev)
    q = flat[shift:].view(codes.shape)              # shift: rows off 16 bytes
    q.copy_(torch.from_numpy(codes))
    got = kernels.query_order(q, n_c).cpu().numpy()
    np.testing.assert_array_equal(got, np.argsort(codes.min(-1), axis=-1, kind="stable"))


@pytest.mark.parametrize("bh,n,a,n_c", [
    (2, 4096, 16, 512), (2, 4097, 15, 512), (2, 4096, 17, 512), (2, 8192, 16, 4095), (2, 8192, 16, 4096),
    (2, 8192, 17, 4096), (31, 8192, 1, 512), (32, 8192, 1, 512), (16, 4096, 33, 1000)])
def test_query_order_on_both_sides_of_its_rule(dev, bh, n, a, n_c):
    """One launch, or the minima and the four kernels: by the rows, codes and heads."""
    from ssa_amd import kernels

    codes = np.random.default_rng(n + a + n_c).integers(0, n_c, (1, bh, n, a)).astype(np.int32)
    got = kernels.query_order(torch.from_numpy(codes).to(dev), n_c).cpu().numpy()
    np.testing.assert_array_equal(got, np.argsort(codes.min(-1), axis=-1, kind="stable"))
    off, post = (t.cpu().numpy() for t in kernels.build_index(torch.from_numpy(codes[..., :1].copy()).to(dev), n_c))
    np.testing.assert_array_equal(post, np.argsort(codes[..., 0], axis=-1, kind="stable"))
    for h in range(bh):
        np.testing.assert_array_equal(off[0, h], np.searchsorted(np.sort(codes[0, h, :, 0]), np.arange(n_c + 1)))
