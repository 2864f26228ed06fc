"""Routing vectors on the fp32 matrix cores: bit-exact with the oracle's canonical
chains at the edges of the kernel's tiles, for every row layout it takes."""

import numpy as np
import pytest
import torch

from tests.helpers import f32, randn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("d,d_s,group,h_out,n", [
    (64, 32, 1, 3, 129),     # a second block of one token
    (64, 8, 8, 2, 200),      # one 16-byte piece of coordinates a lane
    (128, 32, 4, 2, 300),
    (128, 12, 7, 1, 257),    # coordinates that end inside a lane's pieces
    (128, 28, 16, 1, 260)])
def test_route_vectors_bit_exact(dev, orc, dtype, d, d_s, group, h_out, n):
    from ssa_amd import kernels

    B = 2
    x = randn((B, n, h_out * group, d), 11, dtype)
    x[0, 3] = 0.0                                   # a zero row stays zero
    x[1, n - 1, 0] *= 1e-30 if dtype == torch.float32 else 1.0
    w = randn((d_s, d), 12)
    got = kernels.route_vectors(x.to(dev), w.to(dev), group).cpu().numpy()
    # [B, heads, n, d] storage: rows of one head next to each other
    other = kernels.route_vectors(x.to(dev).transpose(1, 2).contiguous().transpose(1, 2), w.to(dev), group)
    np.testing.assert_array_equal(got, other.cpu().numpy())
    for b in range(B):
        np.testing.assert_array_equal(got[b], orc.route_vectors(f32(x[b]), f32(w), group))


def test_route_vectors_unaligned_rows_take_another_kernel(dev, orc):
    """Rows that start off 16 bytes (a slice of a wider tensor) give the same bits."""
    from ssa_amd import kernels

    x, w = randn((1, 300, 4, 72), 13), randn((32, 64), 14)
    xd = x.to(dev)[..., 1:65]
    got = kernels.route_vectors(xd, w.to(dev), 2).cpu().numpy()
    np.testing.assert_array_equal(got[0], orc.route_vectors(f32(x[0, ..., 1:65]), f32(w), 2))


def test_route_codes_queries_and_keys_in_one_launch(dev, orc):
    from ssa_amd import kernels

    B, n, h_q, h_kv, d, d_s, n_c = 1, 321, 6, 2, 64, 16, 128
    q, k = randn((B, n, h_q, d), 15, torch.bfloat16), randn((B, n, h_kv, d), 16, torch.bfloat16)
    wq, wk, cb = randn((d_s, d), 17), randn((d_s, d), 18), randn((h_kv, n_c, d_s), 19)
    qc, kc = kernels.route_codes(q.to(dev), k.to(dev), wq.to(dev), wk.to(dev), cb.to(dev), 8, 4)
    chat = orc.normalize(f32(cb))
    for x, w, g, top, got in ((q, wq, h_q // h_kv, 8, qc), (k, wk, 1, 4, kc)):
        ref = orc.code_topk(orc.route_vectors(f32(x[0]), f32(w), g), chat, top)
        np.testing.assert_array_equal(got[0].cpu().numpy(), ref)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("d,group", [(64, 1), (128, 3)])
def test_route_vectors_denormals_keep_their_bits(dev, orc, dtype, d, group):
    """Rows that are denormal, whose products are, and whose sums pass through the denormals."""
    from ssa_amd import kernels

    n, h_out, d_s = 160, 2, 32
    scale = torch.tensor([1.0, 1e-37, 1e-38, 3e-39, 2e-40, 1e-20])[torch.arange(n) % 6]
    x = (randn((1, n, h_out * group, d), 21) * scale[None, :, None, None]).to(dtype)
    w = randn((d_s, d), 22)
    w[1] *= 1e-20                                   # 1e-20 against 1e-20: products are denormal
    w[2] *= 1e-39                                   # itself denormal
    w[3, ::2] = 1.0
    w[3, 1::2] = -1.0                               # sums that cancel down to them
    got = kernels.route_vectors(x.to(dev), w.to(dev), group).cpu().numpy()
    xs = f32(x)
    assert (np.abs(xs[(xs != 0)]) < 1.1e-38).any()
    np.testing.assert_array_equal(got[0], orc.route_vectors(xs[0], f32(w), group))
