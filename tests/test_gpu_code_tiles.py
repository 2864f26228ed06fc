"""Top codes of a moderate number of rows, the codebook split over a block's waves:
the same codes as the oracle at the edges of its tiles, lists and row counts."""

import numpy as np
import pytest
import torch

from tests.helpers import randn

pytestmark = pytest.mark.gpu


def _inputs(B, h, rows, n_c, d_s, seed):
    x = torch.nn.functional.normalize(randn((B, h, rows, d_s), seed), dim=-1)
    c = torch.nn.functional.normalize(randn((h, n_c, d_s), seed + 1), dim=-1)
    return x, c


@pytest.mark.parametrize("top,n_c,d_s,B,h,rows,temperature", [
    (1, 16, 4, 1, 5, 13, 1.0),       # 65 rows: the first call past the exhaustive path; one code tile
    (16, 16, 8, 1, 1, 81, 1.0),      # every code taken
    (4, 100, 32, 2, 2, 17, 0.7),     # codes that end inside a tile and a group of tiles
    (16, 127, 32, 1, 2, 203, 1.0),   # fewer tiles than the waves take; lists that may overflow
    (16, 640, 20, 1, 3, 333, 2.5),   # a group of tiles for one wave alone
    (16, 2047, 32, 1, 8, 1024, 1.0),  # the last count with 16 rows a block
    (16, 1000, 32, 3, 8, 343, 1.0),   # 32 rows a block, a ragged last one
    (32, 33, 32, 1, 2, 65, 1.0),
    (32, 4100, 32, 1, 4, 129, 1.0),
    (20, 520, 28, 1, 8, 1025, 1.0)])
def test_code_tiles_bit_exact(dev, orc, top, n_c, d_s, B, h, rows, temperature):
    from ssa_amd import kernels

    x, c = _inputs(B, h, rows, n_c, d_s, 31)
    x[0, 0, 3] = 0.0                                # every score ties: the lowest codes
    got = kernels.code_topk(x.to(dev), c.to(dev), top, temperature).cpu().numpy()
    for b in range(B):
        np.testing.assert_array_equal(got[b], orc.code_topk(x[b].numpy(), c.numpy(), top, temperature))


def test_code_tiles_overflowing_lists_and_infinite_rows(dev, orc):
    """Rows that fill their list (300 equal codes) and rows whose bound is infinite run exhaustively."""
    from ssa_amd import kernels

    x, c = _inputs(1, 2, 150, 700, 32, 33)
    c[1, 100:400] = c[1, 7]
    x[0, 1, ::5] = c[1, 7]
    x[0, 0, 11, 2] = float("inf")
    got = kernels.code_topk(x.to(dev), c.to(dev), 16).cpu().numpy()
    np.testing.assert_array_equal(got[0], orc.code_topk(x[0].numpy(), c.numpy(), 16))


@pytest.mark.parametrize("rows", [4096, 4097])      # 65536 query and key rows, and past them
def test_code_tiles_last_size_and_the_next(dev, rows):
    from ssa_amd import kernels

    h, d, d_s, n_c = 8, 64, 16, 512
    q, k = randn((1, rows, h, d), 35).to(dev), randn((1, rows, h, d), 36).to(dev)
    w, cb = randn((d_s, d), 37).to(dev), randn((h, n_c, d_s), 38).to(dev)
    chat = kernels.normalize_rows(cb)
    for got, x, top in zip(kernels.route_codes(q, k, w, w, cb, 16, 4), (q, k), (16, 4)):
        ref = kernels.code_topk(kernels.route_vectors(x, w, 1), chat, top, exhaustive=True)
        assert torch.equal(got, ref)


@pytest.mark.parametrize("shift,d_s", [(0, 20), (1, 32), (3, 12)])
def test_codebook_normalized_with_its_copy(dev, orc, shift, d_s):
    """A codebook off 16 bytes, with a zero code, gives the codes of the normalized rows."""
    from ssa_amd import kernels

    n, h, d, n_c = 150, 2, 64, 270
    q, k, w = randn((1, n, h, d), 41), randn((1, n, h, d), 42), randn((d_s, d), 43)
    cb = randn((h, n_c, d_s), 44)
    cb[0, 5] = 0.0
    flat = torch.empty(cb.numel() + shift, device=dev)
    cbd = flat[shift:].view(cb.shape)
    cbd.copy_(cb)
    chat = orc.normalize(cb.numpy())
    for got, x, top in zip(kernels.route_codes(q.to(dev), k.to(dev), w.to(dev), w.to(dev), cbd, 16, 4), (q, k), (16, 4)):
        ref = orc.code_topk(orc.route_vectors(x[0].numpy(), w.numpy(), 1), chat, top)
        np.testing.assert_array_equal(got[0].cpu().numpy(), ref)


@pytest.mark.parametrize("h,rows,n_c,top", [(2, 4096, 128, 16), (2, 4097, 128, 16), (2, 4097, 112, 16), (2, 4097, 113, 16),
                                            (3, 8192, 256, 8), (3, 8193, 256, 8), (3, 16384, 512, 20), (3, 16385, 512, 16),
                                            (3, 16385, 512, 17), (3, 16385, 64, 32)])
def test_code_tiles_on_both_sides_of_their_rule(dev, h, rows, n_c, top):
    """By the rows, and with a small codebook by what its lists would overrun."""
    from ssa_amd import kernels

    x, c = (t.to(dev) for t in _inputs(1, h, rows, n_c, 32, 51))
    assert torch.equal(kernels.code_topk(x, c, top), kernels.code_topk(x, c, top, exhaustive=True))


@pytest.mark.parametrize("rows,n_c,a", [(2049, 128, 16), (2049, 128, 8), (2049, 256, 32), (3072, 256, 16), (3073, 256, 16)])
def test_route_codes_on_both_sides_of_the_tiles_rule(dev, rows, n_c, a):
    from ssa_amd import kernels

    h, d, d_s = 8, 64, 32
    q, k = randn((1, rows, h, d), 55).to(dev), randn((1, rows, h, d), 56).to(dev)
    w, cb = randn((d_s, d), 57).to(dev), randn((h, n_c, d_s), 58).to(dev)
    chat = kernels.normalize_rows(cb)
    for got, x, top in zip(kernels.route_codes(q, k, w, w, cb, a, 4), (q, k), (a, 4)):
        ref = kernels.code_topk(kernels.route_vectors(x, w, 1), chat, top, exhaustive=True)
        assert torch.equal(got, ref)
