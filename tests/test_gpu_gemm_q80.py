"""Grouped GEMMs of the types with Q8_0 activations: token counts at the edges of a 16-token tile and of a 64-token item,
scales that leave the ordinary range (infinite, NaN and subnormal weight scales, subnormal activation scales)."""
import numpy as np
import pytest
import torch

import oracle as orc
from hyper_amd import moe
from hyper_amd.formats import GType, block_bytes, q8_row_bytes
from tests.helpers import assert_bits_equal, gen, layer, oracle_layer

pytestmark = pytest.mark.gpu

TYPES = [GType.IQ4_NL, GType.MXFP4, GType.Q8_0, GType.Q5_0, GType.Q5_1]


def _grouped(cuda, t, L, x, ids, wts):
    nt, E, d, ff = x.shape[0], L.E, L.n, L.ff
    out_r, h_r, y_r = orc.moe_layer(oracle_layer(L), x.numpy(), ids.numpy(), wts.numpy(), want_hy=True)
    dev = moe.upload_experts(L, device=cuda)
    idsd, wtsd = ids.reshape(-1).to(cuda), wts.reshape(-1).to(cuda)
    order = torch.zeros(nt, dtype=torch.int32, device=cuda)
    order_n = torch.zeros(2, dtype=torch.int32, device=cuda)
    egrp = torch.zeros(3 * E, dtype=torch.int32, device=cuda)
    moe.moe_order(dev, idsd, nt, E, order, order_n, egrp=egrp)
    xq = torch.zeros(nt * q8_row_bytes(GType.Q8_0, d), dtype=torch.uint8, device=cuda)
    moe.q8_quantize(GType.Q8_0, x.to(cuda), d, d, nt, xq)
    h = torch.full((nt, ff), float("nan"), device=cuda)
    moe.moe_gemm_gate_up(dev, xq, 1, nt, order, order_n, egrp, E, h)
    hq = torch.zeros(nt * q8_row_bytes(GType.Q8_0, ff), dtype=torch.uint8, device=cuda)
    moe.q8_quantize(GType.Q8_0, h, ff, ff, nt, hq)
    y = torch.zeros(nt, d, device=cuda)
    moe.moe_gemm_down(dev, hq, nt, order, order_n, egrp, E, wtsd, y)
    torch.cuda.synchronize()
    assert_bits_equal(h.cpu().numpy(), h_r, "h")
    with np.errstate(invalid="ignore"):
        assert_bits_equal(y.cpu().numpy(), (wts.numpy().reshape(-1, 1) * y_r).astype(np.float32), "y")
    return y


@pytest.mark.parametrize("t", TYPES)
@pytest.mark.parametrize("n", [1, 16, 17, 33, 48, 64, 65, 129])
def test_token_edges(cuda, t, n):
    """n tokens of expert 0, five of expert 2, none of expert 1; one span (d 256) and three (ff 768)."""
    L = layer(t, t, 3, 768, 256, seed=41)
    nt = n + 5
    ids = torch.tensor([0] * n + [2] * 5, dtype=torch.int32).reshape(nt, 1)[torch.randperm(nt, generator=gen(42))]
    _grouped(cuda, t, L, torch.randn(nt, 256, generator=gen(43)), ids, torch.rand(nt, 1, generator=gen(44)))


@pytest.mark.parametrize("t", TYPES)
def test_scales_out_of_range(cuda, t):
    """down rows with infinite, NaN and subnormal scales (MXFP4: the largest and smallest exponents), and activations
    small enough for subnormal Q8_0 scales."""
    d, ff, nt = 512, 256, 40
    L = layer(t, t, 2, ff, d, seed=45)
    blk = L.down.view(2, d, ff // 32, block_bytes(t))
    if t == GType.MXFP4:
        for row, e in ((3, 255), (20, 254), (70, 0), (100, 1), (200, 230)):
            blk[:, row, 2, 0] = e
    else:
        for row, bits in ((3, 0x7C00), (20, 0xFC00), (70, 0x7E00), (100, 0x0001), (200, 0x83FF), (300, 0x7BFF)):
            blk[:, row, 2, 0] = bits & 255
            blk[:, row, 2, 1] = bits >> 8
    x = torch.randn(nt, d, generator=gen(46))
    x[::3] *= 1e-4
    ids = torch.arange(nt, dtype=torch.int32).reshape(nt, 1) % 2
    y = _grouped(cuda, t, L, x, ids, torch.ones(nt, 1))
    if t != GType.MXFP4:
        assert not torch.isfinite(y).all() and torch.isfinite(y[:, 300]).all()
