"""Grouped GEMMs of every type against the oracle, on each kernel a launch can take: blocks of 8 waves (grids that leave half
of the CUs idle), each type's own block width (larger grids), and for the types with Q8_0 activations the register-staged
kernel of launches beyond 32-bit activation offsets.  The launch is chosen from n_pairs, an upper bound of the pairs in
`order`; the kernels themselves follow order_n and egrp, so a large bound takes a small problem down the other routes."""
import numpy as np
import pytest
import torch

import oracle as orc
from hyper_amd import moe
from hyper_amd.formats import GType, block_bytes, q8_row_bytes, vec_dot_type
from tests.helpers import ALL_TYPES, assert_bits_equal, gen, layer, oracle_layer

pytestmark = pytest.mark.gpu

TYPES_Q8_0 = [t for t in ALL_TYPES if vec_dot_type(t) == GType.Q8_0]
OWN_WIDTH = 1 << 15      # 512 items: more 16-wave blocks than half of the CUs, whatever the shape
STAGED = 1 << 24         # 4.25 GiB of Q8_0 rows of 256 values
ROUTES = ([(t, b) for t in ALL_TYPES for b in (0, OWN_WIDTH)] + [(t, STAGED) for t in TYPES_Q8_0])
# tokens of each expert: one, the edges of a 16-token tile and of a 64-token item, none, several items
COUNTS = [1, 16, 17, 33, 0, 48, 64, 65, 129]


def grouped(cuda, L, x, ids, wts, bound, k=1):
    """hy_moe_order, gate/up, the quantizer and down of pairs ids [nt, k], launched for `bound` pairs (0: as many as there are)"""
    P, E = ids.numel(), L.E
    dev = moe.upload_experts(L, device=cuda)
    vg, vd = vec_dot_type(L.tg), vec_dot_type(L.td)
    idsd, wtsd = ids.reshape(-1).to(cuda), wts.reshape(-1).to(cuda)
    order = torch.zeros(P, dtype=torch.int32, device=cuda)
    order_n = torch.zeros(2, dtype=torch.int32, device=cuda)
    egrp = torch.zeros(3 * E, dtype=torch.int32, device=cuda)
    moe.moe_order(dev, idsd, P, E, order, order_n, egrp=egrp)
    xq = torch.zeros(x.shape[0] * q8_row_bytes(vg, L.n), dtype=torch.uint8, device=cuda)
    moe.q8_quantize(vg, x.to(cuda), L.n, L.n, x.shape[0], xq)
    h = torch.full((P, L.ff), float("nan"), device=cuda)
    moe.moe_gemm_gate_up(dev, xq, k, bound or P, order, order_n, egrp, E, h)
    hq = torch.zeros(P * q8_row_bytes(vd, L.ff), dtype=torch.uint8, device=cuda)
    moe.q8_quantize(vd, h, L.ff, L.ff, P, hq)
    y = torch.full((P, L.n), float("nan"), device=cuda)
    moe.moe_gemm_down(dev, hq, bound or P, order, order_n, egrp, E, wtsd, y)
    torch.cuda.synchronize()
    return h.cpu().numpy(), y.cpu().numpy()


def check(cuda, L, x, ids, wts, bound, k=1):
    _, h_r, y_r = orc.moe_layer(oracle_layer(L), x.numpy(), ids.numpy(), wts.numpy(), want_hy=True)
    h, y = grouped(cuda, L, x, ids, wts, bound, k)
    assert_bits_equal(h, h_r, "h")
    with np.errstate(invalid="ignore"):
        assert_bits_equal(y, (wts.numpy().reshape(-1, 1) * y_r).astype(np.float32), "y")
    return y


def routed(counts, seed):
    """pairs of one expert each, counts[e] of expert e, in a random order"""
    ids = torch.repeat_interleave(torch.arange(len(counts), dtype=torch.int32), torch.tensor(counts))
    return ids[torch.randperm(ids.numel(), generator=gen(seed))].reshape(-1, 1)


@pytest.mark.parametrize("t,bound", ROUTES)
def test_token_edges(cuda, t, bound):
    """one span (d 256) and three (ff 768)"""
    L = layer(t, t, len(COUNTS), 768, 256, seed=91)
    ids = routed(COUNTS, 92)
    nt = ids.shape[0]
    check(cuda, L, torch.randn(nt, 256, generator=gen(93)), ids, torch.rand(nt, 1, generator=gen(94)), bound)


@pytest.mark.parametrize("t", TYPES_Q8_0)
@pytest.mark.parametrize("bound", [0, STAGED])
def test_rows_shared_by_pairs(cuda, t, bound):
    """three pairs a row of x"""
    L = layer(t, t, 6, 256, 512, seed=95)
    ids = torch.stack([torch.randperm(6, generator=gen(96 + i))[:3] for i in range(50)]).to(torch.int32)
    check(cuda, L, torch.randn(50, 512, generator=gen(97)), ids, torch.rand(50, 3, generator=gen(98)), bound, k=3)


@pytest.mark.parametrize("t,bound", [(t, b) for t in TYPES_Q8_0 for b in (0, OWN_WIDTH, STAGED)])
def test_scales_out_of_range_past_the_first_span(cuda, t, bound):
    """down rows with infinite, NaN and subnormal scales (MXFP4: the largest and smallest exponents) in the second and in the
    last of three spans, items of one to four tiles: the sums of the spans before and after, and the finite rows beside
    them in a wave's sixteen, stay the oracle's"""
    d, ff, counts = 256, 768, [9, 20, 40, 64]
    L = layer(t, t, len(counts), ff, d, seed=99)
    blk = L.down.view(len(counts), d, ff // 32, block_bytes(t))
    marks = ((3, 255, 0x7C00), (20, 254, 0xFC00), (70, 0, 0x7E00), (100, 1, 0x0001), (200, 230, 0x83FF))
    for row, e, bits in marks:
        for at, r in ((10, row), (23, row + 4)):   # a block of the second span, the last block of the last
            if t == GType.MXFP4:
                blk[:, r, at, 0] = e
            else:
                blk[:, r, at, 0], blk[:, r, at, 1] = bits & 255, bits >> 8
    ids = routed(counts, 101)
    y = check(cuda, L, torch.randn(sum(counts), d, generator=gen(102)), ids, torch.ones(sum(counts), 1), bound)
    if t != GType.MXFP4:
        assert not np.isfinite(y).all() and np.isfinite(y[:, [2, 4, 19, 21, 69, 71]]).all()
