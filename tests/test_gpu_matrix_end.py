"""Grouped GEMMs over many experts with expert matrices of whole 2 MiB pages, the last expert among the routed ones.  What
the loads of a span may read is checked on the CPU (tests/test_sanitize.py): here a read past the end would show only where
nothing is mapped behind the matrix."""
import pytest
import torch

import oracle as orc
from hyper_amd import moe
from hyper_amd.formats import GType, q8_row_bytes, vec_dot_type
from tests.helpers import assert_bits_equal, gen, layer, oracle_layer

pytestmark = pytest.mark.gpu

# E x ff x d values of each type in whole 2 MiB pages (the granularity of large device allocations)
CASES = [(GType.Q8_0, 256, 512, 256), (GType.IQ4_NL, 256, 512, 256), (GType.MXFP4, 512, 512, 256)]


@pytest.mark.parametrize("t,E,d,ff", CASES)
def test_grouped_gemm_matrix_ends_the_allocation(cuda, t, E, d, ff):
    L = layer(t, t, E, ff, d, seed=31)
    assert L.gate.numel() % (2 << 20) == 0 and L.down.numel() % (2 << 20) == 0
    nt, k = 20, 2
    # every token takes the last expert and one other
    ids = torch.stack([torch.full((nt,), E - 1), torch.arange(nt) * 3], 1).to(torch.int32)
    wts = torch.rand(nt, k, generator=gen(32))
    x = torch.randn(nt, d, generator=gen(33))
    out_r, h_r, y_r = orc.moe_layer(oracle_layer(L), x.numpy(), ids.numpy(), wts.numpy(), want_hy=True)
    dev = moe.upload_experts(L, device=cuda)
    P, vt = nt * k, vec_dot_type(t)
    idsd, wtsd = ids.reshape(-1).to(cuda), wts.reshape(-1).to(cuda)
    order = torch.zeros(P, dtype=torch.int32, device=cuda)
    order_n = torch.zeros(2, dtype=torch.int32, device=cuda)
    egrp = torch.zeros(3 * E, dtype=torch.int32, device=cuda)
    moe.moe_order(dev, idsd, P, E, order, order_n, egrp=egrp)
    xq = torch.zeros(nt * q8_row_bytes(vt, d), dtype=torch.uint8, device=cuda)
    moe.q8_quantize(vt, x.to(cuda), d, d, nt, xq)
    h = torch.full((P, ff), float("nan"), device=cuda)
    moe.moe_gemm_gate_up(dev, xq, k, P, order, order_n, egrp, P, h)
    hq = torch.zeros(P * q8_row_bytes(vt, ff), dtype=torch.uint8, device=cuda)
    moe.q8_quantize(vt, h, ff, ff, P, hq)
    y = torch.full((P, d), float("nan"), device=cuda)
    moe.moe_gemm_down(dev, hq, P, order, order_n, egrp, P, wtsd, y)
    torch.cuda.synchronize()
    assert_bits_equal(h.cpu().numpy(), h_r, "h")
    assert_bits_equal(y.cpu().numpy(), (wts.numpy().reshape(-1, 1) * y_r).astype("float32"), "y")
