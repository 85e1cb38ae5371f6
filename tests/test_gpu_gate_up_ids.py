"""Decode gate/up by ids from the Q8 rows (hy_moe_gate_up_q8): the bits of hy_moe_gate_up, with and without the Q8_0 hidden
rows, absent experts left unwritten; a sigmoid-routed decode on it, and past its limits, against the oracle."""
import numpy as np
import pytest
import torch

import oracle as orc
from hyper_amd import HyError, moe
from hyper_amd.formats import GType, q8_row_bytes, vec_dot_type
from tests.helpers import assert_bits_equal, gen, layer, oracle_layer

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("t,d,ff,nt,k", [(GType.Q8_0, 2048, 1024, 2, 8), (GType.IQ4_NL, 4096, 256, 1, 3), (GType.MXFP4, 256, 512, 9, 4),
                                         (GType.Q4_K, 2048, 768, 4, 8), (GType.IQ2_XS, 7168, 256, 3, 6), (GType.Q6_K, 512, 256, 33, 16)])
def test_bits_of_moe_gate_up(cuda, t, d, ff, nt, k):
    E = 20
    L = layer(t, t, E, ff, d, seed=51)
    slot = torch.arange(E, dtype=torch.int32)
    slot[4] = -1
    dev = moe.MoeDev(L.to(cuda), slot.to(cuda))
    ids = torch.stack([torch.randperm(E, generator=gen(52 + i))[:k] for i in range(nt)]).to(torch.int32).reshape(-1)
    ids[0] = 4
    x = torch.randn(nt, d, generator=gen(53)).to(cuda)
    idsd = ids.to(cuda)
    ref = torch.full((nt * k, ff), 7.0, device=cuda)
    moe.moe_gate_up(dev, x, d, idsd, k, ref, nt)
    xq = torch.zeros(nt * q8_row_bytes(vec_dot_type(t), d), dtype=torch.uint8, device=cuda)
    moe.q8_quantize(vec_dot_type(t), x, d, d, nt, xq)
    h = torch.full((nt * k, ff), 7.0, device=cuda)
    moe.moe_gate_up_q8(dev, xq, idsd, E, k, h, None, nt)
    torch.cuda.synchronize()
    assert_bits_equal(h.cpu().numpy(), ref.cpu().numpy(), "h")
    hq = torch.zeros(nt * k * q8_row_bytes(GType.Q8_0, ff), dtype=torch.uint8, device=cuda)
    if vec_dot_type(t) != GType.Q8_0:
        with pytest.raises(HyError):
            moe.moe_gate_up_q8(dev, xq, idsd, E, k, h, hq, nt)
        return
    h2 = torch.full((nt * k, ff), 7.0, device=cuda)
    moe.moe_gate_up_q8(dev, xq, idsd, E, k, h2, hq, nt)
    wts = torch.rand(nt * k, generator=gen(54)).to(cuda)
    a, b = torch.zeros(nt, d, device=cuda), torch.zeros(nt, d, device=cuda)
    moe.moe_down_reduce(dev, h, idsd, wts, k, None, None, a, nt)
    moe.moe_down_reduce_q8(dev, hq, idsd, wts, k, None, None, b, False, nt)
    torch.cuda.synchronize()
    assert_bits_equal(h2.cpu().numpy(), ref.cpu().numpy(), "h with hq")
    assert_bits_equal(b.cpu().numpy(), a.cpu().numpy(), "down from hq")


@pytest.mark.parametrize("t,shared", [(GType.Q8_0, False), (GType.IQ4_NL, True)])
def test_sigmoid_decode(cuda, t, shared):
    E, d, ff, k, scale = 24, 1024, 512, 4, 1.5
    L = layer(t, t, E, ff, d, seed=55)
    S = layer(t, t, 1, ff, d, seed=56) if shared else None
    rng = np.random.default_rng(57)
    W_r = (rng.standard_normal((E, d)) * 0.05).astype(np.float32)
    rb = rng.uniform(-0.05, 0.05, E).astype(np.float32)
    dev = moe.MoeDev(L.to(cuda), torch.arange(E, dtype=torch.int32, device=cuda))
    sh = moe.MoeDev(S.to(cuda), torch.zeros(1, dtype=torch.int32, device=cuda)) if shared else None
    r = moe.MoeLayerRunner(dev, torch.from_numpy(W_r).to(cuda), k, max_rows=12, router="sigmoid", shared=sh,
                           router_bias=torch.from_numpy(rb).to(cuda), router_scale=scale)
    for nt in (1, 3, 12):
        x = torch.randn(nt, d, generator=gen(58 + nt)).numpy()
        resid = torch.randn(nt, d, generator=gen(59))
        out = r.decode(torch.from_numpy(x).to(cuda)).clone()
        got = r.decode(torch.from_numpy(x).to(cuda), resid=resid.to(cuda)).clone()
        torch.cuda.synchronize()
        ids, wts, _ = orc.route_sig(orc.gemv_f32(W_r, x), rb, E, k, scale)
        sho = orc.moe_layer(oracle_layer(S), x, np.zeros((nt, 1), np.int32), np.ones((nt, 1), np.float32)) if shared else None
        _, _, y = orc.moe_layer(oracle_layer(L), x, ids, wts, want_hy=True)
        y = (wts.reshape(-1, 1) * y).astype(np.float32).reshape(nt, k, d)
        ref = np.zeros((nt, d), np.float32)
        for i in range(nt):
            acc = sho[i].copy() if shared else None
            for j in np.argsort(ids[i], kind="stable"):
                acc = y[i, j].copy() if acc is None else (acc + y[i, j]).astype(np.float32)
            ref[i] = acc
        assert_bits_equal(out.cpu().numpy(), ref, f"out nt={nt}")
        assert_bits_equal(got.cpu().numpy(), (resid.numpy() + ref).astype(np.float32), f"resid nt={nt}")


@pytest.mark.parametrize("t,d,ff,E,k,nt", [(GType.Q8_0, 256, 256, 20, 16, 4097),    # 65552 pairs: also the fp32 hidden, not the Q8_0 rows
                                           (GType.Q4_K, 8448, 256, 6, 2, 3)])        # d past 8192
def test_sigmoid_decode_past_the_limits(cuda, t, d, ff, E, k, nt):
    """MoeLayerRunner falls back to hy_moe_gate_up"""
    L = layer(t, t, E, ff, d, seed=61)
    rng = np.random.default_rng(62)
    W_r = (rng.standard_normal((E, d)) * 0.05).astype(np.float32)
    rb = rng.uniform(-0.05, 0.05, E).astype(np.float32)
    dev = moe.MoeDev(L.to(cuda), torch.arange(E, dtype=torch.int32, device=cuda))
    r = moe.MoeLayerRunner(dev, torch.from_numpy(W_r).to(cuda), k, max_rows=nt, router="sigmoid",
                           router_bias=torch.from_numpy(rb).to(cuda))
    x = torch.randn(nt, d, generator=gen(63))
    out = r.decode(x.to(cuda)).clone()
    torch.cuda.synchronize()
    tok = np.arange(nt) if nt < 24 else np.r_[0, np.sort(rng.choice(nt, 22, replace=False)), nt - 1]
    xs = x.numpy()[tok]
    ids, wts, _ = orc.route_sig(r.logits.cpu().numpy()[tok, :E], rb, E, k, 1.0)
    _, _, y = orc.moe_layer(oracle_layer(L), xs, ids, wts, want_hy=True)
    y = (wts.reshape(-1, 1) * y).astype(np.float32).reshape(len(tok), k, d)
    ref = np.zeros((len(tok), d), np.float32)
    for i in range(len(tok)):
        order = np.argsort(ids[i], kind="stable")
        acc = y[i, order[0]].copy()
        for j in order[1:]:
            acc = (acc + y[i, j]).astype(np.float32)
        ref[i] = acc
    assert_bits_equal(out.cpu().numpy()[tok], ref, "out")
