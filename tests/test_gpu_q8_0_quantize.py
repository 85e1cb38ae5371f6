"""Q8_0 rows from 16-byte loads (aligned x) against the general kernel (x off its alignment) and the oracle: one block,
odd block counts, partial last groups, zero, infinite, tiny and huge values."""
import numpy as np
import pytest
import torch

import oracle as orc
from hyper_amd import moe
from hyper_amd.formats import GType, q8_row_bytes
from tests.helpers import gen

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,nt,pad", [(32, 1, 0), (32, 33, 4), (96, 5, 0), (256, 3, 8), (1536, 67, 0), (4096, 9, 4)])
def test_routes_agree(cuda, n, nt, pad):
    x = torch.randn(nt, n + pad, generator=gen(71))
    x[0, :32] = 0.0
    x[-1, n - 32:n] *= 1e-30          # a scale below fp16's smallest (127 / the largest value stays finite)
    x[-1, 0] = 3e38
    x[nt // 2, n - 1] = float("inf")
    flat = torch.zeros(x.numel() + 4)
    nb = nt * q8_row_bytes(GType.Q8_0, n)
    out = []
    for off in (0, 1):                # floats off a 16-byte boundary
        flat[off:off + x.numel()] = x.reshape(-1)
        xd = flat.to(cuda)[off:]
        assert xd.data_ptr() % 16 == 4 * off
        q = torch.full((nb + 2,), 0xA5, dtype=torch.uint8, device=cuda)
        moe.q8_quantize(GType.Q8_0, xd, n + pad, n, nt, q)
        torch.cuda.synchronize()
        assert q[nb:].tolist() == [0xA5, 0xA5]   # nothing past the rows
        out.append(q[:nb].cpu().numpy())
    np.testing.assert_array_equal(out[0], out[1])
    fin = [t for t in range(nt) if t != nt // 2]   # (an infinite block's bytes are pinned by the route above alone)
    if fin:
        ref = orc.quantize(GType.Q8_0, x[fin, :n].contiguous().numpy())
        np.testing.assert_array_equal(out[0].reshape(nt, -1)[fin], ref.reshape(len(fin), -1))


def test_routes_agree_on_nan(cuda):
    """NaN beside ordinary values, beside an infinity and alone in a block: the general kernel's bytes"""
    n, nt = 96, 4
    x = torch.randn(nt, n, generator=gen(72))
    x[0, 5] = float("nan")
    x[1, 32:64] = float("nan")
    x[2, 64], x[2, 95] = float("inf"), float("nan")
    x[3, ::4] = float("nan")          # one value of every lane
    flat = torch.zeros(x.numel() + 4)
    out = []
    for off in (0, 1):
        flat[off:off + x.numel()] = x.reshape(-1)
        xd = flat.to(cuda)[off:]
        q = torch.zeros(nt * q8_row_bytes(GType.Q8_0, n), dtype=torch.uint8, device=cuda)
        moe.q8_quantize(GType.Q8_0, xd, n, n, nt, q)
        torch.cuda.synchronize()
        out.append(q.cpu().numpy())
    np.testing.assert_array_equal(out[0], out[1])
