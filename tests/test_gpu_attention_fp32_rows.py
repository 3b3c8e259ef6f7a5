"""How the fp32 attention kernel reads K and V: through a range that ends with
the last row, as long as rows do not overlap and a block's offsets fit 31 bits,
otherwise element by element. Memory outside the rows holds NaN, which no
masked key may bring in; against the oracle at the fp32 contract (1e-5
relative)."""

import numpy as np
import pytest
import torch

import oracle
from helpers import TOL_F32_REL, randn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize("Sk,stride", [
    (1, 0), (15, 4), (17, 4), (47, 60), (131, 0),  # floats between rows
    (17, (1 << 25) - 4), (17, 1 << 25),  # the longest rows the range form takes, and past them
    (17, -16),  # rows that overlap
])
@pytest.mark.parametrize("heads", [1, 260])  # sixteen-row and 32-row work-groups
def test_rows(heads, Sk, stride, D):
    from neptune_hip import ops
    print(f"case: fp32 rows heads={heads} Sk={Sk} D={D} stride={stride}", flush=True)
    row = stride if stride > 1 << 20 else D + stride
    hk = 1  # every query head reads the same K and V head
    n = (Sk - 1) * row + D
    kv = []
    for seed in (1, 2):
        buf = torch.empty(n + 64 * D, device="cuda")
        if row < 1 << 20:
            buf.fill_(float("nan"))
        else:
            buf[n:] = float("nan")
        t = buf.as_strided((1, hk, Sk, D), (n, n, row, 1), 0)
        src = randn((n,) if row < D else (1, hk, Sk, D), seed=seed, dtype=torch.float32)
        if row < D:
            buf[:n] = src.cuda()
        else:
            t.copy_(src)
        kv.append(t)
    q = randn((1, heads, 33, D), seed=3, dtype=torch.float32)
    o = ops.attention(q.cuda(), kv[0], kv[1])
    torch.cuda.synchronize()
    ro, _ = oracle.attn_fwd(q.numpy(), *(t.contiguous().cpu().numpy() for t in kv), oracle.F32)
    assert np.abs(o.cpu().numpy() - ro).max() <= TOL_F32_REL * np.abs(ro).max()
