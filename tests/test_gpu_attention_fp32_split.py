"""The fp32 attention kernel's two splits of the work (16-row work-groups of
eight waves, 32-row ones of four) at their edges, and its element-wise form
for tensors that 16-byte loads cannot read, against the oracle at the fp32
contract (1e-5 relative, LSE included)."""

import numpy as np
import pytest
import torch

import oracle
from helpers import TOL_F32_REL, randn

pytestmark = pytest.mark.gpu


def _check(o, lse, q, k, v, causal):
    ro, rl = oracle.attn_fwd(q.numpy(), k.numpy(), v.numpy(), oracle.F32, causal=causal)
    o, lse = o.cpu().numpy(), lse.cpu().numpy()
    assert np.abs(o - ro).max() <= TOL_F32_REL * np.abs(ro).max()
    assert np.array_equal(np.isneginf(lse), np.isneginf(rl))
    fin = np.isfinite(rl)
    assert np.abs(lse[fin] - rl[fin]).max() <= TOL_F32_REL * max(1.0, np.abs(rl[fin]).max())


@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize("B,Hq,Hk,Sq,Sk,causal", [
    (8, 32, 8, 33, 65, False),    # 512 blocks of 32 rows: one row and one key past a block
    (8, 32, 8, 33, 65, True),     # the causal line
    (8, 16, 16, 64, 7, True),     # fewer keys than one block, rows with no visible key
    (1, 2, 1, 17, 129, False),    # 16-row groups: one row past a block, keys for every wave
    (1, 3, 3, 15, 16, True),      # one partial row block, one key block
    (2, 1, 1, 1, 1, True),        # one query, one key
])
def test_fp32_splits(B, Hq, Hk, Sq, Sk, causal, D):
    from neptune_hip import ops
    print(f"case: fp32 split B={B} Hq={Hq} Hk={Hk} Sq={Sq} Sk={Sk} D={D} causal={causal}",
          flush=True)
    q = randn((B, Hq, Sq, D), seed=1, dtype=torch.float32)
    k, v = (randn((B, Hk, Sk, D), seed=s, dtype=torch.float32) for s in (2, 3))
    o, lse = ops.attention(q.cuda(), k.cuda(), v.cuda(), causal=causal, return_lse=True)
    torch.cuda.synchronize()
    _check(o, lse, q, k, v, causal)


@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize("B,H,Sq,Sk", [(1, 2, 20, 50), (8, 32, 40, 70)])
@pytest.mark.parametrize("what", ["row stride", "base"])
def test_fp32_unaligned(B, H, Sq, Sk, D, what):
    """Rows D + 1 floats apart, or a base 4 bytes past a 16-byte boundary."""
    from neptune_hip import ops
    print(f"case: fp32 unaligned {what} B={B} H={H} Sq={Sq} Sk={Sk} D={D}", flush=True)
    q = randn((B, H, Sq, D), seed=4, dtype=torch.float32)
    k, v = (randn((B, H, Sk, D), seed=s, dtype=torch.float32) for s in (5, 6))

    def place(t):
        if what == "base":
            buf = torch.full((t.numel() + 1,), float("nan"), device="cuda")
            view = buf[1:].view(t.shape)
        else:
            view = torch.full(t.shape[:-1] + (D + 1,), float("nan"), device="cuda")[..., :D]
        return view.copy_(t)

    out = place(torch.zeros_like(q))
    o, lse = ops.attention(place(q), place(k), place(v), causal=True, return_lse=True, out=out)
    torch.cuda.synchronize()
    _check(o.contiguous(), lse, q, k, v, True)
