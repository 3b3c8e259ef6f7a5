"""The head_dim-128 kernel of launches that fill the GPU (more than 512 blocks
of 128 query rows; shorter ones are cut or run in single blocks by another
kernel): pairs of query blocks without the mask, an odd block left over, ragged
ends, grouped heads and the stage counts. Checked bit for bit between stage
counts and, on some heads, against the oracle."""

import numpy as np
import pytest
import torch

import oracle
from helpers import TOL_BF16_ABS, TOL_LSE_ABS, bits, max_abs, oracle_dtype, randn, to_f32

pytestmark = pytest.mark.gpu

SHAPES = [  # B, Hq, Hk, Sq, Sk
    (4, 32, 8, 600, 611),    # five blocks: one left over from the pairs; ragged keys
    (4, 32, 8, 641, 130),    # a last block of one row; fewer keys than queries
    (4, 32, 32, 704, 832),   # six blocks; whole key blocks
    (8, 32, 4, 300, 63),     # less than a key block
]


def check_heads(q, k, v, o, lse, causal, heads=((0, 0), (-1, -1))):
    """o and lse of the given (batch row, query head)s against the oracle."""
    group = q.shape[1] // k.shape[1]
    for b, h in heads:
        h %= q.shape[1]
        qq = q[b, h][None, None].cpu()
        kk, vv = (t[b, h // group][None, None].cpu() for t in (k, v))
        ro, rl = oracle.attn_fwd(bits(qq), bits(kk), bits(vv), oracle_dtype(qq), causal)
        ref = oracle.decode(ro, oracle_dtype(qq))
        got, got_lse = to_f32(o[b, h])[None, None], to_f32(lse[b, h])[None, None]
        assert np.isfinite(got).all()
        assert max_abs(got, ref) <= TOL_BF16_ABS * max(1.0, np.abs(ref).max())
        assert np.array_equal(np.isneginf(got_lse), np.isneginf(rl))
        fin = np.isfinite(rl)
        assert max_abs(got_lse[fin], rl[fin]) <= TOL_LSE_ABS


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_full_launches(shape, causal, dtype):
    from neptune_hip import ops
    B, Hq, Hk, Sq, Sk = shape
    print(f"case: d128 full launch {shape} causal={causal} {dtype}", flush=True)
    assert -(-Sq // 128) * Hq * B > 512
    q = randn((B, Hq, Sq, 128), seed=1, dtype=dtype, scale=0.5).cuda()
    k, v = (randn((B, Hk, Sk, 128), seed=s, dtype=dtype, scale=0.5).cuda() for s in (2, 3))
    o, lse = ops.attention(q, k, v, causal=causal, return_lse=True)
    check_heads(q, k, v, o, lse, causal)
    for stages in (1, 2, 3):
        so, sl = ops.attention(q, k, v, causal=causal, return_lse=True, pipeline_stages=stages)
        assert torch.equal(so.view(torch.int16), o.view(torch.int16)), stages
        assert torch.equal(sl, lse), stages
