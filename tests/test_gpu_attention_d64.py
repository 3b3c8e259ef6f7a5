"""The head_dim-64 16-bit attention kernel at the edges of its 128-row query
blocks and 64-key blocks, its running max where scores climb, and K / V whose
64-row tiles span more than 4 GiB, against the oracle at the 16-bit contract."""

import numpy as np
import pytest
import torch

import oracle
from helpers import TOL_BF16_ABS, TOL_LSE_ABS, bits, max_abs, oracle_dtype, randn, to_f32

pytestmark = pytest.mark.gpu


def _check(ops, q, k, v, causal, dev=None):
    dq, dk, dv = dev or (t.cuda() for t in (q, k, v))
    o, lse = ops.attention(dq, dk, dv, causal=causal, return_lse=True)
    torch.cuda.synchronize()
    ro, rl = oracle.attn_fwd(bits(q), bits(k), bits(v), oracle_dtype(q), causal)
    assert max_abs(to_f32(o), oracle.decode(ro, oracle_dtype(q))) <= TOL_BF16_ABS
    lse = to_f32(lse)
    assert np.array_equal(np.isneginf(lse), np.isneginf(rl))
    fin = np.isfinite(rl)
    assert np.abs(lse[fin] - rl[fin]).max() <= TOL_LSE_ABS


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("Hq,Hk,Sq,Sk,causal", [
    (4, 1, 1, 1, True), (8, 2, 1, 65, False), (2, 2, 127, 63, True), (2, 1, 129, 64, False),
    (3, 3, 128, 129, True), (2, 2, 257, 200, True), (4, 2, 33, 321, True),
])
def test_d64_edges(Hq, Hk, Sq, Sk, causal, dtype):
    from neptune_hip import ops
    print(f"case: d64 edge Hq={Hq} Hk={Hk} Sq={Sq} Sk={Sk} causal={causal} {dtype}", flush=True)
    q = randn((2, Hq, Sq, 64), seed=1, dtype=dtype, scale=0.5)
    k, v = (randn((2, Hk, Sk, 64), seed=s, dtype=dtype, scale=0.5) for s in (2, 3))
    _check(ops, q, k, v, causal)


@pytest.mark.parametrize("step", [0.25, 2.0, 40.0])
def test_d64_climbing_scores(step):
    """Keys grow along the sequence, so block maxima pass the running max: by
    less than the slack, past it, and past fp32's range of exponents."""
    from neptune_hip import ops
    print(f"case: d64 climb step={step}", flush=True)
    q = randn((1, 2, 140, 64), seed=4, scale=0.5).abs()
    ramp = (1.0 + step * (torch.arange(300) // 64).float())[None, None, :, None]
    k = (randn((1, 2, 300, 64), seed=5, scale=0.5).abs().float() * ramp).to(torch.bfloat16)
    v = randn((1, 2, 300, 64), seed=6, scale=0.5)
    for causal in (False, True):
        _check(ops, q, k, v, causal)


def test_d64_tiles_past_4_gib():
    """Key rows 70 MiB apart: a 64-row tile spans more than 32-bit offsets."""
    from neptune_hip import ops
    rows, stride = 66, 35 << 20
    print(f"case: d64 row stride {stride} elements, {rows} keys", flush=True)
    q = randn((1, 1, 70, 64), seed=7, scale=0.5)
    k, v = (randn((1, 1, rows, 64), seed=s, scale=0.5) for s in (8, 9))
    buf = torch.empty(rows * stride, dtype=torch.bfloat16, device="cuda")
    views = [buf[off:].as_strided((1, 1, rows, 64), (rows * stride, rows * stride, stride, 1))
             for off in (0, 64)]
    dk, dv = (view.copy_(t) for view, t in zip(views, (k, v)))
    _check(ops, q, k, v, True, (q.cuda(), dk, dv))
