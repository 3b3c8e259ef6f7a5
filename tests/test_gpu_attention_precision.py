"""Rounding of the attention kernels against 64 bits: no more than the forms
they stand for show on the same inputs."""

import math

import pytest
import torch

from helpers import randn

pytestmark = pytest.mark.gpu


def _rel(got, ref):
    return float((got.double() - ref).norm() / ref.norm())


def _exact_and_htile(q, k, v, causal):
    """softmax(q k^T / sqrt(D)) v in float64; and the same with the HTile
    program's two roundings alone (HTile:92-143): P to the input type against
    the running max of each 64-key block, O on store."""
    exact, rounded = torch.empty_like(q, dtype=torch.float64), torch.empty_like(q)
    Sq, Sk, D = q.shape[2], k.shape[2], q.shape[3]
    hidden = torch.ones((Sq, Sk), dtype=torch.bool, device=q.device).tril(Sk - Sq).logical_not()
    for b in range(q.shape[0]):
        for h in range(q.shape[1]):
            s = torch.matmul(q[b, h].double(), k[b, h].double().t().contiguous())
            s *= math.log2(math.e) / math.sqrt(D)
            if causal:
                s.masked_fill_(hidden, -math.inf)
            w = v[b, h].double()
            p = torch.exp2(s - s.amax(-1, keepdim=True))
            exact[b, h] = torch.matmul(p, w) / p.sum(-1, keepdim=True)
            m = torch.full((Sq, 1), -math.inf, dtype=torch.float64, device=q.device)
            l, o = torch.zeros_like(m), torch.zeros_like(w[:1]).expand(Sq, D)
            for k0 in range(0, Sk, 64):
                m_new = torch.maximum(m, s[:, k0:k0 + 64].amax(-1, keepdim=True))
                p = torch.exp2(s[:, k0:k0 + 64] - m_new)
                alpha = torch.exp2(m - m_new)
                l = l * alpha + p.sum(-1, keepdim=True)
                o = o * alpha + torch.matmul(p.to(q.dtype).double(), w[k0:k0 + 64])
                m = m_new
            rounded[b, h] = (o / l).to(q.dtype)
    return exact, rounded


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("B,H,S,causal", [(8, 16, 300, False), (4, 16, 1024, True)])
def test_d64_rounds_no_more_than_the_tile_program(B, H, S, causal, dtype):
    """N(0, 1) inputs, where a row's largest p weighs most. The kernel's fp32
    arithmetic (about 1e-6 of a p) turns at most a p in some 500 (f16) to the
    other side of its rounding, so its error is the emulation's within 1%.
    A max that lags behind rounds the largest p too: 3% to 6% more."""
    from neptune_hip import ops
    print(f"case: d64 rounding B={B} H={H} S={S} causal={causal} {dtype}", flush=True)
    q, k, v = (randn((B, H, S, 64), seed=s, dtype=dtype).cuda() for s in (1, 2, 3))
    got = ops.attention(q, k, v, causal=causal)
    exact, rounded = _exact_and_htile(q, k, v, causal)
    e, limit = _rel(got, exact), _rel(rounded, exact)
    print(f"  error against 64 bits {e:.4e}, the tile program's {limit:.4e}", flush=True)
    assert e <= 1.01 * limit
