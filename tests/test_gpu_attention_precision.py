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


@pytest.mark.parametrize("B,H,D", [(2, 4, 32), (2, 4, 64), (1, 1, 32)])
def test_fp32_sums_stay_short(B, H, D):
    """fp32 over 2048 keys, no mask: four waves a row block (eight with one
    head), so 512 (256) keys a wave. A sum of n rounded additions whose partial
    sums grow as a random walk is off by u sqrt(n / 2), u = 2^-23 / sqrt(12) *
    0.74 (a half ulp's spread over a binade). Beyond the error at 128 keys (a
    block or two a wave) the long rows may show that of n = 128 terms, plus 10%."""
    from neptune_hip import ops
    print(f"case: fp32 sums B={B} H={H} D={D}", flush=True)
    q, k, v = (randn((B, H, 2048, D), seed=s, dtype=torch.float32).cuda() for s in (4, 5, 6))
    err = {}
    for n in (128, 2048):
        kn, vn = k[:, :, :n].contiguous(), v[:, :, :n].contiguous()
        exact, _ = _exact_and_htile(q, kn, vn, False)
        err[n] = _rel(ops.attention(q, kn, vn), exact)
    chain = 2.0 ** -23 / math.sqrt(12) * 0.74 * math.sqrt(128 / 2)
    print(f"  error against 64 bits {err}, sums of 128 terms {chain:.2e}", flush=True)
    assert err[2048] <= 1.1 * math.hypot(err[128], chain)


def test_fp32_lse_rounds_three_times():
    """fp32 log-sum-exps of 2048 keys, around 8: an rms error of the spacing of
    floats over sqrt(12) for the result (2^-20 from 8 on) and for the one term of
    4 to 8 in it (2^-21), 3.1e-7 together, and 15% more for the sums."""
    from neptune_hip import ops
    print("case: fp32 lse", flush=True)
    q, k, v = (randn((2, 4, 2048, 64), seed=s, dtype=torch.float32).cuda() for s in (7, 8, 9))
    _, lse = ops.attention(q, k, v, return_lse=True)
    ref = torch.stack([torch.logsumexp(
        torch.matmul(q[b, h].double(), k[b, h].double().t().contiguous()) / 8.0, -1)
        for b in range(2) for h in range(4)]).view(2, 4, 2048)
    rms = float((lse.double() - ref).pow(2).mean().sqrt())
    print(f"  rms error {rms:.3e}", flush=True)
    assert rms <= 1.15 * math.hypot(2.0 ** -20, 2.0 ** -21) / math.sqrt(12)
