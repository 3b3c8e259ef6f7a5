"""Rounding of fp8 decode against 64 bits."""

import math

import pytest
import torch

from helpers import randn

pytestmark = pytest.mark.gpu


def _error(B, Hq, Hk, L, splits, v_scale):
    """Relative error against float64 on the same codes, V scaled by v_scale."""
    from neptune_hip import ops
    q = randn((B, Hq, 128), seed=1).cuda()
    k, v = (randn((B, Hk, L, 128), seed=s, dtype=torch.float32).clamp(-4, 4).mul_(100)
            .to(torch.float8_e4m3fn).cuda() for s in (2, 3))
    ks, vs = (torch.full((B, Hk, -(-L // 64)), s, device="cuda") for s in (0.01, v_scale))
    got = ops.decode_splitk(q, k, v, k_scale=ks, v_scale=vs, num_splits=splits)
    ref = torch.empty(got.shape, dtype=torch.float64, device="cuda")
    for b in range(B):
        for h in range(Hq):
            kk, vv = (t[b, h // (Hq // Hk)].double() for t in (k, v))
            p = torch.softmax(torch.matmul(kk, q[b, h].double()) * (ks[0, 0, 0].double() /
                                                                    math.sqrt(128)), 0)
            ref[b, h] = torch.matmul(p, vv) * vs[0, 0, 0].double()
    return float((got.double() - ref).norm() / ref.norm())


@pytest.mark.parametrize("B,Hq,Hk,L,splits", [(16, 32, 8, 250, 0), (16, 8, 1, 3000, 16),
                                              (4, 32, 8, 2048, 1)])
def test_fp8_value_scale_takes_no_precision(B, Hq, Hk, L, splits):
    """P times V's scale is rounded to bf16. A scale of 1.114 / 128, what N(0, 1)
    data get, must round no worse than 1 / 128, where every wave's largest p is a
    power of two: the products' mantissas are the same, so what differs is the
    rounding of the outputs. An rms over n of them has a standard deviation of
    1 / sqrt(2 n), 0.55% at the 16384 outputs of each launch; three of the two
    errors' difference (0.8%) is the 3% allowed."""
    print(f"case: fp8 value scale B={B} Hq={Hq} Hk={Hk} L={L} splits={splits}", flush=True)
    one, other = (_error(B, Hq, Hk, L, splits, s / 128) for s in (1.0, 1.114))
    print(f"  error at scale 1 / 128 {one:.4e}, at 1.114 / 128 {other:.4e}", flush=True)
    assert other <= 1.03 * one
