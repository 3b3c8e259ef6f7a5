"""Calls whose tensors differ only in strides, dtype or options, taken in turn:
each has to get its own checks and descriptor."""

import pytest
import torch

from helpers import randn
from neptune_hip import ops

pytestmark = pytest.mark.gpu


def test_attention_calls_in_turn():
    print("case: attention calls in turn", flush=True)
    q, k, v = (randn((2, 4, 96, 64), seed=s).cuda() for s in (1, 2, 3))
    ref = {(c, sc): ops.attention(q.clone(), k.clone(), v.clone(), causal=c, scale=sc)
           for c in (False, True) for sc in (None, 0.5)}
    wide = torch.zeros((2, 4, 96, 72), dtype=q.dtype, device="cuda")
    qs = wide[..., :64].copy_(q)
    heads_last = torch.empty((2, 96, 4, 64), dtype=q.dtype, device="cuda").transpose(1, 2)
    ks = heads_last.copy_(k)
    out = torch.zeros((2, 4, 96, 80), dtype=q.dtype, device="cuda")[..., :64]
    for _ in range(2):
        for (c, sc), want in ref.items():
            for qq, kk, oo in ((q, k, None), (qs, k, None), (q, ks, out), (qs, ks, None)):
                got, lse = ops.attention(qq, kk, v, causal=c, scale=sc, out=oo, return_lse=True)
                assert torch.equal(got, want) and lse.shape == (2, 4, 96)
        with pytest.raises(ValueError, match="share one of"):
            ops.attention(q, k.half(), v)
        with pytest.raises(ValueError, match="device tensors"):
            ops.attention(q, k.cpu(), v)
        f = [t.float() for t in (q, k, v)]
        assert ops.attention(*f).dtype == torch.float32


def test_decode_and_scan_calls_in_turn():
    print("case: decode and scan calls in turn", flush=True)
    q = randn((2, 8, 128), seed=4).cuda()
    k, v = (randn((2, 2, 500, 128), seed=s).cuda() for s in (5, 6))
    (kc, ks), (vc, vs) = (ops.kv_quantize_fp8(t) for t in (k, v))
    small = torch.empty(16, dtype=torch.uint8, device="cuda")
    want = {n: ops.decode_splitk(q, k, v, num_splits=n) for n in (0, 1, 4)}
    want8 = ops.decode_splitk(q, kc, vc, k_scale=ks, v_scale=vs)
    for _ in range(2):
        for n, w in want.items():
            assert torch.equal(ops.decode_splitk(q, k, v, num_splits=n), w)
        assert torch.equal(ops.decode_splitk(q[:, :, None], kc, vc, k_scale=ks, v_scale=vs), want8)
        with pytest.raises(ValueError, match="need"):
            ops.decode_splitk(q, k, v, workspace=small)
        with pytest.raises(ValueError, match="contiguous"):
            ops.decode_splitk(q, k.transpose(2, 3).contiguous().transpose(2, 3), v)
    u, dr, z = (randn((1, 32, 64), seed=s).cuda() for s in (7, 8, 9))
    Bm, Cm = (randn((1, 16, 64), seed=s).cuda() for s in (10, 11))
    A = -torch.exp(randn((32, 16), seed=12, dtype=torch.float32)).cuda()
    y = {g: ops.selective_scan(u, dr, A, Bm, Cm, None, z if g else None, None) for g in (0, 1)}
    for _ in range(2):
        for g in (0, 1):
            assert torch.equal(ops.selective_scan(u, dr, A, Bm, Cm, None, z if g else None), y[g])
        off = ops.selective_scan(u, dr.abs(), A, Bm, Cm, delta_softplus=False)
        assert not torch.equal(off, y[0])
