"""GPU parity of the lazy softmax rescale under scores that climb block by block.

Random inputs keep every key block's scores near the running max, so the
kernels' rescale paths run on the first block only. Here the keys are
built so that, against q of all ones, the log2-domain scores step through:
  blocks 0-3    around 0
  block 4       +12: the block max passes m + 8, so m moves and O, l rescale
  blocks 5-7    back to 0
  block 8       +242: 2^(s - m) against the old m overflows fp32 to inf
  blocks 9-11   +239
  block 12      +248 on every other key: p = 2^6 each, so a lane's sum
                passes 2^8 while no p does (the max is formed, m stays)
  blocks 13-    +239
Prefill (bf16, f16 and fp32) and split-K decode (bf16 and fp8 KV, splits that
start inside the ramp) are checked against the CPU oracle, which takes the plain
running max. The prefill launches are such that one chain of key blocks holds
the whole ramp: a launch that fills the GPU, one cut into splits of 16 key
blocks or more, and one whose halves of the keys go to four waves each (32 key
blocks, without a workspace); 1024 keys of two heads are cut into splits of two
key blocks, each of which starts inside the ramp.
"""

import ctypes

import numpy as np
import pytest
import torch

import oracle
from helpers import TOL_BF16_ABS, TOL_FP8_ABS, TOL_LSE_ABS, bits, max_abs, oracle_dtype, to_f32
from neptune_hip import _abi
from test_gpu_attention_large import check_heads

pytestmark = pytest.mark.gpu

D = 128
LOG2_PER_UNIT = D * 1.4426950408889634 / D ** 0.5  # log2 score of q = 1, k = 1 per element


@pytest.fixture(scope="module")
def ops():
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    from neptune_hip import ops as _ops
    return _ops


def _log(msg):
    print(msg, flush=True)


def ramp_targets(L):
    """log2-domain score of each key against q = 1 (see the module text)."""
    j = torch.arange(L)
    blk = j // 64
    t = torch.zeros(L)
    t[blk == 4] = 12.0
    t[blk >= 8] = 239.0
    t[blk == 8] = 242.0
    t[(blk == 12) & (j % 2 == 0)] = 248.0
    return t


def ramp_kv(B, H, L, seed, dtype, dim=D):
    g = torch.Generator().manual_seed(seed)
    base = (ramp_targets(L) / (LOG2_PER_UNIT * (dim / D) ** 0.5)).view(1, 1, L, 1)
    k = base + 0.05 * torch.randn((B, H, L, dim), generator=g)
    v = torch.randn((B, H, L, dim), generator=g)
    return k.to(dtype), v.to(dtype)


def ramp_q(shape, seed, dtype):
    g = torch.Generator().manual_seed(seed)
    return (1.0 + 0.02 * torch.randn(shape, generator=g)).to(dtype)


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_prefill_climbing_scores(ops, causal, dtype):
    _log(f"case: prefill climbing scores causal={causal} dtype={dtype}")
    B, H, S = 1, 2, 1024
    q = ramp_q((B, H, S, D), 1, dtype)
    k, v = ramp_kv(B, H, S, 2, dtype)
    o, lse = ops.attention(q.cuda(), k.cuda(), v.cuda(), causal=causal, return_lse=True)
    torch.cuda.synchronize()
    ro, rl = oracle.attn_fwd(bits(q), bits(k), bits(v), oracle_dtype(q), causal)
    ref = oracle.decode(ro, oracle_dtype(q))
    got = to_f32(o)
    assert np.isfinite(got).all()
    assert max_abs(got, ref) <= TOL_BF16_ABS * max(1.0, np.abs(ref).max())
    assert max_abs(to_f32(lse), rl) <= TOL_LSE_ABS


@pytest.mark.parametrize("form,B,Hq,Hk,Sq,Sk,dim", [
    ("whole", 4, 32, 32, 1024, 1024, 128),
    ("whole", 8, 16, 16, 1024, 1024, 64),
    ("splits", 1, 32, 8, 250, 8000, 128),
    ("splits", 2, 32, 8, 250, 8000, 64),
    ("halves", 1, 2, 2, 2048, 2048, 128),
    ("halves", 1, 2, 2, 2048, 2048, 64),
])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_prefill_forms_climbing_scores(ops, form, B, Hq, Hk, Sq, Sk, dim, causal, dtype):
    _log(f"case: prefill {form} climbing scores B={B} {Hq}/{Hk} {Sq}x{Sk} D={dim} "
         f"causal={causal} dtype={dtype}")
    q = ramp_q((B, Hq, Sq, dim), 7, dtype).cuda()
    k, v = (t.cuda() for t in ramp_kv(B, Hk, Sk, 8, dtype, dim))
    lib = _abi.load_library()
    d, n = _abi.AttnDesc(), ctypes.c_size_t()
    d.batch, d.heads_q, d.heads_kv, d.seq_q, d.seq_kv, d.head_dim = B, Hq, Hk, Sq, Sk, dim
    d.dtype = _abi.DTYPE_BF16 if dtype == torch.bfloat16 else _abi.DTYPE_F16
    d.causal = int(causal)
    _abi.check(lib.neptune_attn_workspace_bytes(ctypes.byref(d), ctypes.byref(n)), lib)
    if form == "splits":  # at most Sk / 1024 of them, so 16 key blocks or more in each
        assert 0 < n.value <= B * Hq * Sq * (Sk // 1024 + 1) * (dim + 2) * 4
    elif form == "whole":
        assert n.value == 0
    if form == "halves":
        o = torch.empty_like(q)
        lse = torch.empty((B, Hq, Sq), device="cuda")
        _abi.check(lib.neptune_attn_fwd(ctypes.byref(d), q.data_ptr(), k.data_ptr(), v.data_ptr(),
                                        o.data_ptr(), lse.data_ptr(),
                                        torch.cuda.current_stream().cuda_stream), lib)
    else:
        o, lse = ops.attention(q, k, v, causal=causal, return_lse=True)
    check_heads(q, k, v, o, lse, causal)


@pytest.mark.parametrize("B,H,S", [(4, 32, 1024), (1, 2, 2048)], ids=["four_waves", "eight_waves"])
@pytest.mark.parametrize("dim", [32, 64, 128])
@pytest.mark.parametrize("causal", [False, True])
def test_fp32_climbing_scores(ops, B, H, S, dim, causal):
    """Scores of 248 (log2 units) come from sums of up to 128 products, each
    rounded, in the kernel and in the oracle: 2^-24 sqrt(128) of them, which p
    takes times ln 2: 1.2e-4 each."""
    _log(f"case: fp32 climbing scores B={B} H={H} S={S} D={dim} causal={causal}")
    q = ramp_q((B, H, S, dim), 9, torch.float32).cuda()
    k, v = (t.cuda() for t in ramp_kv(B, H, S, 10, torch.float32, dim))
    o, lse = ops.attention(q, k, v, causal=causal, return_lse=True)
    for b, h in ((0, 0), (B - 1, H - 1)):
        qq, kk, vv = (t[b, h][None, None].cpu() for t in (q, k, v))
        ro, rl = oracle.attn_fwd(bits(qq), bits(kk), bits(vv), oracle.F32, causal)
        ref = oracle.decode(ro, oracle.F32)[0, 0]
        got = to_f32(o[b, h])
        assert np.isfinite(got).all()
        assert max_abs(got, ref) <= 2.4e-4 * np.abs(ref).max()
        assert max_abs(to_f32(lse[b, h]), rl[0, 0]) <= TOL_LSE_ABS


@pytest.mark.parametrize("splits", [1, 3])
def test_decode_bf16_climbing_scores(ops, splits):
    _log(f"case: decode bf16 climbing scores splits={splits}")
    B, Hq, Hk, L = 2, 8, 2, 1024
    q = ramp_q((B, Hq, D), 3, torch.bfloat16)
    k, v = ramp_kv(B, Hk, L, 4, torch.bfloat16)
    o, lse = ops.decode_splitk(q.cuda(), k.cuda(), v.cuda(), num_splits=splits, return_lse=True)
    torch.cuda.synchronize()
    ro, rl, _ = oracle.decode_splitk(bits(q), bits(k), bits(v), oracle.BF16, num_splits=splits)
    ref = oracle.decode(ro, oracle.BF16)
    got = to_f32(o)
    assert np.isfinite(got).all()
    assert max_abs(got, ref) <= TOL_BF16_ABS * max(1.0, np.abs(ref).max())
    assert max_abs(to_f32(lse), rl) <= TOL_LSE_ABS


@pytest.mark.parametrize("splits", [1, 3])
def test_decode_fp8_climbing_scores(ops, splits):
    _log(f"case: decode fp8 climbing scores splits={splits}")
    B, Hq, Hk, L = 2, 8, 2, 1024
    q = ramp_q((B, Hq, D), 5, torch.bfloat16)
    k, v = ramp_kv(B, Hk, L, 6, torch.bfloat16)
    kc, ks = ops.kv_quantize_fp8(k.cuda())
    vc, vs = ops.kv_quantize_fp8(v.cuda())
    o, lse = ops.decode_splitk(q.cuda(), kc, vc, k_scale=ks, v_scale=vs, num_splits=splits,
                               return_lse=True)
    torch.cuda.synchronize()
    ro, rl, _ = oracle.decode_splitk(bits(q), kc.cpu().numpy(), vc.cpu().numpy(), oracle.FP8,
                                     ks.cpu().numpy(), vs.cpu().numpy(), num_splits=splits)
    ref = oracle.decode(ro, oracle.BF16)
    got = to_f32(o)
    assert np.isfinite(got).all()
    assert max_abs(got, ref) <= TOL_FP8_ABS * max(1.0, np.abs(ref).max())
    assert max_abs(to_f32(lse), rl) <= TOL_LSE_ABS


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("B,Hk,L", [
    (70, 8, 1024),   # 560 work-groups: one wave
    (40, 8, 2048),   # 320: two waves (bf16; fp8 four, of which one holds half the ramp)
    (2, 2, 4096),    # four
], ids=["one_wave", "two_waves", "four_waves"])
def test_decode_chains_climbing_scores(ops, B, Hk, L, fp8):
    """One split, whose first wave's chain holds the whole ramp (1024 keys)."""
    _log(f"case: decode chains climbing scores B={B} Hk={Hk} L={L} fp8={fp8}")
    q = ramp_q((B, 4 * Hk, D), 11, torch.bfloat16)
    k, v = (t.repeat(B, 1, 1, 1) for t in ramp_kv(1, Hk, L, 12, torch.bfloat16))
    if fp8:
        (kc, ks), (vc, vs) = (ops.kv_quantize_fp8(t.cuda()) for t in (k, v))
        o, lse = ops.decode_splitk(q.cuda(), kc, vc, k_scale=ks, v_scale=vs, num_splits=1,
                                   return_lse=True)
    else:
        o, lse = ops.decode_splitk(q.cuda(), k.cuda(), v.cuda(), num_splits=1, return_lse=True)
    torch.cuda.synchronize()
    for b in (0, B - 1):
        one = slice(b, b + 1)
        if fp8:
            kv = [t[one].contiguous().cpu().numpy() for t in (kc, vc, ks, vs)]
            ro, rl, _ = oracle.decode_splitk(bits(q[one]), kv[0], kv[1], oracle.FP8, kv[2], kv[3],
                                             num_splits=1)
        else:
            ro, rl, _ = oracle.decode_splitk(bits(q[one]), bits(k[one]), bits(v[one]), oracle.BF16,
                                             num_splits=1)
        ref, got = oracle.decode(ro, oracle.BF16), to_f32(o[one])
        assert np.isfinite(got).all()
        assert max_abs(got, ref) <= (TOL_FP8_ABS if fp8 else TOL_BF16_ABS) * max(1.0, np.abs(ref).max())
        assert max_abs(to_f32(lse[one]), rl) <= TOL_LSE_ABS
