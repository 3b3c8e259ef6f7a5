"""Decode launches short of work-groups (two or four waves share a split), the
combine of many splits (groups of threads share them out) and ragged paged batches (splits scaled to each sequence, sequences taken longest
first), at their edges against the oracle at the decode contract."""

import numpy as np
import pytest
import torch

import oracle
from helpers import TOL_BF16_ABS, TOL_BF16_REL, TOL_FP8_ABS, assert_rel_rows, bits, max_abs, randn, to_f32
from neptune_hip import ops

pytestmark = pytest.mark.gpu


def _check(o, lse, ro, rl, fp8, what):
    ref = oracle.decode(ro, oracle.BF16)
    assert max_abs(to_f32(o), ref) <= (TOL_FP8_ABS if fp8 else TOL_BF16_ABS)
    assert_rel_rows(to_f32(o), ref, TOL_BF16_REL, what)
    lse = to_f32(lse)
    assert np.array_equal(np.isneginf(lse), np.isneginf(rl))
    fin = np.isfinite(rl)
    assert np.abs(lse[fin] - rl[fin]).max() <= 1e-3


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("B,Hq,Hk,L,splits", [
    (1, 4, 1, 1, 1),        # one token for four waves
    (1, 16, 1, 33, 1),      # two waves' worth, the second one token
    (2, 8, 2, 250, 1),      # four waves, the last one short
    (1, 8, 2, 4100, 0),     # the last split four tokens
    (1, 8, 8, 2500, 38),    # 304 work-groups: two waves (bf16)
    (2, 8, 8, 2100, 33),    # 528 work-groups: one wave
])
def test_waves_per_split(B, Hq, Hk, L, splits, fp8):
    print(f"case: decode waves B={B} Hq={Hq} Hk={Hk} L={L} splits={splits} fp8={fp8}", flush=True)
    q = randn((B, Hq, 128), seed=1)
    k, v = (randn((B, Hk, L, 128), seed=s) for s in (2, 3))
    if fp8:
        (kc, ks), (vc, vs) = (ops.kv_quantize_fp8(t.cuda()) for t in (k, v))
        o, lse = ops.decode_splitk(q.cuda(), kc, vc, k_scale=ks, v_scale=vs, num_splits=splits,
                                   return_lse=True)
        torch.cuda.synchronize()
        ro, rl, _ = oracle.decode_splitk(bits(q), kc.cpu().numpy(), vc.cpu().numpy(), oracle.FP8,
                                         ks.cpu().numpy(), vs.cpu().numpy(), num_splits=splits)
    else:
        o, lse = ops.decode_splitk(q.cuda(), k.cuda(), v.cuda(), num_splits=splits, return_lse=True)
        torch.cuda.synchronize()
        ro, rl, _ = oracle.decode_splitk(bits(q), bits(k), bits(v), oracle.BF16, num_splits=splits)
    _check(o, lse, ro, rl, fp8, "waves per split")


@pytest.mark.parametrize("splits", [16, 17, 32, 33, 64, 65, 128, 129])
def test_combine_thread_groups(splits):
    """Split counts around those where the combine takes more thread groups,
    every split one or two 64-token blocks."""
    print(f"case: combine splits={splits}", flush=True)
    L = splits * 64 - 5
    q = randn((1, 8, 128), seed=8)
    k, v = (randn((1, 2, L, 128), seed=s) for s in (9, 10))
    o, lse = ops.decode_splitk(q.cuda(), k.cuda(), v.cuda(), num_splits=splits, return_lse=True)
    torch.cuda.synchronize()
    ro, rl, _ = oracle.decode_splitk(bits(q), bits(k), bits(v), oracle.BF16, num_splits=splits)
    _check(o, lse, ro, rl, False, "combine thread groups")


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("Hk,L,splits,lens", [
    (2, 1200, 2, [1200, 0, 1, 64, 65, 700, 700, 31, 1199]),   # sorted, scaled, ties, empty
    (1, 640, 1, [(97 * i) % 641 for i in range(64)]),         # 64 sequences: every lane
    (1, 600, 1, [(89 * i) % 601 for i in range(65)]),         # one more: not sorted
    (4, 1100, 2, [1100] * 6),                                 # all the same
    (8, 300, 5, [(31 * i) % 301 for i in range(33)]),         # 1320 short work-groups: scaled only
])
def test_ragged_paged(Hk, L, splits, lens, fp8):
    print(f"case: ragged paged Hk={Hk} L={L} splits={splits} B={len(lens)} fp8={fp8}", flush=True)
    B, Hq, ps = len(lens), 2 * Hk, 64
    per = -(-L // ps)
    q = randn((B, Hq, 128), seed=4)
    kp, vp = (randn((B * per, Hk, ps, 128), seed=s) for s in (5, 6))
    scales, host = {}, {}
    if fp8:
        pools = []
        for name, pool in (("k_scales", kp), ("v_scales", vp)):
            c, s = ops.kv_quantize_fp8(pool.cuda(), scale_block=ps)
            pools.append(c)
            scales[name] = s[..., 0].contiguous()
            host[name] = scales[name].cpu().numpy()
    else:
        pools = [kp.cuda(), vp.cuda()]
    table = torch.from_numpy(np.random.default_rng(7).permutation(B * per).astype(np.int32))
    table = table.view(B, per)
    sl = torch.tensor(lens, dtype=torch.int32)
    o, lse = ops.decode_paged(q.cuda(), *pools, table.cuda(), sl.cuda(), max_seq_len=L,
                              num_splits=splits, return_lse=True, **scales)
    torch.cuda.synchronize()
    pool_np = [p.cpu().numpy() if fp8 else bits(p) for p in pools]
    ro, rl = oracle.decode_paged(bits(q), *pool_np, table.numpy(), sl.numpy(), max_seq_len=L,
                                 num_splits=splits, **host)
    _check(o, lse, ro, rl, fp8, "ragged paged")
