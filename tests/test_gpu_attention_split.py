"""Short 16-bit attention launches: keys cut into splits (neptune_attn_fwd_ws),
query heads of a KV head packed into shared row blocks, and both, at their
edges against the oracle at the 16-bit contract; the same calls without a
workspace; and the workspace's size checks. The workspace starts as NaN, so a
state read without having been written shows."""

import ctypes

import numpy as np
import pytest
import torch

import oracle
from helpers import TOL_BF16_ABS, TOL_LSE_ABS, bits, max_abs, oracle_dtype, randn, to_f32
from neptune_hip import _abi

pytestmark = pytest.mark.gpu

SHAPES = [  # B, Hq, Hk, Sq, Sk, D, causal
    (1, 4, 1, 250, 2100, 128, True),   # splits over a chunk of queries, ragged ends
    (1, 8, 2, 3, 1500, 128, True),     # packed rows of three positions, one row block
    (2, 8, 1, 40, 700, 128, True),     # packed: heads change inside a wave's rows
    (1, 2, 2, 900, 900, 128, True),    # early row blocks leave later splits empty
    (1, 2, 1, 700, 300, 128, True),    # too few key blocks: not cut; rows that see no key
    (1, 2, 2, 900, 700, 128, True),    # cut, with rows that see no key of any split
    (1, 2, 2, 700, 600, 64, True),
    (1, 2, 2, 130, 1000, 128, False),  # no mask, one row past a block
    (1, 2, 2, 300, 130, 128, False),   # no mask, one split, single blocks
    (3, 6, 2, 1, 64 * 9 + 1, 64, False),
    (1, 4, 4, 129, 1900, 64, True),
    (1, 16, 1, 17, 1000, 64, True),
    (1, 1, 1, 1, 4000, 64, True),      # one row, many splits
]


def _desc(B, Hq, Hk, Sq, Sk, D, causal, dtype):
    d = _abi.AttnDesc()
    d.batch, d.heads_q, d.heads_kv, d.seq_q, d.seq_kv, d.head_dim = B, Hq, Hk, Sq, Sk, D
    d.dtype = _abi.DTYPE_BF16 if dtype == torch.bfloat16 else _abi.DTYPE_F16
    d.causal = int(causal)
    return d


@pytest.mark.parametrize("ws", [True, False], ids=["workspace", "none"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,Hq,Hk,Sq,Sk,D,causal", SHAPES)
def test_short_launches(B, Hq, Hk, Sq, Sk, D, causal, dtype, ws):
    print(f"case: split B={B} Hq={Hq} Hk={Hk} Sq={Sq} Sk={Sk} D={D} causal={causal} {dtype} "
          f"ws={ws}", flush=True)
    lib = _abi.load_library()
    q = randn((B, Hq, Sq, D), seed=1, dtype=dtype, scale=0.5)
    k, v = (randn((B, Hk, Sk, D), seed=s, dtype=dtype, scale=0.5) for s in (2, 3))
    dq, dk, dv = (t.cuda() for t in (q, k, v))
    o = torch.full_like(dq, float("nan"))
    lse = torch.full((B, Hq, Sq), float("nan"), device="cuda")
    d = _desc(B, Hq, Hk, Sq, Sk, D, causal, dtype)
    args = [ctypes.byref(d), dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), o.data_ptr(),
            lse.data_ptr()]
    stream = torch.cuda.current_stream().cuda_stream
    if ws:
        n = ctypes.c_size_t()
        _abi.check(lib.neptune_attn_workspace_bytes(ctypes.byref(d), ctypes.byref(n)), lib)
        assert (n.value > 0) == (Sk > 300)  # cut, from ten key blocks on here
        buf = torch.full((n.value // 4 + 4,), float("nan"), device="cuda")
        _abi.check(lib.neptune_attn_fwd_ws(*args, buf.data_ptr(), n.value, stream), lib)
    else:
        _abi.check(lib.neptune_attn_fwd(*args, stream), lib)
    torch.cuda.synchronize()
    if ws:  # nothing past the workspace's bytes
        assert torch.isnan(buf[n.value // 4:]).all()
    ro, rl = oracle.attn_fwd(bits(q), bits(k), bits(v), oracle_dtype(q), causal)
    assert max_abs(to_f32(o), oracle.decode(ro, oracle_dtype(q))) <= TOL_BF16_ABS
    lse = to_f32(lse)
    assert np.array_equal(np.isneginf(lse), np.isneginf(rl))
    fin = np.isfinite(rl)
    assert np.abs(lse[fin] - rl[fin]).max() <= TOL_LSE_ABS


@pytest.mark.parametrize("ws", [True, False], ids=["workspace", "none"])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
def test_non_finite_values_far_below_the_max(bad, D, ws):
    """A V row that is not finite, at a key whose probability underflows next to
    a later split's: the column is not finite, cut or not."""
    from neptune_hip import ops
    print(f"case: split V={bad} D={D} ws={ws}", flush=True)
    q = torch.ones((1, 1, 3, D), dtype=torch.bfloat16, device="cuda")
    k = torch.zeros((1, 1, 4000, D), dtype=torch.bfloat16, device="cuda")
    k[:, :, 3000] = 400.0 / D ** 0.5  # 577 (log2 units) above the other keys
    v = torch.ones_like(k)
    v[:, :, 10, 5] = bad
    if ws:
        o = ops.attention(q, k, v)
    else:
        lib = _abi.load_library()
        o, d = torch.empty_like(q), _desc(1, 1, 1, 3, 4000, D, False, torch.bfloat16)
        _abi.check(lib.neptune_attn_fwd(ctypes.byref(d), q.data_ptr(), k.data_ptr(), v.data_ptr(),
                                        o.data_ptr(), None,
                                        torch.cuda.current_stream().cuda_stream), lib)
    finite = torch.isfinite(o.cpu())
    assert not finite[..., 5].any()
    finite[..., 5] = True
    assert finite.all()


def test_workspace_too_small():
    lib = _abi.load_library()
    d = _desc(1, 4, 1, 250, 2100, 128, True, torch.bfloat16)
    n = ctypes.c_size_t()
    _abi.check(lib.neptune_attn_workspace_bytes(ctypes.byref(d), ctypes.byref(n)), lib)
    assert n.value > 0
    x = torch.zeros(4 * 2100 * 128, dtype=torch.bfloat16, device="cuda")
    p = x.data_ptr()
    for ws, size in ((p, n.value - 1), (None, 0)):
        st = lib.neptune_attn_fwd_ws(ctypes.byref(d), p, p, p, p, None, ws, size, None)
        assert st == _abi.ERR_WORKSPACE_TOO_SMALL
    assert lib.neptune_attn_fwd_ws(ctypes.byref(d), p, p, p, p, None, p + 4, n.value, None) == \
        _abi.ERR_UNSUPPORTED
    # a launch that is not cut needs none
    d = _desc(4, 32, 32, 512, 512, 128, True, torch.bfloat16)
    _abi.check(lib.neptune_attn_workspace_bytes(ctypes.byref(d), ctypes.byref(n)), lib)
    assert n.value == 0
