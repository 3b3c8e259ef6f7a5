"""The scan's sequence-parallel path where rows do not start on 4 bytes (odd
lengths, or a base 2 bytes off): the state pass reads 16-bit steps and each
chunk's scratch starts at its segment's first multiple of 4 bytes. Against the
fp64 oracle, at the scan contract (2e-2 max(1, |ref|) of the bf16 result)."""

import ctypes

import numpy as np
import pytest
import torch

import oracle
from helpers import bits, randn, to_f32
from neptune_hip import _abi, ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("b,d,L,gate,softplus,shift", [
    (1, 16, 4097, True, True, 0),    # 64 chunks, the last one step past whole units
    (2, 20, 1001, False, True, 0),   # ragged channel block, no gate
    (1, 33, 641, True, False, 0),    # delta as given
    (1, 40, 2048, True, True, 1),    # even length, every base 2 bytes off
    (1, 2048, 415, True, True, 0),   # too few units for its channel blocks: the single pass
])
def test_chunked_unaligned_rows(b, d, L, gate, softplus, shift):
    print(f"case: scan chunked b={b} d={d} L={L} gate={gate} softplus={softplus} shift={shift}",
          flush=True)
    u, z = randn((b, d, L), seed=1), randn((b, d, L), seed=2)
    Bm, Cm = (randn((b, 16, L), seed=s) for s in (3, 4))
    dr = randn((b, d, L), seed=5) if softplus else randn((b, d, L), seed=5).abs() * 0.1
    A = -torch.exp(randn((d, 16), seed=6, dtype=torch.float32))
    D, bias = (randn((d,), seed=s, dtype=torch.float32) for s in (7, 8))
    if not softplus:
        bias = bias.abs() * 0.1

    def place(t):
        buf = torch.full((t.numel() + 2,), float("nan"), dtype=t.dtype, device="cuda")
        return buf[shift:shift + t.numel()].view(t.shape).copy_(t)

    du, ddr, dB, dC = (place(t) for t in (u, dr, Bm, Cm))
    dz = place(z) if gate else None
    if shift:  # ops allocates y aligned: through the C entry point
        y = place(torch.zeros_like(u))
        desc = _abi.ScanDesc(b, d, L, 16, _abi.DTYPE_BF16, int(softplus))
        lib = _abi.load_library()
        dA, dD, dbias = A.cuda(), D.cuda(), bias.cuda()
        _abi.check(lib.neptune_selective_scan_fwd(
            ctypes.byref(desc), du.data_ptr(), ddr.data_ptr(), dA.data_ptr(), dB.data_ptr(),
            dC.data_ptr(), dD.data_ptr(), dz.data_ptr(), dbias.data_ptr(), y.data_ptr(),
            torch.cuda.current_stream().cuda_stream), lib)
    else:
        y = ops.selective_scan(du, ddr, A.cuda(), dB, dC, D.cuda(), dz, bias.cuda(),
                               delta_softplus=softplus)
    torch.cuda.synchronize()
    ref_bits, _ = oracle.selective_scan(bits(u), bits(dr), A.numpy(), bits(Bm), bits(Cm),
                                        D.numpy(), bits(z) if gate else None, bias.numpy(),
                                        softplus=softplus)
    ref = oracle.decode(ref_bits, oracle.BF16).astype(np.float64)
    got = to_f32(y).astype(np.float64)
    assert np.isfinite(got).all()
    assert (np.abs(got - ref) <= 2e-2 * np.maximum(1.0, np.abs(ref))).all()


@pytest.mark.parametrize("d,L", [(64, 2047), (16, 16383)], ids=["walk", "wave"])
@pytest.mark.parametrize("sign_a,delta", [(1.0, 1.0), (-1.0, -1.0)])
def test_growing_states(d, L, sign_a, delta):
    """Decays above 1, whose product over a chunk (e^96 and more) fp32 does not
    hold: states stay 0 while u is 0 and grow from where it starts, as they do
    step by step; an infinite one stays infinite."""
    print(f"case: scan growing d={d} L={L} A={sign_a} delta={delta}", flush=True)
    u = randn((1, d, L), seed=1)
    u[:, :, :L - 40] = 0
    u[:, 0, 10] = float("inf")
    dr = torch.full((1, d, L), delta, dtype=torch.bfloat16)
    A = torch.full((d, 16), sign_a)
    ones = torch.ones((1, 16, L), dtype=torch.bfloat16)
    y = ops.selective_scan(u.cuda(), dr.cuda(), A.cuda(), ones.cuda(), ones.cuda(),
                           delta_softplus=False)
    ref_bits, _ = oracle.selective_scan(bits(u), bits(dr), A.numpy(), bits(ones), bits(ones),
                                        softplus=False)
    ref = oracle.decode(ref_bits, oracle.BF16).astype(np.float64)
    got = to_f32(y).astype(np.float64)
    assert not np.isfinite(got[0, 0, 10:]).any()
    got, ref = got[0, 1:], ref[0, 1:]
    assert np.isfinite(got).all()
    assert (np.abs(got - ref) <= 2e-2 * np.maximum(1.0, np.abs(ref))).all()
