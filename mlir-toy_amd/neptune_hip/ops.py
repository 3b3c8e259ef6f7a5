"""torch-tensor front of the C-ABI (device memory and streams only).

Every function hands raw device pointers, sizes and the current HIP stream
to libneptune_hip.so; no computation happens in Python and there is no
fallback path: if the library is missing, ``load_library`` raises.
"""

from __future__ import annotations

import ctypes
import functools
import math

import torch

from . import _abi
from ._abi import check, load_library

LOG2E = 1.4426950408889634

_TORCH_TO_DTYPE = {
    torch.float32: _abi.DTYPE_F32,
    torch.float16: _abi.DTYPE_F16,
    torch.bfloat16: _abi.DTYPE_BF16,
}


# The checks of a call and its descriptor depend on the tensors' shapes,
# strides, dtypes and devices and on the options alone, so each entry point
# keeps them by those values (bounded; a call that fails its checks is not
# kept) and by the options' types: 4.0 is no split count, equal to 4 or not.
# Working them out took 3-8 us of every call, as long as the smallest
# kernels run: now a lookup.
_PLANS = 1024


def _meta(t: torch.Tensor | None):
    """What a plan may know of a tensor."""
    return None if t is None else (t.shape, t.stride(), t.dtype, t.device)


_raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None) or (
    lambda index: torch.cuda.current_stream(index).cuda_stream)


def _launch(lib, device: torch.device, fn, *args) -> None:
    """fn(*args, stream) on the device's current stream, that device current."""
    index = device.index
    if torch.cuda.current_device() == index:
        st = fn(*args, _raw_stream(index))
    else:
        with torch.cuda.device(device):
            st = fn(*args, _raw_stream(index))
    if st:
        check(st, lib)


def _contiguous(meta) -> bool:
    """Tensor.is_contiguous() of such a tensor."""
    shape, stride = meta[0], meta[1]
    want = 1
    for n, s in zip(reversed(shape), reversed(stride)):
        if n == 0:
            return True
        if n != 1:
            if s != want:
                return 0 in shape
            want *= n
    return True


def _check_workspace(workspace: torch.Tensor | None, device: torch.device) -> None:
    if workspace is None:
        return
    if not workspace.is_cuda:
        raise ValueError("neptune_hip ops take device tensors")
    if workspace.device != device:
        raise ValueError("all tensors must be on the same device")
    # the library writes numel * element_size bytes from data_ptr
    if not workspace.is_contiguous():
        raise ValueError("workspace must be a contiguous tensor")


def _require_cuda(*metas) -> None:
    dev = None
    for m in metas:
        if m is None:
            continue
        if m[3].type != "cuda":
            raise ValueError("neptune_hip ops take device tensors")
        if dev is None:
            dev = m[3]
        elif m[3] != dev:
            raise ValueError("all tensors must be on the same device")


def _strides_bhs(meta) -> tuple[int, int, int]:
    shape, stride = meta[0], meta[1]
    if len(shape) != 4 or stride[-1] != 1:
        raise ValueError("expected a [batch, heads, seq, head_dim] tensor with unit head_dim stride")
    return stride[:3]


def scale_to_log2(scale: float | None, head_dim: int) -> float:
    """Softmax scale (default 1/sqrt(D)) expressed in the exp2 domain."""
    if scale is None:
        return 0.0  # library default: log2(e)/sqrt(head_dim), HTile:24
    return float(scale) * LOG2E


@functools.lru_cache(maxsize=_PLANS, typed=True)
def _attn_plan(q, k, v, out, lse, causal, scale, scale_log2, stages, k_dim_order):
    """(descriptor, bytes of the split states' workspace, LSE shape)."""
    _require_cuda(q, k, v, out, lse)
    if q[2] not in _TORCH_TO_DTYPE or k[2] != q[2] or v[2] != q[2]:
        raise ValueError(f"q, k, v must share one of {list(_TORCH_TO_DTYPE)}")
    B, Hq, Sq, D = q[0]
    if k_dim_order not in (0, 1):
        raise ValueError("k_dim_order must be 0 or 1")
    if k_dim_order:
        Bk, Hk, Dk, Sk = k[0]
    else:
        Bk, Hk, Sk, Dk = k[0]
    if (Bk, Dk) != (B, D) or tuple(v[0]) != (Bk, Hk, Sk, Dk):
        raise ValueError(f"shape mismatch: q {tuple(q[0])} k {tuple(k[0])} v {tuple(v[0])}")
    if out is not None and (out[0] != q[0] or out[2] != q[2]):
        raise ValueError("out must match q's shape and dtype")
    if lse is not None and (tuple(lse[0]) != (B, Hq, Sq) or lse[2] != torch.float32 or
                            not _contiguous(lse)):
        raise ValueError("lse must be a contiguous float32 [B, Hq, Sq] tensor")
    desc = _abi.AttnDesc()
    desc.batch, desc.heads_q, desc.heads_kv = B, Hq, Hk
    desc.seq_q, desc.seq_kv, desc.head_dim = Sq, Sk, D
    desc.q_stride[:] = _strides_bhs(q)
    desc.k_stride[:] = _strides_bhs(k)
    desc.v_stride[:] = _strides_bhs(v)
    desc.o_stride[:] = _strides_bhs(out) if out is not None else (Hq * Sq * D, Sq * D, D)
    desc.dtype = _TORCH_TO_DTYPE[q[2]]
    desc.causal = 1 if causal else 0
    desc.scale_log2 = scale_log2 if scale_log2 is not None else scale_to_log2(scale, D)
    desc.pipeline_stages = stages
    desc.k_dim_order = int(k_dim_order)
    lib = load_library()
    n = ctypes.c_size_t()
    # what the library refuses, the launch itself reports
    st = lib.neptune_attn_workspace_bytes(ctypes.byref(desc), ctypes.byref(n))
    return ctypes.byref(desc), n.value if st == _abi.OK else 0, (B, Hq, Sq)


def attention(
    q: torch.Tensor,
    k: torch.Tensor,
    v: torch.Tensor,
    *,
    causal: bool = False,
    scale: float | None = None,
    return_lse: bool = False,
    out: torch.Tensor | None = None,
    lse: torch.Tensor | None = None,
    scale_log2: float | None = None,
    pipeline_stages: int = 0,
    k_dim_order: int = 0,
):
    """softmax(q k^T * scale) v with the HTile numeric policy.

    q [B, Hq, Sq, D], k/v [B, Hkv, Skv, D] in float32, float16 or bfloat16;
    returns out [B, Hq, Sq, D] (and lse [B, Hq, Sq] fp32 if asked).
    ``scale_log2`` gives the score scale already in the exp2 domain (the
    HTile program's own constant, HTile:24), in place of ``scale``.
    ``pipeline_stages`` (0 = default 2, or 1..3) sets how many K/V tiles the
    kernel stages in LDS ahead of use; with ``k_dim_order=1`` k is given as
    [B, Hkv, D, Skv] (seq contiguous), the order of a dimension_order =
    [1, 0] tile load. The stage count does not change the result, and short
    launches may keep two tiles whatever it says. Short launches with
    ``k_dim_order=0`` may be cut along the keys and those with 1 are not, so
    their results may differ by the 16-bit rounding of the probabilities.
    """
    if scale is not None and scale_log2 is not None:
        raise ValueError("give scale or scale_log2, not both")
    desc, ws_bytes, lse_shape = _attn_plan(
        _meta(q), _meta(k), _meta(v), _meta(out), _meta(lse), bool(causal),
        None if scale is None else float(scale),
        None if scale_log2 is None else float(scale_log2), int(pipeline_stages), k_dim_order)
    if out is None:
        out = torch.empty_like(q, memory_format=torch.contiguous_format)
    if lse is not None:
        return_lse = True
    elif return_lse:
        lse = torch.empty(lse_shape, dtype=torch.float32, device=q.device)
    # states of split keys (short launches only): held by the caching allocator
    # until the current stream is past this call
    ws = torch.empty(ws_bytes, dtype=torch.uint8, device=q.device) if ws_bytes else None
    lib = load_library()
    _launch(lib, q.device, lib.neptune_attn_fwd_ws, desc, q.data_ptr(), k.data_ptr(),
            v.data_ptr(), out.data_ptr(), lse.data_ptr() if lse is not None else None,
            ws.data_ptr() if ws is not None else None, ws_bytes)
    return (out, lse) if return_lse else out


def _decode_desc(q_shape, k_shape, num_splits, scale_block, scale, kv_dtype) -> _abi.DecodeDesc:
    B, Hq, D = q_shape
    Bk, Hk, L, Dk = k_shape
    desc = _abi.DecodeDesc()
    desc.batch, desc.heads_q, desc.heads_kv = B, Hq, Hk
    desc.seq_kv, desc.head_dim = L, D
    desc.num_splits = num_splits
    desc.scale_block = scale_block
    desc.q_dtype = _abi.DTYPE_BF16
    desc.kv_dtype = kv_dtype
    desc.scale_log2 = scale_to_log2(scale, D)
    return desc


def _decode_bytes(desc: _abi.DecodeDesc) -> int:
    n = ctypes.c_size_t()
    lib = load_library()
    check(lib.neptune_decode_workspace_bytes(ctypes.byref(desc), ctypes.byref(n)), lib)
    return n.value


def decode_workspace_bytes(q, k, *, num_splits: int = 0, fp8: bool = False) -> int:
    return _decode_bytes(_decode_desc(_as_q3(q).shape, k.shape, num_splits, 64, None,
                                      _abi.DTYPE_FP8_E4M3 if fp8 else _abi.DTYPE_BF16))


def _as_q3(q: torch.Tensor) -> torch.Tensor:
    if q.dim() == 4:
        if q.shape[2] != 1:
            raise ValueError("decode takes one query token per sequence")
        q = q[:, :, 0, :]
    return q


@functools.lru_cache(maxsize=_PLANS, typed=True)
def _decode_plan(q, k, v, k_scale, v_scale, num_splits, scale_block, scale):
    """(descriptor, workspace bytes)."""
    fp8 = k[2] in (torch.uint8, torch.float8_e4m3fn)
    if q[2] != torch.bfloat16:
        raise ValueError("decode query must be bfloat16")
    if not fp8 and k[2] != torch.bfloat16:
        raise ValueError("decode KV must be bfloat16 or E4M3 codes")
    if len(q[0]) != 3 or len(k[0]) != 4:
        raise ValueError("decode takes q [B, Hq, D] and k, v [B, Hkv, L, D]")
    if v[2] != k[2] or v[0] != k[0]:
        raise ValueError("k and v must match")
    B, _, D = q[0]
    Bk, Hk, L, Dk = k[0]
    if (Bk, Dk) != (B, D):
        raise ValueError(f"k {tuple(k[0])} does not match q {tuple(q[0])} in batch or "
                         "head_dim")
    for m in (q, k, v):
        if not _contiguous(m):
            raise ValueError("decode tensors must be contiguous")
    if fp8:
        if scale_block <= 0:
            raise ValueError("scale_block must be positive")
        want = (B, Hk, -(-L // scale_block))
        for name, m in (("k_scale", k_scale), ("v_scale", v_scale)):
            if m is None or m[2] != torch.float32 or not _contiguous(m) or tuple(m[0]) != want:
                raise ValueError(f"fp8 KV needs {name}: contiguous float32 {list(want)} "
                                 f"(scale_block {scale_block})")
    elif k_scale is not None or v_scale is not None:
        raise ValueError("k_scale / v_scale apply to E4M3 KV only")
    _require_cuda(q, k, v, k_scale, v_scale)
    desc = _decode_desc(q[0], k[0], num_splits, scale_block, scale,
                        _abi.DTYPE_FP8_E4M3 if fp8 else _abi.DTYPE_BF16)
    return ctypes.byref(desc), _decode_bytes(desc)


def decode_splitk(
    q: torch.Tensor,
    k: torch.Tensor,
    v: torch.Tensor,
    *,
    k_scale: torch.Tensor | None = None,
    v_scale: torch.Tensor | None = None,
    num_splits: int = 0,
    scale_block: int = 64,
    scale: float | None = None,
    return_lse: bool = False,
    workspace: torch.Tensor | None = None,
):
    """Split-K flash-decoding over grouped KV heads.

    q [B, Hq, D] (or [B, Hq, 1, D]) bf16; k/v [B, Hkv, L, D] bf16, or E4M3
    codes (uint8 / torch.float8_e4m3fn) with k_scale/v_scale
    [B, Hkv, ceil(L/scale_block)] fp32. Returns o [B, Hq, D] bf16.
    """
    q3 = _as_q3(q)
    desc, need = _decode_plan(_meta(q3), _meta(k), _meta(v), _meta(k_scale), _meta(v_scale),
                              num_splits, scale_block, None if scale is None else float(scale))
    _check_workspace(workspace, q3.device)
    if workspace is None:
        workspace = torch.empty(max(need, 1), dtype=torch.uint8, device=q3.device)
    out = torch.empty_like(q3)
    lse = torch.empty(q3.shape[:2], dtype=torch.float32, device=q3.device) if return_lse else None
    lib = load_library()
    _launch(lib, q3.device, lib.neptune_decode_splitk, desc, q3.data_ptr(), k.data_ptr(),
            v.data_ptr(), k_scale.data_ptr() if k_scale is not None else None,
            v_scale.data_ptr() if v_scale is not None else None, out.data_ptr(),
            lse.data_ptr() if lse is not None else None, workspace.data_ptr(),
            workspace.numel() * workspace.element_size())
    return (out, lse) if return_lse else out


@functools.lru_cache(maxsize=_PLANS, typed=True)
def _paged_plan(q, k_pages, v_pages, block_table, seq_lens, k_scales, v_scales, max_seq_len,
                num_splits, scale):
    """(descriptor, page descriptor, workspace bytes, whether the pools are E4M3)."""
    fp8 = k_pages[2] in (torch.uint8, torch.float8_e4m3fn)
    if q[2] != torch.bfloat16 or k_pages[2] != v_pages[2] or \
            not (fp8 or k_pages[2] == torch.bfloat16):
        raise ValueError("paged decode takes bfloat16 q and bfloat16 or E4M3 KV pages")
    if len(k_pages[0]) != 4 or k_pages[0] != v_pages[0] or k_pages[1][-1] != 1 or \
            v_pages[1][-1] != 1:
        raise ValueError("k_pages / v_pages: matching [pages, Hkv, page_size, D] views, D contiguous")
    for name, m in (("block_table", block_table), ("seq_lens", seq_lens)):
        if m[2] != torch.int32 or not _contiguous(m):
            raise ValueError(f"{name} must be a contiguous int32 tensor")
    npages, Hk, psize, D = k_pages[0]
    if len(q[0]) != 3 or q[0][2] != D:
        raise ValueError(f"q {tuple(q[0])} does not match the pools' head_dim {D}")
    if fp8:
        for name, m in (("k_scales", k_scales), ("v_scales", v_scales)):
            if m is None or m[2] != torch.float32 or not _contiguous(m) or \
                    tuple(m[0]) != (npages, Hk):
                raise ValueError(f"fp8 pages need {name}: contiguous float32 [num_pages, Hkv]")
    elif k_scales is not None or v_scales is not None:
        raise ValueError("k_scales / v_scales apply to E4M3 pools only")
    B = q[0][0]
    if len(block_table[0]) != 2 or block_table[0][0] != B or tuple(seq_lens[0]) != (B,):
        raise ValueError("block_table [B, max_pages] and seq_lens [B] must match q's batch")
    _require_cuda(q, k_pages, v_pages, block_table, seq_lens, k_scales, v_scales)
    max_pages = block_table[0][1]
    L = max_seq_len if max_seq_len is not None else max_pages * psize
    desc = _decode_desc(q[0], (B, Hk, L, D), num_splits, psize if fp8 else 64, scale,
                        _abi.DTYPE_FP8_E4M3 if fp8 else _abi.DTYPE_BF16)
    pk = _abi.PagedKvDesc()
    pk.num_pages, pk.page_size, pk.max_pages = npages, psize, max_pages
    pk.k_stride[:] = k_pages[1][:3]
    pk.v_stride[:] = v_pages[1][:3]
    return ctypes.byref(desc), ctypes.byref(pk), _decode_bytes(desc), fp8


def decode_paged(
    q: torch.Tensor,
    k_pages: torch.Tensor,
    v_pages: torch.Tensor,
    block_table: torch.Tensor,
    seq_lens: torch.Tensor,
    *,
    max_seq_len: int | None = None,
    num_splits: int = 0,
    scale: float | None = None,
    return_lse: bool = False,
    workspace: torch.Tensor | None = None,
    k_scales: torch.Tensor | None = None,
    v_scales: torch.Tensor | None = None,
):
    """Split-K decode over a paged KV cache.

    q [B, Hq, D] bf16; k_pages / v_pages [num_pages, Hkv, page_size, D]
    views (any page/head/position strides with D contiguous, e.g. a permuted
    [num_pages, page_size, Hkv, D] pool) of bf16, or of E4M3 codes (uint8 /
    torch.float8_e4m3fn) with k_scales / v_scales fp32 [num_pages, Hkv]
    (one scale per page and kv head); block_table [B, max_pages] and
    seq_lens [B] int32 on the device. ``max_seq_len`` (default
    max_pages * page_size) is the longest sequence and sets the split
    layout. Returns o [B, Hq, D] bf16.
    """
    q3 = _as_q3(q)
    desc, pk, need, fp8 = _paged_plan(
        _meta(q3), _meta(k_pages), _meta(v_pages), _meta(block_table), _meta(seq_lens),
        _meta(k_scales), _meta(v_scales), None if max_seq_len is None else int(max_seq_len),
        num_splits, None if scale is None else float(scale))
    _check_workspace(workspace, q3.device)
    if workspace is None:
        workspace = torch.empty(max(need, 1), dtype=torch.uint8, device=q3.device)
    out = torch.empty_like(q3)
    lse = torch.empty(q3.shape[:2], dtype=torch.float32, device=q3.device) if return_lse else None
    tail = (block_table.data_ptr(), seq_lens.data_ptr(), out.data_ptr(),
            lse.data_ptr() if lse is not None else None, workspace.data_ptr(),
            workspace.numel() * workspace.element_size())
    lib = load_library()
    if fp8:
        _launch(lib, q3.device, lib.neptune_decode_paged_fp8, desc, pk, q3.data_ptr(),
                k_pages.data_ptr(), v_pages.data_ptr(), k_scales.data_ptr(), v_scales.data_ptr(),
                *tail)
    else:
        _launch(lib, q3.device, lib.neptune_decode_paged, desc, pk, q3.data_ptr(),
                k_pages.data_ptr(), v_pages.data_ptr(), *tail)
    return (out, lse) if return_lse else out


def kv_quantize_fp8(kv: torch.Tensor, *, scale_block: int = 64):
    """bf16 [B, Hkv, L, D] -> (E4M3 codes uint8, scales fp32 [B, Hkv, nblocks])."""
    if not kv.is_cuda:
        raise ValueError("neptune_hip ops take device tensors")
    if kv.dtype != torch.bfloat16 or kv.dim() != 4 or not kv.is_contiguous():
        raise ValueError("kv_quantize_fp8 takes a contiguous bf16 [B, Hkv, L, D] tensor")
    B, Hk, L, D = kv.shape
    device = kv.device
    codes = torch.empty(kv.shape, dtype=torch.uint8, device=device)
    scales = torch.empty((B, Hk, -(-L // scale_block)), dtype=torch.float32, device=device)
    lib = load_library()
    _launch(lib, device, lib.neptune_kv_quantize_fp8, B, Hk, L, D, scale_block, kv.data_ptr(),
            codes.data_ptr(), scales.data_ptr())
    return codes, scales


@functools.lru_cache(maxsize=_PLANS, typed=True)
def _scan_plan(u, delta, A, B, C, D, z, delta_bias, delta_softplus):
    """The descriptor."""
    for name, m in (("u", u), ("delta", delta), ("B", B), ("C", C), ("z", z)):
        if m is not None and (m[2] != torch.bfloat16 or not _contiguous(m)):
            raise ValueError(f"{name} must be contiguous bfloat16")
    for name, m in (("A", A), ("D", D), ("delta_bias", delta_bias)):
        if m is not None and (m[2] != torch.float32 or not _contiguous(m)):
            raise ValueError(f"{name} must be contiguous float32")
    if len(u[0]) != 3 or len(A[0]) != 2:
        raise ValueError("selective_scan takes u [batch, dim, L] and A [dim, d_state]")
    bsz, dim, L = u[0]
    N = A[0][1]
    want = {"delta": (bsz, dim, L), "A": (dim, N), "B": (bsz, N, L), "C": (bsz, N, L),
            "z": (bsz, dim, L), "D": (dim,), "delta_bias": (dim,)}
    for name, m in (("delta", delta), ("A", A), ("B", B), ("C", C), ("z", z), ("D", D),
                    ("delta_bias", delta_bias)):
        if m is not None and tuple(m[0]) != want[name]:
            raise ValueError(f"selective_scan: {name} is {tuple(m[0])}, expected "
                             f"{want[name]}")
    _require_cuda(u, delta, A, B, C, D, z, delta_bias)
    return ctypes.byref(_abi.ScanDesc(bsz, dim, L, N, _abi.DTYPE_BF16, 1 if delta_softplus else 0))


def selective_scan(
    u: torch.Tensor,
    delta: torch.Tensor,
    A: torch.Tensor,
    B: torch.Tensor,
    C: torch.Tensor,
    D: torch.Tensor | None = None,
    z: torch.Tensor | None = None,
    delta_bias: torch.Tensor | None = None,
    delta_softplus: bool = True,
) -> torch.Tensor:
    """Mamba-1 selective scan (selective_scan_fn argument order).

    u, delta, z [batch, dim, L] and B, C [batch, d_state, L] bf16; A
    [dim, d_state], D and delta_bias [dim] fp32. Returns y [batch, dim, L] bf16.
    """
    desc = _scan_plan(_meta(u), _meta(delta), _meta(A), _meta(B), _meta(C), _meta(D), _meta(z),
                      _meta(delta_bias), bool(delta_softplus))
    y = torch.empty_like(u)
    lib = load_library()
    _launch(lib, u.device, lib.neptune_selective_scan_fwd, desc, u.data_ptr(), delta.data_ptr(),
            A.data_ptr(), B.data_ptr(), C.data_ptr(), D.data_ptr() if D is not None else None,
            z.data_ptr() if z is not None else None,
            delta_bias.data_ptr() if delta_bias is not None else None, y.data_ptr())
    return y


def default_scale(head_dim: int) -> float:
    return 1.0 / math.sqrt(head_dim)
