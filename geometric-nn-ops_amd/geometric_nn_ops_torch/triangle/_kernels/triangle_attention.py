"""Host side of the HIP triangle-attention forward.

``triangle_attention_hip`` takes the canonical 5D layout with a boolean mask and stands
in for the reference's ``triangle_attention_triton`` + ``EvoformerAttention.forward``
(geometric_nn_ops_torch/triangle/_kernels/triangle_attention.py:1447-1484, :1091-1276):
same argument meaning, same shape assertions, ``scale=None`` meaning ``D**-0.5``, and the
masked-key bias rounded to the input dtype. It is forward-only. q/k/v/bias views are
passed to the kernel through their strides (no copies unless a stride or alignment is
unusable), and the output is a fresh contiguous ``[B, N_seq, N_res, H, D]`` tensor.
"""

import ctypes
import functools

import torch

from ... import _lib, _precision
from .._masking import rounded_mask_value

MAX_HEAD_DIM = 256  # the kernel's largest head-dim tile (16-bit inputs)
MAX_HEAD_DIM_FP32 = 128  # fp32 tiles take twice the LDS
MAX_N_RES = 32768


def max_head_dim(dtype: torch.dtype) -> int:
    return MAX_HEAD_DIM_FP32 if dtype == torch.float32 else MAX_HEAD_DIM


def supports(q: torch.Tensor) -> bool:
    """Whether the HIP kernel covers this input (dtype handled by the caller)."""
    return q.shape[-1] <= max_head_dim(q.dtype) and q.shape[-3] <= MAX_N_RES


def _vectorizable(t: torch.Tensor) -> bool:
    """Unit stride on the last of five dims, the other strides multiples of 8 elements, 16-byte
    base."""
    s0, s1, s2, s3, s4 = t.stride()
    return s4 == 1 and (s0 | s1 | s2 | s3) % 8 == 0 and t.data_ptr() % 16 == 0


def _prepare(t: torch.Tensor) -> torch.Tensor:
    """q/k/v in a form the kernel can address: unit stride on D, other strides multiples
    of 8 elements and a 16-byte aligned base; D padded to a multiple of 8."""
    d = t.shape[-1]
    if d % 8:
        t = torch.nn.functional.pad(t, (0, 8 - d % 8))
    if not _vectorizable(t):
        t = t.contiguous()
        if not _vectorizable(t):
            t = t.clone()
    return t


def _bias_readable(bias: torch.Tensor) -> bool:
    """Whether every row ``[b, 0, h, i, :]`` starts on 16 bytes, has unit stride and can be read up to
    round_up(N, 8): inside its own pitch (a bias broadcast over the queries has none) and, for the
    last row, inside the storage."""
    B, _, H, N, _ = bias.shape
    b, _, h, i, j = bias.stride()
    if j != 1 or i % 8 or (H > 1 and h % 8) or (B > 1 and b % 8) or bias.data_ptr() % 16:
        return False
    if N % 8 == 0:
        return True
    end = bias.storage_offset() + (B - 1) * b + (H - 1) * h + (N - 1) * i + (N + 7) // 8 * 8
    return i >= N and end * bias.element_size() <= bias.untyped_storage().nbytes()


def _prepare_bias(bias: torch.Tensor, dtype: torch.dtype) -> torch.Tensor:
    """``[B, 1, H, N, N]`` bias in ``dtype``. The 16-bit row kernel reads any strides (its
    pre-pass rewrites the bias in fragment order); the tiled kernel and the backward read rows in
    aligned groups of 8 elements, so a view whose rows cannot be read that way (``_bias_readable``)
    is copied with the pitch padded. No kernel uses what lies past N, so the padding is not
    filled (the fill cost 5 us of a 145 us forward at N = 333 in fp32)."""
    bias = bias.to(dtype)
    if _bias_readable(bias):
        return bias
    B, _, H, N, _ = bias.shape
    pitch = (N + 7) // 8 * 8
    padded = torch.empty((B, 1, H, N, pitch), device=bias.device, dtype=bias.dtype)
    padded[..., :N] = bias
    return padded[..., :N]


def _set_bias(args, bias: torch.Tensor) -> None:
    args.bias = bias.data_ptr()
    args.bias_stride = _lib.I64x4(bias.stride(0), bias.stride(2), bias.stride(3), bias.stride(4))


def workspace_for(args, device) -> torch.Tensor | None:
    """Sets ``args.workspace`` to a fresh scratch tensor of the size the library asks for
    (``None`` when the call needs none); the caller keeps the tensor alive over the launch."""
    nbytes = _lib.load().gnn_triattn_workspace_bytes(ctypes.byref(args))
    if nbytes == 0:
        return None
    ws = torch.empty(nbytes, device=device, dtype=torch.uint8)
    args.workspace, args.workspace_bytes = ws.data_ptr(), nbytes
    return ws


def bias_and_workspace(args, bias, device):
    """``(bias, workspace)`` for a forward whose ``args`` (shapes and dtype set) point at the
    ``[B, 1, H, N, N]`` pair bias; the caller keeps both alive. The library asks for fragment-order
    scratch exactly when its row-resident kernel runs, and that kernel's pre-pass reads any strides;
    otherwise the bias takes the layout that the tiled kernel needs. Asking the library keeps this
    decision in one place (``triattn_row_applicable`` in the C sources)."""
    if bias is None:
        return None, None
    ws = workspace_for(args, device)
    if ws is None:
        bias = _prepare_bias(bias, bias.dtype)
        _set_bias(args, bias)
    return bias, ws


def triangle_attention_hip(q, k, v, bias=None, mask=None, scale=None, dynamic=False, use_exp2=False,
                           lse=None, mask_value=None, row_max=None, precision=None):
    """Triangle attention forward on the canonical 5D layout.

    q/k/v ``[B, N_seq, N_res, H, D]`` (bf16, fp16 or fp32, on a HIP device); bias
    ``[B, 1, H, N_res, N_res]`` or ``None``; mask ``[B, N_seq, 1, 1, N_res]`` bool or
    ``None``. ``dynamic`` is accepted for API parity and has no effect (N is always a
    runtime argument); ``use_exp2`` likewise (the kernel always evaluates the softmax in
    base 2). ``lse``, if given, is a float32 ``[B, N_seq, H, N_res]`` tensor that receives
    the natural-log log-sum-exp of each query's logits; ``row_max``, likewise shaped, receives
    each query's largest logit (scaled q.k + bias + mask term). ``mask_value`` overrides the logit
    offset of masked keys (default: the dtype's sentinel rounded to the dtype, as the
    reference launcher applies it).
    """
    del dynamic, use_exp2
    if q.dtype not in _lib.DTYPE_CODE:
        raise TypeError(f"triangle_attention_hip: unsupported dtype {q.dtype}")
    dim_q, dim_k, dim_v = q.shape[-1], k.shape[-1], v.shape[-1]
    assert dim_q == dim_k and dim_k == dim_v
    B, S, N, H, D = q.shape
    assert k.shape == q.shape and v.shape == q.shape, f"{tuple(k.shape)} / {tuple(v.shape)} != {tuple(q.shape)}"
    if mask is not None:
        assert mask.shape == (B, S, 1, 1, N), f"{tuple(mask.shape)} != {(B, S, 1, 1, N)}"
    if bias is not None:
        assert bias.shape == (B, 1, H, N, N), f"{tuple(bias.shape)} != {(B, 1, H, N, N)}"
    if scale is None:
        scale = D**-0.5

    qk, kk, vk = _prepare(q), _prepare(k), _prepare(v)
    Dp = qk.shape[-1]
    o = torch.empty((B, S, N, H, Dp), device=q.device, dtype=q.dtype)

    bias_ptr, (b0, b1, b2, b3) = 0, (0, 0, 0, 0)
    if bias is not None:
        bias = bias.to(q.dtype)
        bias_ptr, (b0, _, b1, b2, b3) = bias.data_ptr(), bias.stride()
    mask_ptr, (m0, m1, _, _, m2) = 0, (0, 0, 0, 0, 0)
    if mask is not None:
        if mask.dtype != torch.bool:
            raise ValueError(f"mask must be bool (keep=True/mask=False), got {mask.dtype}")
        mask_ptr, (m0, m1, _, _, m2) = mask.data_ptr(), mask.stride()
    for t in (lse, row_max):
        assert t is None or (t.shape == (B, S, H, N) and t.dtype == torch.float32 and t.is_contiguous())
    if precision is None:
        precision = _precision.matmul_precision(fp32_operands=q.dtype == torch.float32)
    args = _lib.TriAttnArgs()
    _lib.pack_triattn(
        args, 0, qk.data_ptr(), kk.data_ptr(), vk.data_ptr(), o.data_ptr(), bias_ptr, mask_ptr,
        0 if lse is None else lse.data_ptr(), 0 if row_max is None else row_max.data_ptr(), B, S, N, H, Dp,
        *qk.stride()[:4], *kk.stride()[:4], *vk.stride()[:4], *o.stride()[:4], b0, b1, b2, b3, m0, m1, m2,
        0.0, 0.0, _lib.DTYPE_CODE[q.dtype], _lib.PRECISION_CODE[precision], 0, 0)
    args.scale = float(scale)
    args.mask_value = rounded_mask_value(q.dtype) if mask_value is None else float(mask_value)

    bias, ws = bias_and_workspace(args, bias, q.device)
    _lib.call("gnn_triattn_fwd", args, q.device)
    del ws
    if Dp != D:
        o = o[..., :D].contiguous()
    return o


def backward_supported(q: torch.Tensor) -> bool:
    """Whether the HIP backward covers these inputs: a head dim that is a multiple of 8, at
    most 128 for bf16 / fp16 and at most 64 for fp32 (whose tiles take twice the LDS)."""
    d = q.shape[-1]
    if d % 8 != 0:
        return False
    if q.dtype in (torch.bfloat16, torch.float16):
        return d <= 128
    return q.dtype == torch.float32 and d <= 64


_CUS = 256  # MI355X compute units; the pair-bias kernel's LDS ring holds one workgroup each
_ROW_S = 1.5e-6  # one N_seq row of a 128 x 128 tile (measured at D = 32)
_PLANE_BPS = 5.0e12  # a partial plane is written once and read once by the ordered reduction


@functools.lru_cache(maxsize=256)
def dbias_splits(B: int, S: int, N: int, H: int) -> int:
    """N_seq ranges for the pair-bias gradient (at most N_seq and 64), minimising a cost
    model: the rounds of (128 x 128 tile, range) workgroups over the compute units times the
    rows per range, plus the fp32 partial plane that each range writes and the ordered
    reduction reads back."""
    tiles = B * H * ((N + 127) // 128) ** 2
    plane = B * H * N * N * 4
    best, best_cost = 1, None
    for s in range(1, min(S, 64) + 1):
        rounds = -(-tiles * s // _CUS)
        cost = rounds * -(-S // s) * _ROW_S + (2 * s * plane / _PLANE_BPS if s > 1 else 0.0)
        if best_cost is None or cost < best_cost:
            best, best_cost = s, cost
    return best


def triangle_attention_bwd_hip(q, k, v, o, dout, lse, bias=None, mask=None, scale=None, mask_value=None,
                               need_dbias=True, precision=None):
    """Gradients of the HIP forward: ``(dq, dk, dv, dbias)`` with dq/dk/dv like q and dbias
    ``[B, 1, H, N, N]`` fp32 (``None`` without a bias or when ``need_dbias`` is false).
    Replaces EvoformerAttention.backward (triangle_attention.py:1278-1442); ``lse`` is the
    forward's ``[B, N_seq, H, N]`` natural-log log-sum-exp. fp32 products run as the
    forward's did: ``precision`` is the resolved ``'ieee'`` or ``'bf16x3'`` (``None``:
    resolved now from ``torch.backends.cuda.matmul.fp32_precision``)."""
    B, S, N, H, D = q.shape
    if scale is None:
        scale = D**-0.5
    qk, kk, vk, ok, dk_ = (_prepare(t) for t in (q, k, v, o, dout.to(q.dtype)))
    assert qk.shape[-1] == D, "the HIP backward needs a head dim that is a multiple of 8"
    dq = torch.empty((B, S, N, H, D), device=q.device, dtype=q.dtype)
    dk = torch.empty_like(dq)
    dv = torch.empty_like(dq)
    delta = torch.empty((B, S, H, N), device=q.device, dtype=torch.float32)
    lse = lse.contiguous()
    dbias, ws, splits = None, None, 0
    bias_ptr, (b0, b1, b2, b3) = 0, (0, 0, 0, 0)
    if bias is not None:
        bias = _prepare_bias(bias, q.dtype)
        bias_ptr, (b0, _, b1, b2, b3) = bias.data_ptr(), bias.stride()
        if need_dbias:
            dbias = torch.empty((B, 1, H, N, N), device=q.device, dtype=torch.float32)
            splits = dbias_splits(B, S, N, H)
            if splits > 1:
                ws = torch.empty((splits, B, H, N, N), device=q.device, dtype=torch.float32)
    mask_ptr, (m0, m1, _, _, m2) = 0, (0, 0, 0, 0, 0)
    if mask is not None:
        mask_ptr, (m0, m1, _, _, m2) = mask.data_ptr(), mask.stride()
    if precision is None:
        precision = _precision.matmul_precision(fp32_operands=q.dtype == torch.float32)
    grad_stride = dq.stride()[:4]  # dk and dv have it too
    a = _lib.TriAttnBwdArgs()
    _lib.pack_triattn_bwd(
        a, 0, qk.data_ptr(), kk.data_ptr(), vk.data_ptr(), ok.data_ptr(), dk_.data_ptr(), bias_ptr, mask_ptr,
        lse.data_ptr(), dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), 0 if dbias is None else dbias.data_ptr(),
        delta.data_ptr(), 0 if ws is None else ws.data_ptr(), splits, B, S, N, H, D,
        *qk.stride()[:4], *kk.stride()[:4], *vk.stride()[:4], *ok.stride()[:4], *dk_.stride()[:4],
        *grad_stride, *grad_stride, *grad_stride, b0, b1, b2, b3, m0, m1, m2,
        0.0, 0.0, _lib.DTYPE_CODE[q.dtype], _lib.PRECISION_CODE[precision])
    a.scale = float(scale)
    a.mask_value = rounded_mask_value(q.dtype) if mask_value is None else float(mask_value)
    _lib.call("gnn_triattn_bwd", a, q.device)
    return dq, dk, dv, dbias
