"""Host side of the HIP triangle multiplicative update forward.

``trimul_hip`` takes the same arguments as the reference's ``trimul_triton``
(geometric_nn_ops_torch/triangle/_kernels/trimul.py:404-448) and runs the whole op as
three HIP kernels through ``gnn_trimul_fwd``: LN-in + gated projections, the per-channel
N x N x N contraction, and LN-out + p_out + gate. Forward only. The intermediates live in
one workspace tensor allocated here through torch's caching allocator.
"""

import ctypes
import functools
import math

import torch

from ... import _lib, _precision
from .._reference.trimul import is_outgoing

_WEIGHT_KEYS = (
    "norm_in_weight", "norm_in_bias", "p_in_weight", "p_in_bias", "g_in_weight", "g_in_bias",
    "norm_out_weight", "norm_out_bias", "p_out_weight", "p_out_bias", "g_out_weight", "g_out_bias",
)
MAX_CHANNELS = 512
WIDE_MAX_CHANNELS = 8192  # the wide-row LayerNorm's limit (gnn_layernorm_rows forward)


def _pad32(n: int) -> int:
    return (n + 31) // 32 * 32


def supports(x: torch.Tensor, p_in_weight: torch.Tensor, *, padded: bool = True) -> bool:
    """Whether the HIP kernels cover these channel counts: at most 512 once rounded up to a
    multiple of 32 (256 for fp32). Widths that are not multiples of 32 run the forward on
    zero-padded copies (``padded``); the HIP backward takes multiples of 32 only."""
    c_z, c_hidden = x.shape[-1], p_in_weight.shape[0] // 2
    if c_z < 1 or c_hidden < 1 or x.dim() < 3:
        return False
    if not padded and (c_z % 32 or c_hidden % 32):
        return False
    limit = 256 if x.dtype == torch.float32 else MAX_CHANNELS
    return _pad32(c_z) <= limit and _pad32(c_hidden) <= limit


def wide_supported(x: torch.Tensor, p_in_weight: torch.Tensor) -> bool:
    """Whether ``trimul_wide_hip`` covers these widths: 16-bit inputs whose c_z or c_hidden
    is above the fused kernels' 512, both multiples of 32 and at most 8192."""
    C, Ch = x.shape[-1], p_in_weight.shape[0] // 2
    return (x.dtype in (torch.bfloat16, torch.float16) and x.dim() >= 3 and C % 32 == 0 and Ch % 32 == 0
            and max(C, Ch) > MAX_CHANNELS and max(C, Ch) <= WIDE_MAX_CHANNELS)


def _pad_channels(x, weights):
    """x and the weights zero-padded to channel counts that are multiples of 32, for the
    forward kernels, with the real widths the LayerNorms average over. The a / b halves of
    the stacked input projections are padded separately (rows [0, Ch) and [Ch', Ch' + Ch)),
    so padded hidden channels give a = b = 0, o = 0, and padded input channels meet zero
    weight columns; the padded output channels are sliced off by the caller.

    Returns (x', weights', C', Ch')."""
    C = x.shape[-1]
    Ch = weights["p_in_weight"].shape[0] // 2
    Cp, Chp = _pad32(C), _pad32(Ch)

    def pad(t, shape, blocks):
        """t copied into zeros of ``shape``; blocks: per dim, the offsets of its parts."""
        out = t.new_zeros(shape)
        if t.dim() == 1:
            for o, (lo, hi) in zip(blocks[0], _parts(t.shape[0], len(blocks[0]))):
                out[o:o + hi - lo] = t[lo:hi]
        else:
            for o, (lo, hi) in zip(blocks[0], _parts(t.shape[0], len(blocks[0]))):
                out[o:o + hi - lo, :t.shape[1]] = t[lo:hi]
        return out

    xp = torch.nn.functional.pad(x, (0, Cp - C))
    w = dict(weights)
    stacked = {"p_in_weight": (2 * Chp, Cp), "g_in_weight": (2 * Chp, Cp), "p_in_bias": (2 * Chp,),
               "g_in_bias": (2 * Chp,)}
    plain = {"p_out_weight": (Cp, Chp), "g_out_weight": (Cp, Cp), "p_out_bias": (Cp,), "g_out_bias": (Cp,),
             "norm_in_weight": (Cp,), "norm_in_bias": (Cp,), "norm_out_weight": (Chp,), "norm_out_bias": (Chp,)}
    for key, shape in stacked.items():
        if w.get(key) is not None:
            w[key] = pad(w[key], shape, [(0, Chp)])
    for key, shape in plain.items():
        if w.get(key) is not None:
            w[key] = pad(w[key], shape, [(0,)])
    return xp, w, Cp, Chp


def _parts(n, k):
    """k equal consecutive parts of range(n)."""
    step = n // k
    return [(i * step, (i + 1) * step) for i in range(k)]


def _aligned(t: torch.Tensor) -> torch.Tensor:
    t = t.contiguous()
    return t if t.data_ptr() % 16 == 0 else t.clone()


def _kernel_ready(t: torch.Tensor, like: torch.Tensor) -> torch.Tensor:
    """``t`` on ``like``'s device and dtype, contiguous and 16-byte aligned (as is, when it
    already is: the usual case for parameters, and the checks are cheaper than the copies)."""
    if t.dtype == like.dtype and t.device == like.device and t.is_contiguous() and t.data_ptr() % 16 == 0:
        return t
    return _aligned(t.to(device=like.device, dtype=like.dtype))


@functools.lru_cache(maxsize=256)
def _workspace_layout(B, N, C, Ch, dtype):
    """(bytes, offsets of a, b, gate and o) of the forward's workspace."""
    offsets = (ctypes.c_size_t * 4)()
    nbytes = _lib.load().gnn_trimul_workspace_bytes(B, N, C, Ch, dtype, offsets)
    return nbytes, tuple(offsets)


def build_args(x, direction, mask, eps, weights, separate_gate=False):
    """Validated, kernel-ready tensors and the filled ``gnn_trimul_args``. With
    ``separate_gate`` the output gate gets a buffer of its own (in the keepalive list) and the
    workspace holds only a, b and o, which is what a backward needs.

    Returns (args, keepalive, out, workspace, offsets)."""
    outgoing = is_outgoing(direction)
    if x.dtype not in _lib.DTYPE_CODE:
        raise TypeError(f"trimul_hip: unsupported dtype {x.dtype}")
    N, N2, C = x.shape[-3], x.shape[-2], x.shape[-1]
    if N != N2:
        raise ValueError(f"x must be [*, N, N, C_z], got {tuple(x.shape)}")
    for key in ("p_in_weight", "g_in_weight", "p_out_weight", "g_out_weight"):
        if weights.get(key) is None:
            raise ValueError(f"{key} is required")
    Ch = weights["p_in_weight"].shape[0] // 2
    expected = {
        "p_in_weight": (2 * Ch, C), "g_in_weight": (2 * Ch, C), "p_out_weight": (C, Ch),
        "g_out_weight": (C, C), "norm_in_weight": (C,), "norm_in_bias": (C,),
        "norm_out_weight": (Ch,), "norm_out_bias": (Ch,), "p_in_bias": (2 * Ch,),
        "g_in_bias": (2 * Ch,), "p_out_bias": (C,), "g_out_bias": (C,),
    }
    for key, shape in expected.items():
        w = weights.get(key)
        if w is not None and w.shape != shape:
            raise ValueError(f"{key} has shape {tuple(w.shape)}, expected {tuple(shape)}")
    lead = x.shape[:-3]
    B = math.prod(lead)

    xk = _aligned(x.reshape(B, N, N, C))
    out = torch.empty((B, N, N, C), device=x.device, dtype=x.dtype)
    keep = [xk]

    mask_ptr, mask_stride = 0, (0, 0, 0)
    if mask is not None:
        m = mask.to(device=x.device, dtype=x.dtype).expand(*x.shape[:-1]).reshape(B, N, N)
        keep.append(m)
        mask_ptr, mask_stride = m.data_ptr(), m.stride()
    ptrs = []  # in _WEIGHT_KEYS order, which is the order of the structure's fields
    xdt, xdev = x.dtype, x.device
    for key in _WEIGHT_KEYS:
        w = weights.get(key)
        if w is None:
            ptrs.append(0)
            continue
        p = w.data_ptr()
        if p % 16 or w.dtype != xdt or w.device != xdev or not w.is_contiguous():
            w = _kernel_ready(w, x)
            p = w.data_ptr()
        keep.append(w)
        ptrs.append(p)
    dtype = _lib.DTYPE_CODE[xdt]
    nbytes, offsets = _workspace_layout(B, N, C, Ch, dtype)
    gate_ptr = 0
    if separate_gate:  # the gate region is the workspace's last: stop before it
        nbytes = offsets[2]
        gate = torch.empty((B, N, N, C), device=x.device, dtype=x.dtype)
        keep.append(gate)
        gate_ptr = gate.data_ptr()
    workspace = torch.empty(nbytes, device=x.device, dtype=torch.uint8)
    precision = _precision.matmul_precision(fp32_operands=x.dtype == torch.float32)
    args = _lib.TrimulArgs()
    _lib.pack_trimul(args, 0, xk.data_ptr(), out.data_ptr(), mask_ptr, *mask_stride, *ptrs, workspace.data_ptr(),
                     nbytes, B, N, C, Ch, 0.0, 1 if outgoing else 0, dtype, _lib.PRECISION_CODE[precision], gate_ptr,
                     0, 0)
    args.eps = float(eps)
    return args, keep, out, workspace, offsets


def run_stage(fn_name: str, args, device) -> None:
    _lib.call(fn_name, args, device)


def trimul_hip(
    x,
    direction="outgoing",
    mask=None,
    *,
    eps=1e-5,
    norm_in_weight=None,
    norm_in_bias=None,
    p_in_weight=None,
    p_in_bias=None,
    g_in_weight=None,
    g_in_bias=None,
    norm_out_weight=None,
    norm_out_bias=None,
    p_out_weight=None,
    p_out_bias=None,
    g_out_weight=None,
    g_out_bias=None,
):
    """Triangle multiplicative update on the HIP kernels. Forward only.

    ``x`` ``[*, N, N, C_z]`` (bf16, fp16 or fp32 on a HIP device), ``mask`` ``[*, N, N]``
    (broadcastable; 1 = keep) or ``None``; weights as in the torch path.
    """
    weights = dict(
        norm_in_weight=norm_in_weight, norm_in_bias=norm_in_bias,
        p_in_weight=p_in_weight, p_in_bias=p_in_bias,
        g_in_weight=g_in_weight, g_in_bias=g_in_bias,
        norm_out_weight=norm_out_weight, norm_out_bias=norm_out_bias,
        p_out_weight=p_out_weight, p_out_bias=p_out_bias,
        g_out_weight=g_out_weight, g_out_bias=g_out_bias,
    )
    C, Ch = x.shape[-1], p_in_weight.shape[0] // 2
    if wide_supported(x, p_in_weight):  # widths above the fused kernels' tiles
        return trimul_wide_hip(x, direction, mask, eps, weights)
    if C % 32 or Ch % 32:  # zero-padded copies; the LayerNorms average over the real widths
        xp, wp, _, _ = _pad_channels(x, weights)
        args, keep, out, workspace, _ = build_args(xp, direction, mask, eps, wp)
        args.ln_in_channels, args.ln_out_channels = C, Ch
        run_stage("gnn_trimul_fwd", args, x.device)
        del keep, workspace
        return out[..., :C].reshape(x.shape)
    args, keep, out, workspace, _ = build_args(x, direction, mask, eps, weights)
    run_stage("gnn_trimul_fwd", args, x.device)
    del keep, workspace
    return out.reshape(x.shape)


def trimul_wide_hip(x, direction, mask, eps, weights):
    """The forward for 16-bit widths above the fused kernels' 512 (``wide_supported``), on
    this library's kernels where the math is not a plain matrix product: LN_in and LN_out on
    ``gnn_layernorm_rows`` (its wide-row kernel), the contraction on ``gnn_trimul_contract``
    (stage 2 takes any width), a / b moved into the contraction's per-channel planes and o out
    of them by ``gnn_trimul_relayout``; the three input projections as one ``[4 Ch + C, C]``
    linear and p_out on the vendor GEMM; the sigmoid gates and the mask in torch, in the
    reference's order and roundings (``_reference/trimul.py:57-97``). The pair grid is taken
    to NP = round_up(N, 32) with the pixels past N masked out (a = b = 0 there), so that the
    relayout's row blocks are the contraction's; the output is cut back to N."""
    outgoing = is_outgoing(direction)
    lead, N, C = x.shape[:-3], x.shape[-3], x.shape[-1]
    Ch = weights["p_in_weight"].shape[0] // 2
    B, NP = math.prod(lead), _pad32(N)
    dev, dt = x.device, x.dtype
    w = {k: (None if v is None else _kernel_ready(v, x)) for k, v in weights.items()}
    xb = x.reshape(B, N, N, C)
    m = (torch.ones((B, N, N), device=dev, dtype=dt) if mask is None
         else mask.to(device=dev, dtype=dt).expand(*x.shape[:-1]).reshape(B, N, N))
    if NP != N:
        xb = torch.nn.functional.pad(xb, (0, 0, 0, NP - N, 0, NP - N))
        m = torch.nn.functional.pad(m, (0, NP - N, 0, NP - N))
    M = B * NP * NP
    z = layernorm_rows_hip(_aligned(xb.reshape(M, C)), w.get("norm_in_weight"), w.get("norm_in_bias"), eps)

    def bias(key, n):
        return torch.zeros(n, device=dev, dtype=dt) if w.get(key) is None else w[key]

    lin = torch.nn.functional.linear(
        z, torch.cat([w["p_in_weight"], w["g_in_weight"], w["g_out_weight"]], 0),
        torch.cat([bias("p_in_bias", 2 * Ch), bias("g_in_bias", 2 * Ch), bias("g_out_bias", C)]))
    del z
    p = lin[:, :2 * Ch] * torch.sigmoid(lin[:, 2 * Ch:4 * Ch])
    p = _aligned(p * m.reshape(M, 1))
    gate_out = torch.sigmoid(lin[:, 4 * Ch:])
    del lin
    # a and b into the contraction's k-blocked planes (outgoing: plane row i, column k;
    # incoming: transposed per channel), then the contraction at NP. The stage-2 call reads
    # only the workspace's a / b and writes its o (x, out, the weights and the gate buffer it
    # is given are checked, not read), so the workspace stops before the gate region.
    dtc = _lib.DTYPE_CODE[dt]
    off = (ctypes.c_size_t * 4)()
    _lib.load().gnn_trimul_workspace_bytes(B, NP, C, Ch, dtc, off)
    workspace = torch.empty(off[2], device=dev, dtype=torch.uint8)
    args = _lib.TrimulArgs()
    any_ptr = w["p_in_weight"].data_ptr()
    args.x = args.out = args.gate = any_ptr
    args.p_in_w, args.g_in_w = w["p_in_weight"].data_ptr(), w["g_in_weight"].data_ptr()
    args.p_out_w, args.g_out_w = w["p_out_weight"].data_ptr(), w["g_out_weight"].data_ptr()
    args.workspace, args.workspace_bytes = workspace.data_ptr(), off[2]
    args.B, args.N, args.C, args.Ch = B, NP, C, Ch
    args.eps, args.outgoing, args.dtype = float(eps), int(outgoing), dtc
    args.precision = _lib.PRECISION_CODE["ieee"]
    for i, c0 in ((0, 0), (1, Ch)):
        relayout_hip(p, workspace[off[i]:], _lib.RELAYOUT_PIXELS_TO_BLOCKED, B, NP, Ch, src_ld=2 * Ch,
                     dst_ld=32, src_c0=c0, transposed=outgoing)
    del p
    run_stage("gnn_trimul_contract", args, dev)
    o = torch.empty((M, Ch), device=dev, dtype=dt)
    o_planes = workspace[off[3]:off[3] + B * Ch * NP * NP * o.element_size()].view(dt)
    relayout_hip(o_planes, o, _lib.RELAYOUT_PLANES_TO_PIXELS, B, NP, Ch, src_ld=NP, dst_ld=Ch)
    del workspace
    on = layernorm_rows_hip(o, w.get("norm_out_weight"), w.get("norm_out_bias"), eps)
    del o
    out = torch.nn.functional.linear(on, w["p_out_weight"], w.get("p_out_bias")) * gate_out
    out = out.view(B, NP, NP, C)
    if NP != N:
        out = out[:, :N, :N]
    return out.reshape(*lead, N, N, C)


# ------------------------------------------------------------------------------ backward
# The reference has no native trimul backward: with gradients it runs trimul_torch under
# autograd (geometric_nn_ops_torch/triangle/_trimul.py:31-36; math in
# triangle/_reference/trimul.py:57-97). trimul_bwd_hip differentiates the same math. The
# LayerNorms (forward recompute and backward, with deterministic per-workgroup weight-gradient
# partials) and the two sigmoid gates run on this library's kernels (gnn_layernorm_rows,
# gnn_trimul_gate_bwd), as do the contraction's two N^3 products per channel, on the forward's
# a and b in place (gnn_trimul_contract_bwd; fp32: gnn_rows_product), the moves between
# pixel-major tensors and per-channel planes (gnn_trimul_relayout, gnn_relayout_f32) and the
# weight gradients (gnn_rows_product); gnn_reduce_parts adds every parameter's partial sums in
# one launch. The remaining matrix products (the three input projections as one [4 Ch + C, C]
# linear, p_out, and dz) go to the vendor GEMM through torch.
# a, b and o come from the forward's workspace.

def layernorm_rows_hip(x2d, weight=None, bias=None, eps=1e-5, *, dy=None, partials=False, raw=False):
    """Row LayerNorm of ``x2d`` ``[R, K]`` (columns contiguous): ``LN(x)`` when ``dy`` is
    None, else ``dx`` and, with ``partials``, ``(dweight, dbias)`` in fp32 summed over the
    kernel's per-workgroup partial rows (``raw``: those rows themselves, ``[parts, 2, K]``)."""
    lib = _lib.load()
    R, K = x2d.shape
    out = torch.empty((R, K), device=x2d.device, dtype=x2d.dtype)
    a = _lib.LayerNormArgs()
    a.x, a.out = x2d.data_ptr(), out.data_ptr()
    a.weight = None if weight is None else weight.data_ptr()
    a.rows, a.K = R, K
    a.x_stride, a.out_stride = x2d.stride(0), out.stride(0)
    a.eps, a.dtype = float(eps), _lib.DTYPE_CODE[x2d.dtype]
    part = None
    if dy is None:
        a.bias = None if bias is None else bias.data_ptr()
    else:
        a.dy, a.dy_stride = dy.data_ptr(), dy.stride(0)
        if partials:
            part = torch.empty((lib.gnn_layernorm_partials(R, K), 2, K), device=x2d.device,
                               dtype=torch.float32)
            a.partial = part.data_ptr()
    _lib.call("gnn_layernorm_rows", a, x2d.device)
    if part is None:
        return out
    if raw:
        return out, part
    sums = part.sum(0)
    return out, sums[0], sums[1]


def gate_bwd_hip(grad, value, gate_pre, mask_rows=None, *, d_value=None, d_gate_pre=None, sums=False,
                 gate_is_sigmoid=False, raw=False):
    """Backward of ``value * sigmoid(gate_pre) * mask_rows[:, None]`` for ``[R, K]`` row
    views (columns contiguous); writes into ``d_value`` / ``d_gate_pre`` (allocated when
    None) and returns them, followed with ``sums`` by their fp32 column sums (the bias
    gradients of the layers behind value and gate_pre), from the kernel's per-workgroup
    partial rows where K allows it (``raw``: followed by the partial rows, ``[parts, 2, K]``). With
    ``gate_is_sigmoid`` the third operand is the saved ``sigmoid(gate_pre)`` itself."""
    lib = _lib.load()
    R, K = grad.shape
    if d_value is None:
        d_value = torch.empty((R, K), device=grad.device, dtype=grad.dtype)
    if d_gate_pre is None:
        d_gate_pre = torch.empty((R, K), device=grad.device, dtype=grad.dtype)
    nparts = lib.gnn_gate_bwd_partials(R, K) if sums else 0
    part = torch.empty((nparts, 2, K), device=grad.device, dtype=torch.float32) if nparts else None
    a = _lib.GateBwdArgs()
    a.partial = None if part is None else part.data_ptr()
    a.grad, a.value, a.gate_pre = grad.data_ptr(), value.data_ptr(), gate_pre.data_ptr()
    a.d_value, a.d_gate_pre = d_value.data_ptr(), d_gate_pre.data_ptr()
    if mask_rows is not None:
        a.mask, a.mask_stride = mask_rows.data_ptr(), mask_rows.stride(0)
    a.rows, a.K = R, K
    a.grad_stride, a.value_stride, a.gate_stride = grad.stride(0), value.stride(0), gate_pre.stride(0)
    a.dv_stride, a.dg_stride = d_value.stride(0), d_gate_pre.stride(0)
    a.dtype = _lib.DTYPE_CODE[grad.dtype]
    a.gate_is_sigmoid = int(gate_is_sigmoid)
    _lib.call("gnn_trimul_gate_bwd", a, grad.device)
    if not sums:
        return d_value, d_gate_pre
    if raw:
        if part is None:
            part = torch.stack((d_value.sum(0, dtype=torch.float32), d_gate_pre.sum(0, dtype=torch.float32)))[None]
        return d_value, d_gate_pre, part
    if part is not None:
        colsum = part.sum(0)
        return d_value, d_gate_pre, colsum[0], colsum[1]
    return (d_value, d_gate_pre, d_value.sum(0, dtype=torch.float32), d_gate_pre.sum(0, dtype=torch.float32))


def proj_bwd_supported(dtype, C, Ch):
    """Whether gnn_trimul_proj_bwd covers these widths (16-bit, C in {64, 128}, 2 Ch <= 256)."""
    return dtype in (torch.bfloat16, torch.float16) and C in (64, 128) and 16 <= Ch <= 128 and (2 * Ch) % 32 == 0


def proj_bwd_hip(xk, w, mask_rows, dab, d_p, d_g, eps):
    """gnn_trimul_proj_bwd: z = LN_in(x) and the backward of a|b = p * sigmoid(g) * mask
    with p / g recomputed on the fly; writes ``d_p`` / ``d_g`` (row views) and returns ``z`` and the
    per-workgroup rows ``[parts, 2, 2 Ch]`` (fp32) whose sums are the p_in and g_in bias gradients."""
    lib = _lib.load()
    M, C = xk.shape
    Ch = w["p_in_weight"].shape[0] // 2
    z = torch.empty((M, C), device=xk.device, dtype=xk.dtype)
    part = torch.empty((lib.gnn_trimul_proj_bwd_partials(M), 2, 2 * Ch), device=xk.device, dtype=torch.float32)
    w = {k: (None if v is None else _kernel_ready(v, xk)) for k, v in w.items()}
    a = _lib.TrimulProjBwdArgs()
    a.x, a.z, a.partial = xk.data_ptr(), z.data_ptr(), part.data_ptr()
    ptr = lambda t: None if t is None else t.data_ptr()  # noqa: E731
    a.ln_w, a.ln_b = ptr(w.get("norm_in_weight")), ptr(w.get("norm_in_bias"))
    a.p_in_w, a.p_in_b = w["p_in_weight"].data_ptr(), ptr(w.get("p_in_bias"))
    a.g_in_w, a.g_in_b = w["g_in_weight"].data_ptr(), ptr(w.get("g_in_bias"))
    if mask_rows is not None:
        a.mask, a.mask_stride = mask_rows.data_ptr(), mask_rows.stride(0)
    a.d_ab, a.d_p, a.d_g = dab.data_ptr(), d_p.data_ptr(), d_g.data_ptr()
    a.rows, a.C, a.Ch = M, C, Ch
    a.x_ld, a.dab_ld, a.dl_ld = xk.stride(0), dab.stride(0), d_p.stride(0)
    a.eps, a.dtype = float(eps), _lib.DTYPE_CODE[xk.dtype]
    _lib.call("gnn_trimul_proj_bwd", a, xk.device)
    return z, part


def out_bwd_supported(dtype, C, Ch):
    """Whether gnn_trimul_out_bwd covers these widths (16-bit, C in {64, 128}, c_hidden in {32, 64, 128})."""
    return dtype in (torch.bfloat16, torch.float16) and C in (64, 128) and Ch in (32, 64, 128)


def out_bwd_hip(o_cm, w, gate_pm, dout2, d_go, B, N, eps):
    """gnn_trimul_out_bwd: from the channel-major ``o_cm`` [B, Ch, N, NP], the saved gate and
    the output gradient (pixel-major rows), ``(on, dy, d_o, part)`` with on = LN_out(o), dy the
    gradient of p_out's output, d_o that of o (pixel-major) and ``part`` ``[parts, 4, 128]`` fp32 rows
    whose sums are the p_out / g_out bias and the LN_out weight / bias gradients, each from column
    0; d(g_out pre-activation) goes into ``d_go`` (a row view)."""
    lib = _lib.load()
    M, C = dout2.shape
    Ch = o_cm.shape[1]
    dev, dt = dout2.device, dout2.dtype
    on = torch.empty((M, Ch), device=dev, dtype=dt)
    dy = torch.empty((M, C), device=dev, dtype=dt)
    d_o = torch.empty((M, Ch), device=dev, dtype=dt)
    part = torch.empty((lib.gnn_trimul_out_bwd_partials(B, N), 4, 128), device=dev, dtype=torch.float32)
    w = {k: (None if v is None else _kernel_ready(v, dout2)) for k, v in w.items()}
    ptr = lambda t: None if t is None else t.data_ptr()  # noqa: E731
    a = _lib.TrimulOutBwdArgs()
    a.o, a.gate, a.dout = o_cm.data_ptr(), gate_pm.data_ptr(), dout2.data_ptr()
    a.ln_w, a.ln_b = ptr(w.get("norm_out_weight")), ptr(w.get("norm_out_bias"))
    a.p_out_w, a.p_out_b = w["p_out_weight"].data_ptr(), ptr(w.get("p_out_bias"))
    a.on, a.dy, a.d_go, a.d_o, a.partial = on.data_ptr(), dy.data_ptr(), d_go.data_ptr(), d_o.data_ptr(), part.data_ptr()
    a.B, a.N, a.C, a.Ch = B, N, C, Ch
    a.dgo_ld = d_go.stride(0)
    a.eps, a.dtype = float(eps), _lib.DTYPE_CODE[dt]
    _lib.call("gnn_trimul_out_bwd", a, dev)
    return on, dy, d_o, part


def rows_products_hip(pairs, slice_rows=0):
    """Partials of ``d^T t`` for up to ``_lib.ROWS_PRODUCT_MAX`` pairs of ``[M, O]`` / ``[M, I]`` row
    views over the same M rows (columns contiguous): one fp32 ``[slices, O, I]`` tensor per pair,
    to be added with ``reduce_parts_hip``; with ``slice_rows``, slice s is the product over rows
    ``s slice_rows .. (s + 1) slice_rows``."""
    lib = _lib.load()
    a = _lib.RowsProductArgs()
    d0 = pairs[0][0]
    a.rows, a.slice_rows, a.count, a.dtype = d0.shape[0], slice_rows, len(pairs), _lib.DTYPE_CODE[d0.dtype]
    for p, (d, t) in zip(a.p, pairs):
        p.d, p.t, p.d_ld, p.t_ld, p.O, p.I = (d.data_ptr(), t.data_ptr(), d.stride(0), t.stride(0), d.shape[1],
                                              t.shape[1])
    slices = lib.gnn_rows_product_slices(ctypes.byref(a))
    if slices and not slice_rows:  # that count depends on the device current here, the launch must not: pin its split
        a.slice_rows = (-(-a.rows // slices) + 31) // 32 * 32
    parts = [torch.empty((slices, d.shape[1], t.shape[1]), device=d0.device, dtype=torch.float32) for d, t in pairs]
    for p, part in zip(a.p, parts):
        p.partial = part.data_ptr()
    _lib.call("gnn_rows_product", a, d0.device)
    return parts


def reduce_parts_hip(segments, device):
    """Ordered sums of partial results in one launch: ``segments`` are ``(src, offset, n, dst)`` with
    ``src`` an fp32 ``[parts, ...]`` tensor, the segment being elements ``offset .. offset + n`` of
    each part, and ``dst`` a contiguous tensor of n elements."""
    a = _lib.ReduceArgs()
    a.count = len(segments)
    for g, (src, offset, n, dst) in zip(a.seg, segments):
        g.src, g.dst = src.data_ptr() + 4 * offset, dst.data_ptr()
        g.parts, g.stride, g.n, g.dtype = src.shape[0], src.stride(0), n, _lib.DTYPE_CODE[dst.dtype]
    _lib.call("gnn_reduce_parts", a, device)


def relayout_hip(src, dst, mode, B, N, Ch, *, src_ld, dst_ld, src_c0=0, dst_c0=0, transposed=False, plane_rows=0):
    """gnn_trimul_relayout (16-bit) or gnn_relayout_f32 between pixel-major rows and per-channel
    planes."""
    a = _lib.TrimulRelayoutArgs()
    a.src, a.dst = src.data_ptr(), dst.data_ptr()
    a.B, a.N, a.Ch = B, N, Ch
    a.src_ld, a.dst_ld, a.src_c0, a.dst_c0 = src_ld, dst_ld, src_c0, dst_c0
    a.mode, a.transposed, a.dtype, a.plane_rows = mode, int(transposed), _lib.DTYPE_CODE[src.dtype], plane_rows
    _lib.call("gnn_relayout_f32" if src.dtype == torch.float32 else "gnn_trimul_relayout", a, src.device)
    return dst


def contract_bwd_hip(workspace, offsets, do_pm, B, Ch, N):
    """``(dA, dB)`` ``[B, Ch, N, NP]`` of the contraction o_c = A_c B_c^T for 16-bit types:
    ``dA_c = dO_c B_c`` and ``dB_c = dO_c^T A_c``, with A and B read in place from the
    forward's ``workspace`` and dO given pixel-major, ``do_pm`` ``[B N N, Ch]`` (plane c of
    batch b: dO_c[i, j] = do_pm[(b, i, j), c])."""
    dt, dev = do_pm.dtype, do_pm.device
    NP = (N + 31) // 32 * 32
    do_i = torch.empty((B, Ch, NP // 32, NP, 32), device=dev, dtype=dt)  # [i / 32][j][i % 32]
    do_j = torch.empty_like(do_i)                                       # [j / 32][i][j % 32]
    for t, transposed in ((do_i, False), (do_j, True)):
        relayout_hip(do_pm, t, _lib.RELAYOUT_PIXELS_TO_BLOCKED, B, N, Ch, src_ld=do_pm.stride(0), dst_ld=32,
                     transposed=transposed)
    da = torch.empty((B, Ch, N, NP), device=dev, dtype=dt)
    db = torch.empty_like(da)
    a = _lib.TrimulContractBwdArgs()
    a.a = workspace.data_ptr() + offsets[0]
    a.b = workspace.data_ptr() + offsets[1]
    a.do_i, a.do_j, a.da, a.db = do_i.data_ptr(), do_j.data_ptr(), da.data_ptr(), db.data_ptr()
    a.planes, a.N, a.dtype = B * Ch, N, _lib.DTYPE_CODE[dt]
    _lib.call("gnn_trimul_contract_bwd", a, dev)
    return da, db


def contract_bwd_f32_hip(workspace, offsets, do_pm, B, Ch, N):
    """``contract_bwd_hip`` for fp32: ``(dA, dB)`` ``[B, Ch, N8, N8]`` (N8 = round_up(N, 8); rows and
    columns past N hold nothing), as batches of products over the rows of the planes, with A and B
    ``[N, NP]`` read in place and dO brought into planes in both orientations:
    ``dA[i][k] = sum_j dO[i][j] B[j][k]``, ``dB[j][k] = sum_i dO[i][j] A[i][k]``."""
    dev, planes, NP, N8 = do_pm.device, B * Ch, _pad32(N), (N + 7) // 8 * 8
    d = torch.empty((2, planes * N, N8), device=dev, dtype=torch.float32)
    for t, transposed in ((d[0], False), (d[1], True)):
        relayout_hip(do_pm, t, _lib.RELAYOUT_PIXELS_TO_PLANES, B, N, Ch, src_ld=do_pm.stride(0), dst_ld=N8,
                     transposed=transposed)
    ab = [workspace[o:o + planes * N * NP * 4].view(torch.float32).view(planes * N, NP)[:, :N8] for o in offsets[:2]]
    return rows_products_hip([(d[1], ab[1]), (d[0], ab[0])], slice_rows=N)


def trimul_bwd_hip(x, direction, mask, eps, weights, workspace, offsets, dout, gate=None, fused=None):
    """Gradients ``(dx, {weight name: grad or None})`` of the triangle multiplicative update
    given the forward's ``workspace`` / ``offsets`` (a, b, o), its output gate ``gate``
    (sigmoid(g_out(z)), or None) and the output gradient. With the saved gate, 16-bit inputs
    and widths gnn_trimul_proj_bwd covers (``fused`` None or True), the input side runs as
    that one kernel: the output gate's backward uses the saved gate, and z, the recomputed
    input projections and their gate backward never pass through a [M, 4 Ch + C] tensor;
    otherwise LN_in(x) and the three input projections are recomputed as one linear."""
    outgoing = is_outgoing(direction)
    N, C = x.shape[-2], x.shape[-1]
    lead = x.shape[:-3]
    B = math.prod(lead)
    M = B * N * N
    dt = x.dtype
    dev = x.device
    w = {k: (None if v is None else v.to(device=dev, dtype=dt)) for k, v in weights.items()}
    Ch = w["p_in_weight"].shape[0] // 2
    NP = (N + 31) // 32 * 32

    def zeros_or(t, n):
        return t if t is not None else torch.zeros(n, device=dev, dtype=dt)

    use_fused = gate is not None and proj_bwd_supported(dt, C, Ch) and fused is not False
    if fused and not use_fused:
        raise ValueError("trimul_bwd_hip: the fused input-side backward does not cover this call")
    xk = _aligned(x.reshape(M, C))
    dout2 = _aligned(dout.reshape(M, C).to(dt))
    # the three projections of z as one linear: [p_in (2 Ch); g_in (2 Ch); g_out (C)]
    wcat = torch.cat([w["p_in_weight"], w["g_in_weight"], w["g_out_weight"]], 0)
    if use_fused:
        gate_pm = _aligned(gate.reshape(M, C))
    else:
        z = layernorm_rows_hip(xk, w["norm_in_weight"], w["norm_in_bias"], eps)
        bcat = torch.cat([zeros_or(w["p_in_bias"], 2 * Ch), zeros_or(w["g_in_bias"], 2 * Ch),
                          zeros_or(w["g_out_bias"], C)])
        lin = torch.nn.functional.linear(z, wcat, bcat)  # [M, 4 Ch + C]
        p, gpre, gopre = lin[:, :2 * Ch], lin[:, 2 * Ch:4 * Ch], lin[:, 4 * Ch:]
    # output stage: out = p_out(LN_out(o)) * sigmoid(gopre)
    o_cm = workspace[offsets[3]:offsets[3] + B * Ch * N * NP * x.element_size()].view(dt).view(B, Ch, N, NP)
    dlin = torch.empty((M, 4 * Ch + C), device=dev, dtype=dt)
    grads = {}
    if use_fused and out_bwd_supported(dt, C, Ch):
        # the output side in one kernel, from the channel-major o and the saved gate
        on, dy, do_pm, part = out_bwd_hip(o_cm, w, gate_pm, dout2, dlin[:, 4 * Ch:], B, N, eps)
        for i, key in enumerate(("p_out_bias", "g_out_bias", "norm_out_weight", "norm_out_bias")):
            grads[key] = part, 128 * i
    else:
        o_pm = relayout_hip(o_cm, torch.empty((M, Ch), device=dev, dtype=dt), _lib.RELAYOUT_PLANES_TO_PIXELS,
                            B, N, Ch, src_ld=NP, dst_ld=Ch)
        on = layernorm_rows_hip(o_pm, w["norm_out_weight"], w["norm_out_bias"], eps)
        y = torch.nn.functional.linear(on, w["p_out_weight"], w["p_out_bias"])
        if use_fused:  # torch's sigmoid backward reads the saved output as well
            dy, _, part = gate_bwd_hip(dout2, y, gate_pm, d_gate_pre=dlin[:, 4 * Ch:], sums=True,
                                       gate_is_sigmoid=True, raw=True)
        else:
            dy, _, part = gate_bwd_hip(dout2, y, gopre, d_gate_pre=dlin[:, 4 * Ch:], sums=True, raw=True)
        grads["p_out_bias"], grads["g_out_bias"] = (part, 0), (part, C)
        don = dy @ w["p_out_weight"]
        do_pm, part = layernorm_rows_hip(o_pm, w["norm_out_weight"], eps=eps, dy=don, partials=True, raw=True)
        grads["norm_out_weight"], grads["norm_out_bias"] = (part, 0), (part, Ch)
    # contraction: o_c = A_c B_c^T per (batch, channel) plane; dO_c[i, j] is pixel (i, j).
    # dA / dB planes go back to the pixel layout of a / b (plane [i, k] is pixel (i, k)
    # outgoing, (k, i) incoming), into the two halves of dab.
    dab = torch.empty((M, 2 * Ch), device=dev, dtype=dt)
    contract = contract_bwd_f32_hip if dt == torch.float32 else contract_bwd_hip
    dA, dB = contract(workspace, offsets, do_pm, B, Ch, N)
    for t, c0 in ((dA, 0), (dB, Ch)):
        relayout_hip(t, dab, _lib.RELAYOUT_PLANES_TO_PIXELS, B, N, Ch, src_ld=t.shape[-1], dst_ld=2 * Ch, dst_c0=c0,
                     transposed=not outgoing, plane_rows=t.shape[-2])
    m_rows = None
    if mask is not None:
        m_rows = mask.to(device=dev, dtype=dt).expand(*x.shape[:-1]).reshape(M).contiguous()
    if use_fused:
        z, part = proj_bwd_hip(xk, w, m_rows, dab, dlin[:, :2 * Ch], dlin[:, 2 * Ch:4 * Ch], eps)
    else:
        _, _, part = gate_bwd_hip(dab, p, gpre, m_rows, d_value=dlin[:, :2 * Ch],
                                  d_gate_pre=dlin[:, 2 * Ch:4 * Ch], sums=True, raw=True)
    grads["p_in_bias"], grads["g_in_bias"] = (part, 0), (part, 2 * Ch)
    dwcat, dwout = rows_products_hip([(dlin, z), (dy, on)])
    grads["p_in_weight"], grads["g_in_weight"], grads["g_out_weight"] = (
        (dwcat, 0), (dwcat, 2 * Ch * C), (dwcat, 4 * Ch * C))
    grads["p_out_weight"] = dwout, 0
    dz = dlin @ wcat
    dx, part = layernorm_rows_hip(xk, w["norm_in_weight"], eps=eps, dy=dz, partials=True, raw=True)
    grads["norm_in_weight"], grads["norm_in_bias"] = (part, 0), (part, C)
    # every parameter gradient is a sum of fp32 partials here: one launch adds and converts them
    # all, into one flat tensor per parameter dtype
    keys = [k for k in _WEIGHT_KEYS if weights.get(k) is not None]
    out = dict.fromkeys(_WEIGHT_KEYS)
    segments = []
    for pdt in {weights[k].dtype for k in keys}:
        mine = [k for k in keys if weights[k].dtype == pdt]
        sizes = [weights[k].numel() for k in mine]
        kdt = pdt if pdt in _lib.DTYPE_CODE else torch.float32
        views = torch.empty(sum(sizes), device=dev, dtype=kdt).split(sizes)
        segments += [(*grads[k], n, v) for k, n, v in zip(mine, sizes, views)]
        for k, v in zip(mine, views):
            out[k] = v.view(weights[k].shape)
    reduce_parts_hip(segments, dev)
    for k in keys:
        if out[k].dtype != weights[k].dtype:
            out[k] = out[k].to(weights[k].dtype)
    return dx.reshape(x.shape), out
