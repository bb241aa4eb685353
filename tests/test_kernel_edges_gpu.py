"""Kernels at the sizes where their tiles, remainders and dispatch lines lie, against the fp64
oracle. Tolerances: one rounding of a result costs at most half an ulp (bf16 2^-9, fp16 2^-12,
fp32 2^-24 relative), and the bounds below allow for the two or three roundings a value passes."""

import pytest
import torch

from helpers import gen, np_weights, pair_input, to_np, trimul_weights
from oracle import triangle_oracle as O

pytestmark = pytest.mark.gpu

DEV = "cuda"
DEV_T = torch.device(DEV)
DTYPES = pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32], ids=["bf16", "fp16", "fp32"])
TOL = {torch.bfloat16: 1e-2, torch.float16: 2e-3, torch.float32: 1e-5}


def _misaligned(t):
    """A contiguous copy of t whose storage starts one element past a 16-byte boundary."""
    buf = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)
    out = buf[1:].view(t.shape)
    out.copy_(t)
    assert out.data_ptr() % 16 != 0 and out.is_contiguous()
    return out


# ------------------------------------------------------------------ pair-bias projection
@DTYPES
@pytest.mark.parametrize(("Zc", "H", "U", "V"), [(8, 1, 1, 1), (24, 3, 5, 7), (64, 32, 4, 16), (72, 33, 3, 43),
                                                 (128, 16, 31, 33), (200, 40, 2, 65), (256, 4, 9, 8)])
def test_pair_bias_projection_tiles(Zc, H, U, V, dtype):
    """Channel counts below, at and past each unrolled width, heads past the 32 of one MFMA tile,
    pixel counts that leave a tile of 32 and a workgroup part empty; weights and gamma off a
    16-byte boundary; no gamma."""
    from geometric_nn_ops_torch.triangle._kernels.attention_pair_bias import pair_bias_projection_hip

    g = gen(100 + Zc)
    z = torch.randn(2, U, V, Zc, generator=g).to(dtype)
    w = (torch.randn(H, Zc, generator=g) * Zc ** -0.5).to(dtype)
    lw = (1.0 + 0.1 * torch.randn(Zc, generator=g)).to(dtype)
    want = O.pair_bias_projection(to_np(z), to_np(lw), to_np(w), 1e-5)
    for place in (lambda t: t.to(DEV), lambda t: _misaligned(t.to(DEV))):
        got = pair_bias_projection_hip(z.to(DEV), place(lw), place(w), 1e-5)
        assert got.shape == (2, H, U, V)
        assert O.rel_fro(to_np(got), want) <= TOL[dtype]
    got = pair_bias_projection_hip(z.to(DEV), None, w.to(DEV), 1e-5)
    want = O.pair_bias_projection(to_np(z), to_np(torch.ones(Zc)), to_np(w), 1e-5)
    assert O.rel_fro(to_np(got), want) <= TOL[dtype]


@DTYPES
@pytest.mark.parametrize("V", [128, 129, 256, 257])
@pytest.mark.parametrize(("Zc", "heads"), [(8, (1, 2, 3, 6, 7, 8, 9)), (64, (1, 3, 4)), (72, (4, 5, 6, 7, 10, 11, 16, 17)),
                                           (256, (3, 4, 6, 7, 10, 11, 12, 13, 16, 17))])
def test_pair_bias_head_counts(Zc, heads, V, dtype):
    """Head counts on both sides of where the dot products give way to the matrix unit, at 16384 and
    32768 pixels, where those change, and one row past them."""
    from geometric_nn_ops_torch.triangle._kernels.attention_pair_bias import pair_bias_projection_hip

    g = torch.Generator(device=DEV).manual_seed(Zc)
    z = torch.randn(2, 64, V, Zc, generator=g, device=DEV).to(dtype)
    lw = (1.0 + 0.1 * torch.randn(Zc, generator=g, device=DEV)).to(dtype)
    zn = torch.nn.functional.layer_norm(z.double(), (Zc,), lw.double())
    for H in heads:
        w = (torch.randn(H, Zc, generator=g, device=DEV) * Zc ** -0.5).to(dtype)
        want = torch.nn.functional.linear(zn, w.double()).permute(0, 3, 1, 2)
        got = pair_bias_projection_hip(z, lw, w, 1e-5)
        assert got.shape == want.shape
        assert (got.double() - want).norm() <= TOL[dtype] * want.norm(), H


@pytest.mark.parametrize("Zc", [64, 128, 256])
def test_fp32_pair_bias_sums(Zc):
    """A running sum of m products of random signs is off by about 2^-24 sqrt(m / 11) of itself: sums of
    8 or 16 channels added as a tree stay near the 0.9e-7 that the LayerNorm alone costs, a single one
    comes to 1.5e-7 (64 channels), 2.1e-7 (128) and 2.9e-7 (256)."""
    from geometric_nn_ops_torch.triangle._kernels.attention_pair_bias import pair_bias_projection_hip

    g = torch.Generator(device=DEV).manual_seed(Zc)
    z = torch.randn(1, 96, 96, Zc, generator=g, device=DEV)
    w = torch.randn(24, Zc, generator=g, device=DEV) * Zc ** -0.5  # heads for the matrix unit
    lw = 1.0 + 0.1 * torch.randn(Zc, generator=g, device=DEV)
    zn = torch.nn.functional.layer_norm(z.double(), (Zc,), lw.double())
    want = torch.nn.functional.linear(zn, w.double()).permute(0, 3, 1, 2)
    got = pair_bias_projection_hip(z, lw, w, 1e-5)
    assert (got.double() - want).norm() <= 1.3e-7 * want.norm()


@DTYPES
@pytest.mark.parametrize(("M", "Cs", "D", "Co"), [(1, 32, 128, 128), (33, 64, 160, 32), (31, 384, 384, 384),
                                                  (40, 96, 544, 576), (32, 1024, 1024, 64)])
def test_gate_out_widths(M, Cs, D, Co, dtype):
    """Widths at and past one pass of four waves and of the wide workgroup, and the largest tiles,
    which leave no LDS for the wide output pass."""
    from geometric_nn_ops_torch.triangle._kernels.attention_pair_bias import gate_out_hip

    if dtype == torch.float32 and Cs + D > 1024:
        Cs = D = 512
    g = gen(200 + D)
    r = lambda *shape, scale=1.0: (torch.randn(*shape, generator=g) * scale).to(dtype)  # noqa: E731
    s, o, gw, ow = r(M, Cs), r(M, D), r(D, Cs, scale=Cs ** -0.5), r(Co, D, scale=D ** -0.5)
    gb, ob = r(D, scale=0.3), r(Co, scale=0.3)
    got = gate_out_hip(*(t.to(DEV) for t in (s, o, gw, gb, ow, ob)))
    q = to_np
    want = O.linear(q(o) * O.sigmoid(O.linear(q(s), q(gw), q(gb))), q(ow), q(ob))
    assert O.rel_fro(to_np(got), want) <= TOL[dtype]


# --------------------------------------------------------------- multiplicative update, forward
def _trimul_forward_error(N, C, Ch, dtype, direction, B=1):
    """Worst relative error of the forward over sampled rows and columns (first, last and the ones
    at tile edges)."""
    from geometric_nn_ops_torch.triangle import triangle_multiplicative_update

    w = trimul_weights(C, Ch, dtype, seed=N, biases=True, ln_random=True)
    x, mask = pair_input(B, N, C, dtype, seed=N + 1)
    with torch.no_grad():
        got = triangle_multiplicative_update(x.to(DEV), direction, mask.to(DEV), **{k: v.to(DEV) for k, v in w.items()})
    at = sorted({i for i in (0, 31, 32, 63, 64, 127, 128, 191, N - 1) if i < N})
    want = O.trimul_grid(to_np(x), direction, to_np(mask), at, at, **np_weights(w))
    return O.rel_fro(to_np(got[:, at][:, :, at]), want)


@pytest.mark.parametrize("direction", ["outgoing", "incoming"])
@pytest.mark.parametrize("N", [1, 33, 64, 65, 129, 192, 193, 449])
def test_fp32_contraction_tiles(N, direction):
    """Both tile edges of the full-precision contraction, at and past their multiples."""
    assert _trimul_forward_error(N, 32, 32, torch.float32, direction) <= TOL[torch.float32]


@pytest.mark.parametrize("precision", ["ieee", "bf16x3"])
@pytest.mark.parametrize("N", [1, 33, 64, 131, 250])
def test_fp32_contraction_ignores_the_padding(N, precision):
    """Stage 2 by itself: fp32 a and b are specified up to column N only (16-bit types have zeros
    there), on tiles of 64 and of 128."""
    from geometric_nn_ops_torch import _lib
    from geometric_nn_ops_torch.triangle._kernels import trimul as K

    C, Ch = 32, 32
    x, _ = pair_input(1, N, C, torch.float32, seed=N, device=DEV)
    args, _keep, _out, workspace, offsets = K.build_args(x, "outgoing", None, 1e-5,
                                                         trimul_weights(C, Ch, torch.float32, device=DEV))
    args.precision = _lib.PRECISION_CODE[precision]
    NP = (N + 31) // 32 * 32
    workspace.view(torch.float32).fill_(float("nan"))
    a, b, o = (workspace[offsets[i]:offsets[i] + 4 * Ch * N * NP].view(torch.float32).view(Ch, N, NP)
               for i in (0, 1, 3))
    g = gen(N)
    for t in (a, b):
        t[..., :N] = torch.randn(Ch, N, N, generator=g).to(DEV)
    K.run_stage("gnn_trimul_contract", args, DEV_T)
    want = a[..., :N].double() @ b[..., :N].double().transpose(1, 2).contiguous()
    assert O.rel_fro(to_np(o[..., :N]), to_np(want)) <= (1e-5 if precision == "ieee" else 5e-5)


@pytest.mark.parametrize("direction", ["outgoing", "incoming"])
@pytest.mark.parametrize(("dtype", "N", "C", "Ch", "B"), [
    # one to four workgroups on a tile (256 compute units over N ceil(N / 64) B tiles)
    (torch.float32, 3, 128, 128, 1), (torch.float32, 64, 128, 128, 1), (torch.float32, 45, 128, 128, 2),
    (torch.float32, 40, 256, 96, 1), (torch.float32, 64, 64, 32, 1), (torch.bfloat16, 33, 256, 128, 1),
    (torch.bfloat16, 64, 96, 160, 1), (torch.float16, 63, 32, 256, 2),
    # full-precision weights held in registers: both widths, c_hidden below c_z, row tails
    (torch.float32, 130, 128, 128, 1), (torch.float32, 91, 128, 128, 2), (torch.float32, 131, 128, 64, 1),
    (torch.float32, 135, 64, 128, 1)])
def test_projection_dispatch(dtype, N, C, Ch, B, direction):
    assert _trimul_forward_error(N, C, Ch, dtype, direction, B) <= TOL[dtype]


@pytest.mark.parametrize(("N", "C", "Ch", "B"), [(1, 128, 128, 1), (32, 128, 128, 1), (33, 128, 128, 3),
                                                 (97, 32, 96, 1), (127, 128, 128, 1), (128, 128, 128, 1),
                                                 (65, 256, 32, 1), (31, 160, 256, 2), (85, 64, 64, 1), (86, 64, 64, 1),
                                                 (128, 64, 64, 2)])
def test_fp32_output_tiles(N, C, Ch, B):
    """Output tiles of 32 pixels (up to 256 of them) and 64, their row tails, and more output channels
    than one pass."""
    assert _trimul_forward_error(N, C, Ch, torch.float32, "outgoing", B) <= TOL[torch.float32]


# ------------------------------------------------------- products over rows, ordered sums
@DTYPES
@pytest.mark.parametrize(("M", "shapes"), [
    (1, [(8, 8)]), (15, [(32, 24), (8, 136)]), (33, [(128, 128)]), (255, [(640, 128), (128, 128)]),
    (1000, [(136, 72), (64, 256), (8, 8), (192, 64)]), (40401, [(192, 64), (64, 32)])])
def test_rows_product(M, shapes, dtype):
    """Rows short of a stage and of a slice, output blocks part empty, one to four products a launch,
    operands inside wider rows. The products are exact in fp32, so the sum of M of them errs by at
    most M 2^-24 of the sum of magnitudes, far below the bound for these sizes (random signs)."""
    from geometric_nn_ops_torch.triangle._kernels.trimul import reduce_parts_hip, rows_products_hip

    g = torch.Generator(device=DEV).manual_seed(M)
    pairs = []
    for O_, I_ in shapes:
        d = torch.randn(M, O_ + 16, generator=g, device=DEV).to(dtype)
        t = torch.randn(M, I_ + 8, generator=g, device=DEV).to(dtype)
        pairs.append((d[:, 16:], t[:, :I_]) if dtype != torch.float32 else (d[:, 8:O_ + 8], t[:, 8:]))
    parts = rows_products_hip(pairs)
    sums = [torch.empty(d.shape[1] * t.shape[1], device=DEV) for d, t in pairs]
    reduce_parts_hip([(p, 0, s.numel(), s) for p, s in zip(parts, sums)], DEV_T)
    for (d, t), s in zip(pairs, sums):
        want = d.double().t().contiguous() @ t.double()
        assert (s.view_as(want).double() - want).norm() <= 2e-6 * want.norm()


def test_rows_product_ignores_what_lies_past_the_rows():
    """The rows behind the last one (of a larger tensor) hold NaN; the result does not."""
    from geometric_nn_ops_torch.triangle._kernels.trimul import rows_products_hip

    for dtype in TOL:
        d, t = (torch.randn(64, 128, device=DEV).to(dtype) for _ in range(2))
        d[37:], t[37:] = float("nan"), float("nan")
        (part,) = rows_products_hip([(d[:37], t[:37])])
        want = d[:37].double().t().contiguous() @ t[:37].double()
        assert (part.sum(0).double() - want).norm() <= 2e-6 * want.norm()


@DTYPES
@pytest.mark.parametrize(("parts", "n"), [(1, 1), (7, 300), (128, 257), (129, 9), (1024, 31)])
def test_reduce_parts(parts, n, dtype):
    """Both ways of adding (up to 128 parts a thread adds an element alone), element counts that leave a
    block part empty, a segment inside wider parts, results in each dtype, the same bits twice."""
    from geometric_nn_ops_torch.triangle._kernels.trimul import reduce_parts_hip

    src = torch.randn(parts, n + 5, device=DEV)
    out = [torch.empty(n, device=DEV, dtype=dtype) for _ in range(2)]
    for o in out:
        reduce_parts_hip([(src, 3, n, o)], DEV_T)
    want = src[:, 3:3 + n].double().sum(0)
    assert torch.equal(out[0], out[1])
    assert (out[0].double() - want).norm() <= TOL[dtype] * want.norm()


def test_fp32_sums_are_short():
    """How far sums of random signs end from 64 bits (2^-24 sqrt(m / 11) for a running sum of m): 128 partial
    results as eight sums and a tree, 0.9e-7 (one sum 2.0e-7); products over 128 rows as two sums,
    1.47e-7 (one sum 2.04e-7)."""
    from geometric_nn_ops_torch.triangle._kernels.trimul import reduce_parts_hip, rows_products_hip

    g = torch.Generator(device=DEV).manual_seed(1)
    src = torch.randn(128, 20000, generator=g, device=DEV)
    out = torch.empty(20000, device=DEV)
    reduce_parts_hip([(src, 0, 20000, out)], DEV_T)
    want = src.double().sum(0)
    assert (out.double() - want).norm() <= 1.2e-7 * want.norm()
    d, t = (torch.randn(4096, n, generator=g, device=DEV) for n in (640, 128))
    (part,) = rows_products_hip([(d, t)], slice_rows=128)
    want = d.double().view(32, 128, 640).transpose(1, 2).contiguous() @ t.double().view(32, 128, 128)
    assert (part.double() - want).norm() <= 1.7e-7 * want.norm()


@pytest.mark.parametrize("direction", ["outgoing", "incoming"])
@pytest.mark.parametrize(("N", "C", "Ch", "B"), [(1, 32, 32, 1), (5, 64, 32, 2), (33, 32, 96, 1), (130, 64, 64, 1)])
def test_fp32_backward_planes(N, C, Ch, B, direction):
    """Full-precision backward: plane rows short of and past a vector, a stage and an output block,
    every gradient against the fp64 oracle."""
    from geometric_nn_ops_torch.triangle import triangle_multiplicative_update

    w = trimul_weights(C, Ch, torch.float32, seed=N, biases=True, ln_random=True)
    x, mask = pair_input(B, N, C, torch.float32, seed=N + 1)
    dout = torch.randn(x.shape, generator=gen(N + 2))
    xg = x.to(DEV).requires_grad_()
    wg = {k: v.to(DEV).requires_grad_() for k, v in w.items()}
    out = triangle_multiplicative_update(xg, direction, mask.to(DEV), **wg)
    got = torch.autograd.grad(out, [xg, *wg.values()], dout.to(DEV))
    want = O.trimul_grad(to_np(x), direction, to_np(mask), to_np(dout), **np_weights(w))
    # a LayerNorm divides by the spread of its row, at least sqrt(eps) = 3e-3: 2^-24 / 3e-3 = 2e-5
    scale = max(float(abs(want[k]).max()) for k in wg)
    assert O.rel_fro(to_np(got[0]), want["x"]) <= 1e-4
    for k, g in zip(wg, got[1:]):
        assert abs(to_np(g) - want[k]).max() <= 1e-4 * max(float(abs(want[k]).max()), 1e-2 * scale), k


# --------------------------------------------------------------------- attention, backward
def _attention_grads(q, k, v, bias, mask, dout):
    from geometric_nn_ops_torch.triangle import triangle_attention

    leaves = [t.to(DEV).requires_grad_() for t in (q, k, v)]
    leaves += [] if bias is None else [bias.to(DEV).requires_grad_()]
    out = triangle_attention(*leaves[:3], None if bias is None else leaves[3], None if mask is None else mask.to(DEV))
    return torch.autograd.grad(out, leaves, dout.to(DEV))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize(("N", "with_bias", "with_mask"), [
    (1, True, False), (31, True, True), (32, False, True), (33, True, True), (64, True, False), (65, False, False),
    (96, True, True), (255, True, True), (256, False, True), (257, True, True), (288, True, False),
    (384, True, True), (385, True, True), (500, False, True), (512, True, True), (513, True, True)])
def test_attention_backward_rows(N, with_bias, with_mask, dtype):
    """Rows at and past a block of 32, the change of waves and blocks per wave (256, 384) and the longest
    fused row (512); a key block of which a wave owns nothing (odd block counts); rows with no, some
    and only masked keys side by side (fp16 without the last, whose sentinel does not swamp its
    logits). Probabilities and their gradients are rounded once to the input dtype before each product
    and the result once: about 3 roundings of 2^-9 (bf16) or 2^-12 (fp16)."""
    S, H, D = 3, 2, 32
    g = gen(300 + N)
    q, k, v, dout = (torch.randn(1, S, N, H, D, generator=g).to(dtype) for _ in range(4))
    bias = torch.randn(1, 1, H, N, N, generator=g).to(dtype) if with_bias else None
    mask = None
    if with_mask:
        mask = torch.rand(1, S, 1, 1, N, generator=g) < 0.7
        mask[:, 0] = True
        mask[:, 1, ..., 0] = True
        mask[:, 2] = dtype == torch.float16
    got = _attention_grads(q, k, v, bias, mask, dout)
    want = O.triangle_attention_grad(*(to_np(t) for t in (q, k, v)), None if bias is None else to_np(bias),
                                     None if mask is None else mask.numpy(), D ** -0.5, to_np(dout))
    for a, b in zip(got, want):
        assert torch.isfinite(a).all()
        # a single key's logit gradients are zeros, and rounding's leftovers have no relative error
        assert O.rel_fro(to_np(a).reshape(b.shape), b) <= TOL[dtype] or abs(b).max() < 1e-12
    again = _attention_grads(q, k, v, bias, mask, dout)
    assert all(torch.equal(a, b) for a, b in zip(got, again))


@pytest.mark.parametrize(("N", "S", "D", "dtype"), [
    (70, 70, 32, torch.bfloat16), (70, 3, 64, torch.bfloat16), (521, 2, 32, torch.float16), (70, 3, 128, torch.float16),
    (70, 3, 32, torch.float32), (131, 3, 64, torch.float32)])
def test_attention_bias_padding_is_not_used(N, S, D, dtype):
    """A bias view whose padding (keys past N) holds NaN, and strided q / k / v views: the same bits
    as from packed tensors, forward and backward."""
    from geometric_nn_ops_torch.triangle import triangle_attention

    H = 2
    g = gen(7)
    q, k, v, dout = (torch.randn(1, N, S, H, D, generator=g).to(dtype) for _ in range(4))
    wide = torch.full((1, 1, H, N, (N + 15) // 8 * 8), float("nan"), dtype=dtype)
    wide[..., :N] = torch.randn(1, 1, H, N, N, generator=g)
    bias = wide.to(DEV)[..., :N].detach().requires_grad_()
    leaves = [t.to(DEV).transpose(1, 2).detach().requires_grad_() for t in (q, k, v)]
    out = triangle_attention(*leaves, bias)
    got = torch.autograd.grad(out, [*leaves, bias], dout.to(DEV).transpose(1, 2))
    want = _attention_grads(*(t.transpose(1, 2).contiguous() for t in (q, k, v)), wide[..., :N].contiguous(), None,
                            dout.transpose(1, 2).contiguous())
    assert torch.isfinite(out).all()
    for a, b in zip(got, want):
        assert torch.equal(a, b)


@pytest.mark.parametrize(("N", "D", "with_bias", "with_mask"), [
    (1, 32, True, False), (31, 32, True, True), (33, 64, True, True), (64, 32, True, True), (65, 48, True, False),
    (97, 32, False, True), (128, 64, True, True), (129, 32, True, True), (160, 32, True, True), (161, 40, True, True)])
def test_fp32_attention_partial_tiles(N, D, with_bias, with_mask):
    """fp32 rows that end within a half tile of 32, leave a half tile or a wave's 32 queries or keys
    empty, and their neighbours, with NaN in the bias's padding where the view has any. Sums of at
    most 161 products of fp32 operands against fp64: a few hundred roundings of 2^-24 at the worst."""
    from geometric_nn_ops_torch.triangle import triangle_attention

    S, H = 3, 2
    g = gen(500 + N)
    q, k, v, dout = (torch.randn(1, S, N, H, D, generator=g) for _ in range(4))
    bias = torch.randn(1, 1, H, N, N, generator=g) if with_bias else None
    mask = None
    if with_mask:
        mask = torch.rand(1, S, 1, 1, N, generator=g) < 0.7
        mask[:, 0] = True
        mask[:, 1, ..., 0] = True
        mask[:, 2] = False
    leaves = [t.to(DEV).requires_grad_() for t in (q, k, v)]
    if with_bias:
        wide = torch.full((1, 1, H, N, (N + 7) // 8 * 8), float("nan"))
        wide[..., :N] = bias
        leaves.append(wide.to(DEV)[..., :N].detach().requires_grad_())
    out = triangle_attention(*leaves[:3], leaves[3] if with_bias else None, None if mask is None else mask.to(DEV))
    got = torch.autograd.grad(out, leaves, dout.to(DEV))
    args = (*(to_np(t) for t in (q, k, v)), None if bias is None else to_np(bias),
            None if mask is None else mask.numpy(), D ** -0.5)
    assert O.rel_fro(to_np(out), O.triangle_attention(*args).reshape(out.shape)) <= 3e-5
    for a, b in zip(got, O.triangle_attention_grad(*args, to_np(dout))):
        assert torch.isfinite(a).all()
        assert O.rel_fro(to_np(a).reshape(b.shape), b) <= 3e-5 or abs(b).max() < 1e-12


@pytest.mark.parametrize("direction", ["outgoing", "incoming"])
@pytest.mark.parametrize(("N", "C", "Ch", "B", "dtype"), [
    (1, 128, 128, 3, torch.bfloat16), (33, 64, 128, 2, torch.bfloat16), (65, 128, 32, 1, torch.float16),
    (129, 64, 64, 1, torch.bfloat16), (200, 128, 128, 1, torch.float16), (512, 64, 32, 1, torch.bfloat16)])
def test_fused_trimul_backward_tiles(N, C, Ch, B, dtype, direction):
    """The fused input and output sides at every width of weight fragments, row tails of a tile, one
    tile and several for a workgroup, and both sides of the launch's rounds (256 workgroups below 4096
    tiles, 512 from there: N = 512), against the unfused launches on the same forward, and up to N = 200
    both against the fp64 oracle. A gradient passes about five roundings (gate, recomputed linears, the
    products' operands, the LayerNorm's, the result) of at most 2^-9 (bf16) or 2^-12 (fp16) each: 1e-2 and
    1.25e-3. One whose own size is far below the others' (a bias where the outputs cancel) is held to theirs."""
    from geometric_nn_ops_torch.triangle._kernels import trimul as K

    w = {k: v.to(DEV) for k, v in trimul_weights(C, Ch, dtype, seed=61, biases=True, ln_random=True).items()}
    x, mask = (t.to(DEV) for t in pair_input(B, N, C, dtype, seed=62))
    dout = torch.randn(B, N, N, C, generator=gen(63)).to(DEV, dtype)
    with torch.no_grad():
        args, keep, _, ws, off = K.build_args(x, direction, mask, 1e-5, w, separate_gate=True)
        K.run_stage("gnn_trimul_fwd", args, x.device)
        fused, plain = (K.trimul_bwd_hip(x, direction, mask, 1e-5, w, ws, off, dout, gate=keep[-1], fused=f)
                        for f in (True, False))
    fused, plain = ({"x": g[0], **g[1]} for g in (fused, plain))
    pairs = [(fused, {k: to_np(v) for k, v in plain.items()})]
    if N <= 200:
        want = O.trimul_grad(to_np(x), direction, to_np(mask), to_np(dout), **np_weights(w))
        pairs += [(fused, want), (plain, want)]
    bound = 1e-2 if dtype == torch.bfloat16 else 1.25e-3
    for got, want in pairs:
        rms = {k: float((want[k] ** 2).mean() ** 0.5) for k in got}
        floor = 1e-2 * max(rms[k] for k in w)
        for k, g in got.items():
            assert torch.isfinite(g).all()
            d = float(((to_np(g) - want[k]) ** 2).mean() ** 0.5)
            assert d <= bound * max(rms[k], floor if k != "x" else 0.0), k
