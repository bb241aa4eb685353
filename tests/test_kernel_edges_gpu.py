"""Kernels at the sizes where their tiles, remainders and dispatch lines lie, against the fp64
oracle. Tolerances: one rounding of a result costs at most half an ulp (bf16 2^-9, fp16 2^-12,
fp32 2^-24 relative), and the bounds below allow for the two or three roundings a value passes."""

import pytest
import torch

from helpers import gen, to_np
from oracle import triangle_oracle as O

pytestmark = pytest.mark.gpu

DEV = "cuda"
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
