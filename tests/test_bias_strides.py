"""Pair-bias views whose rows cannot be read in aligned groups of 8 keys: the tiled attention kernel and
the backward get a copy of them, and the C entry points refuse them before any launch."""

import ctypes

import pytest
import torch

from helpers import TRIANGLE_ATTENTION_TOL, assert_close_to_oracle, attention_inputs, gen, to_np
from oracle import triangle_oracle as O


def _views(n, h, dtype, device="cpu"):
    """(bias [2, 1, h, n, n], whether it may be used in place) by name."""
    def rand(*shape):
        return torch.randn(*shape, generator=gen(n)).to(device, dtype)

    pitch = (n + 15) // 8 * 8
    whole = n % 8 == 0
    return {
        "contiguous": (rand(2, 1, h, n, n), whole),
        "wide_pitch": (rand(2, 1, h, n, pitch)[..., :n], True),
        "over_queries": (rand(2, 1, h, 1, n).expand(2, 1, h, n, n), whole),
        "over_heads": (rand(2, 1, 1, n, pitch)[..., :n].expand(2, 1, h, n, n), True),
        "over_all": (rand(1, 1, 1, 1, n).expand(2, 1, h, n, n), whole),
        "transposed": (rand(2, 1, h, n, pitch)[..., :n].transpose(-1, -2), False),
        # planes off a 16-byte boundary although the rows' pitch is a multiple of 8
        "odd_planes": (rand(2 * h * (n * pitch + 4)).as_strided((2, 1, h, n, n),
                                                               (h * (n * pitch + 4), 1, n * pitch + 4, pitch, 1)),
                       False),
        # the last row ends with the storage
        "no_room_after_the_end": (rand(2 * h * n * pitch - (pitch - n)).as_strided(
            (2, 1, h, n, n), (h * n * pitch, 1, n * pitch, pitch, 1)), whole),
    }


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32], ids=["bf16", "fp32"])
@pytest.mark.parametrize("n", [1, 64, 131])
@pytest.mark.parametrize("view", list(_views(8, 2, torch.float32)))
def test_rows_of_a_prepared_bias_can_be_read(view, n, dtype):
    from geometric_nn_ops_torch.triangle._kernels.triangle_attention import _prepare_bias

    bias, usable = _views(n, 3, dtype)[view]
    got = _prepare_bias(bias, dtype)
    assert torch.equal(got, bias)
    b, _, h, i, j = got.stride()
    last = got.storage_offset() + b * (got.shape[0] - 1) + h * 2 + i * (n - 1)
    assert j == 1 and b % 8 == 0 and h % 8 == 0 and got.data_ptr() % 16 == 0 and (n == 1 or i % 8 == 0)
    assert n == 1 or n % 8 == 0 or i >= n
    assert (last + (n + 7) // 8 * 8) * got.element_size() <= got.untyped_storage().nbytes()
    if usable and n > 1:
        assert got.data_ptr() == bias.data_ptr()


@pytest.mark.parametrize(("n", "stride", "refused"), [
    (131, (2 * 131, 131, 0, 1), True),         # broadcast over the queries: no room past a row
    (131, (2 * 136, 136, 0, 1), True),
    (131, (2 * 131 * 136 + 8, 131 * 136 + 4, 136, 1), True),
    (131, (2 * 131 * 136 + 4, 131 * 136, 136, 1), True),
    (131, (2 * 131 * 136, 131 * 136, 136, 1), False),
    (128, (2 * 128, 128, 0, 1), False)])
def test_entry_points_refuse_rows_they_cannot_read(n, stride, refused):
    """The accepted strides end at the next check, which needs no device either."""
    from geometric_nn_ops_torch import _lib

    lib = _lib.load()
    a = _lib.TriAttnBwdArgs()
    for name in ("q", "k", "v", "o", "dout", "lse", "dq", "dk", "dv", "delta", "bias", "dbias"):
        setattr(a, name, 4096)
    a.B, a.S, a.N, a.H, a.D = 2, 3, n, 2, 32
    for st in ("q_stride", "k_stride", "v_stride", "o_stride", "do_stride"):
        setattr(a, st, _lib.I64x4(3 * n * 64, n * 64, 64, 32))
    a.bias_stride = _lib.I64x4(*stride)
    a.dtype, a.dbias_splits = _lib.GNN_F32, 2  # without dbias_ws
    assert lib.gnn_triattn_bwd(ctypes.byref(a), None) == _lib.GNN_ERR_ARG
    assert (b"readable" in lib.gnn_last_error()) == refused
    assert (b"dbias_ws" in lib.gnn_last_error()) != refused
    if refused:
        f = _lib.TriAttnArgs()
        f.q = f.k = f.v = f.o = f.bias = 4096
        f.B, f.S, f.N, f.H, f.D = 2, 3, n, 2, 32
        for st in ("q_stride", "k_stride", "v_stride", "o_stride"):
            setattr(f, st, _lib.I64x4(3 * n * 64, n * 64, 64, 32))
        f.bias_stride, f.dtype = _lib.I64x4(*stride), _lib.GNN_F32
        assert lib.gnn_triattn_fwd(ctypes.byref(f), None) == _lib.GNN_ERR_ARG
        assert b"readable" in lib.gnn_last_error()


@pytest.mark.gpu
@pytest.mark.parametrize(("dtype", "d"), [(torch.bfloat16, 32), (torch.bfloat16, 48), (torch.float32, 32)],
                         ids=["bf16", "bf16_d48", "fp32"])
@pytest.mark.parametrize("view", ["over_queries", "over_heads", "over_all", "odd_planes", "no_room_after_the_end"])
def test_gradients_with_such_a_bias(view, dtype, d):
    from geometric_nn_ops_torch.triangle import triangle_attention

    B, S, N, H = 2, 2, 131, 3
    t = attention_inputs(B, S, N, H, d, dtype, seed=9, with_bias=False, device="cuda")
    bias = _views(N, H, dtype, "cuda")[view][0]
    q, k, v = (t[x].requires_grad_() for x in "qkv")
    leaf = bias.detach().requires_grad_()
    dout = torch.randn(B, S, N, H, d, generator=gen(10)).to("cuda", dtype)
    with torch.no_grad():
        alone = triangle_attention(q, k, v, bias)
    out = triangle_attention(q, k, v, leaf)
    got = torch.autograd.grad(out, (q, k, v, leaf), dout)
    args = (to_np(q), to_np(k), to_np(v), to_np(bias))
    tol = TRIANGLE_ATTENTION_TOL[dtype, "ieee"]
    for o in (alone, out):
        assert_close_to_oracle("o", o, O.triangle_attention(*args), tol)
    for name, g, w in zip(("dq", "dk", "dv", "dbias"), got, O.triangle_attention_grad(*args, None, None, to_np(dout))):
        assert_close_to_oracle(name, g, w, tol)
