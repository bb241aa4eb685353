"""Triangle-attention gradients where some queries' logits lie far from zero: the pair bias alone holds
a query at the mask sentinel, or anywhere at all, next to ordinary queries and fully masked rows.

The backward gets o and lse as fp32 logits give them (at 1e9 one ulp swallows q . k) and is compared with
its own definition in float64: P = exp(S - lse), Delta = dO . o. Held queries have q = 0, so that their
S is the bias exactly. Tolerance: the table that the gradient tests use."""

import pytest
import torch

from helpers import TRIANGLE_ATTENTION_TOL, assert_close_to_oracle, attention_inputs, gen, key_mask, to_np

pytestmark = pytest.mark.gpu

DEV = "cuda"
MASK_VALUE = {torch.bfloat16: 1e9, torch.float16: torch.finfo(torch.float16).max / 2, torch.float32: 1e9}


def heads_first(t):
    return t.double().transpose(2, 3).contiguous()


def scores(q, k, bias, mask):
    """[B, S, H, N, N] in fp32, the mask term added last; and the scaled q."""
    qs = heads_first((q.float() * q.shape[-1] ** -0.5).to(q.dtype))
    s = (qs @ heads_first(k).transpose(-1, -2).contiguous() + bias.double()).float()
    if mask is not None:
        value = torch.tensor(-MASK_VALUE[q.dtype]).to(q.dtype).float().to(s.device)
        s = torch.where(~mask, s + value, s)
    return s, qs


def gradients(q, k, v, bias, mask, o, dout, lse, *, divides_queries):
    """(dq, dk, dv, dbias). P of a masked key is divided by N, and so is, in dq, dk and dv of the
    row-resident kernels, P of a query of a masked call whose lse has lost log(l) to the sentinel."""
    n, d = q.shape[2], q.shape[4]
    s, qs = scores(q, k, bias, mask)
    k, v, dout, o = (heads_first(t) for t in (k, v, dout, o))
    p = torch.exp((s - lse[..., None]).double())
    if mask is not None:
        p = torch.where(mask, p, p / n)
    dp = dout @ v.transpose(-1, -2).contiguous() - (dout * o).sum(-1, keepdim=True)
    dbias = (p * dp).sum(1, keepdim=True)
    if mask is not None and divides_queries:
        held = (lse <= min(-0.5 * MASK_VALUE[q.dtype], -(2.0**27)))[..., None]
        p = torch.where(held & mask, p / n, p)
    ds = p * dp
    t = lambda x: x.transpose(-1, -2).contiguous()  # noqa: E731
    dq, dk, dv = d**-0.5 * (ds @ k), t(ds) @ qs, t(p) @ dout
    return (*(x.transpose(2, 3) for x in (dq, dk, dv)), dbias)


def check(n, dtype, held_at, masked, *, d=32, rows=(0, 5, -1), divides_queries=True):
    from geometric_nn_ops_torch.triangle._kernels import triangle_attention as K

    shape = B, S, N, H, D = 1, 3, n, 2, d
    t = attention_inputs(*shape, dtype, seed=n, with_bias=True, bias_scale=0.5, device=DEV)
    mask = None
    if masked:
        mask = key_mask(B, S, N, seed=n + 1, frac_keep=0.75, device=DEV)
        mask[:, 1] = False  # a row whose keys are all masked
    q, k, v, bias = (t[x] for x in ("q", "k", "v", "bias"))
    q[:, :, list(rows)] = 0
    bias[..., list(rows), :] = held_at
    dout = torch.randn(*shape, generator=gen(n + 2)).to(DEV, dtype)
    s = scores(q, k, bias, mask)[0].double()
    lse = torch.logsumexp(s, -1).float()
    o = (torch.softmax(s, -1) @ heads_first(v)).transpose(2, 3).to(dtype).contiguous()
    got = K.triangle_attention_bwd_hip(q, k, v, o, dout, lse, bias=bias, mask=mask, precision="ieee")
    want = gradients(q, k, v, bias, mask, o, dout, lse, divides_queries=divides_queries)
    tol = TRIANGLE_ATTENTION_TOL[dtype, "ieee"]
    for name, g, w in zip(("dq", "dk", "dv", "dbias"), got, want):
        assert_close_to_oracle(name, g, to_np(w), tol)
    # the other queries by themselves: a held one must not move them
    others = torch.ones(N, dtype=torch.bool, device=DEV)
    others[list(rows)] = False
    assert_close_to_oracle("dq of the others", got[0][:, :, others], to_np(want[0][:, :, others]), tol)
    assert_close_to_oracle("dbias of the others", got[3][..., others, :], to_np(want[3][..., others, :]), tol)


# the fused kernel with two key blocks a wave and with one, its largest N, and the two-kernel path
SIZES = pytest.mark.parametrize("n", [64, 130, 300, 512, 600])


@SIZES
@pytest.mark.parametrize(("dtype", "held_at"), [(torch.bfloat16, -1e9), (torch.float16, -3e4)], ids=["bf16", "fp16"])
@pytest.mark.parametrize("rows", [(0,), (0, 5, -1)], ids=["first", "several"])
def test_masked_call_with_a_query_held_at_the_sentinel(n, dtype, held_at, rows):
    """A padded first query (left padding) says nothing about the row's keys: the others keep their P."""
    check(n, dtype, held_at, True, rows=rows)


@pytest.mark.parametrize(("dtype", "d"), [(torch.bfloat16, 24), (torch.float32, 32)], ids=["bf16_d24", "fp32"])
def test_masked_call_on_the_tiled_kernels(dtype, d):
    """Their dq, dk, dv and pair-bias gradient divide per masked key only."""
    check(130, dtype, -1e9, True, d=d, rows=(0, 128), divides_queries=False)


@SIZES
@pytest.mark.parametrize("masked", [False, True], ids=["plain", "masked"])
@pytest.mark.parametrize("held_at", [-250.0, -300.0, -1e7, 1e7, -1e9, torch.finfo(torch.bfloat16).min],
                         ids=["m250", "m300", "m1e7", "p1e7", "m1e9", "lowest"])
def test_queries_held_far_from_zero(n, masked, held_at):
    """On both sides of where the row kernels change from one fma to subtracting lse first, where lse
    times log2(e) loses the exponent (1e7, 1e9), and where that product overflows."""
    check(n, torch.bfloat16, held_at, masked, rows=(3, n // 2))
