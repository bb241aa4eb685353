"""The calls a pairformer makes through this package's public entry points, over the sizes it makes them at.

A case is a dict of plain values:

  op          "attention" (triangle_attention), "trimul" (triangle_multiplicative_update),
              "pair_bias" (attention_pair_bias) or "block" (the four pair updates in a row)
  train       the forward with everything requiring grad, and the backward from a given output
              gradient; otherwise the forward under inference_mode
  dtype       "bf16", "fp16" or "fp32"; precision is torch's fp32 matmul setting, "ieee" or "tf32"
  mask        "none", "tail" (the last eighth of the residues is padding) or, for attention,
              "ragged" (every row has a length of its own between n / 2 and n)

Work counts each input read once and each output written once, and the operations of the
contractions. exact() states the same math in float64 torch.
"""

import os
import sys

import torch
import torch.nn.functional as F

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "geometric-nn-ops_amd"))

import cuequivariance_ops_torch as cueq  # noqa: E402
from geometric_nn_ops_torch.triangle import (attention_pair_bias, triangle_attention,  # noqa: E402
                                             triangle_multiplicative_update)

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
SIZE = {"bf16": 2, "fp16": 2, "fp32": 4}


def _attention(name, n, dtype="bf16", *, train=False, h=4, d=32, b=1, mask="none", layout="start", precision="ieee",
               bias_scale=1.0):
    c = {"op": "attention", "b": b, "n": n, "h": h, "d": d, "dtype": dtype, "precision": precision, "train": train,
         "mask": mask, "layout": layout, "bias_scale": bias_scale}
    return dict(c, name=name) if name else c


def _trimul(name, n, dtype="bf16", *, train=False, c=128, ch=128, b=1, mask="tail", direction="outgoing",
            precision="ieee", biases=False):
    k = {"op": "trimul", "b": b, "n": n, "c": c, "ch": ch, "dtype": dtype, "precision": precision, "train": train,
         "mask": mask, "direction": direction, "biases": biases}
    return dict(k, name=name) if name else k


def _pair_bias(name, n, dtype="bf16", *, h=16, d=24, b=1, m=1, cs=384, cz=128, mask="tail", precision="ieee"):
    c = {"op": "pair_bias", "b": b, "m": m, "n": n, "h": h, "d": d, "cs": cs, "cz": cz, "dtype": dtype,
         "precision": precision, "train": False, "mask": mask}
    return dict(c, name=name) if name else c


def listed():
    return [
        # a short chain or a unit test: the call itself costs more than the kernels
        _trimul("trimul_n64_fp32", 64, "fp32", mask="none"),
        # a small protein through the cuequivariance entry point, in its [B, N, H, S, D] layout
        _attention("attention_n256_bf16_cueq", 256, mask="tail", layout="cueq"),
        # inference on an ordinary protein, without padding
        _attention("attention_n512_bf16", 512),
        # inference on a padded batch of a larger one: each row has its own valid length
        _attention("attention_n768_bf16_ragged", 768, mask="ragged", bias_scale=2.0),
        # full-precision inference around the ending node (transposed views), at tf32 and an odd size
        _attention("attention_n333_fp32_tf32_ending", 333, "fp32", mask="tail", layout="end", precision="tf32"),
        # training at the usual crop
        _attention("attention_train_n384_bf16", 384, train=True, mask="tail"),
        # training in full precision at a small odd crop
        _attention("attention_train_n131_fp32", 131, "fp32", train=True, mask="tail"),
        # the multiplicative update at inference, ordinary size, over the first index
        _trimul("trimul_n512_bf16_incoming", 512, direction="incoming"),
        # its training at the usual crop
        _trimul("trimul_train_n384_bf16", 384, train=True),
        # its training in full precision, which the first stages of a model use, at an odd crop
        _trimul("trimul_train_n201_fp32_incoming", 201, "fp32", train=True, direction="incoming", biases=True),
        # the single track's attention at 384 tokens: 16 heads of 24
        _pair_bias("pair_bias_n384_bf16", 384),
        # the pair stack of a large complex: both multiplicative updates and both attentions
        {"name": "block_n1024_bf16", "op": "block", "b": 1, "n": 1024, "h": 4, "d": 32, "c": 128, "ch": 128,
         "dtype": "bf16", "precision": "ieee", "train": False, "mask": "none"},
    ]


def draw(rng):
    def size(lo, hi):
        return int(round(lo * (hi / lo) ** rng.random()))

    kind = rng.choice(("attention", "attention", "attention_train", "trimul", "trimul", "trimul_train", "pair_bias"))
    dtype = rng.choice(("bf16", "bf16", "bf16", "fp16", "fp32"))
    precision = rng.choice(("ieee", "tf32")) if dtype == "fp32" else "ieee"
    if kind == "pair_bias":
        return _pair_bias(None, size(48, 768), dtype, h=rng.choice((8, 16)), d=rng.choice((24, 32, 48)),
                          m=rng.choice((1, 1, 2)), cz=rng.choice((64, 128)), mask=rng.choice(("none", "tail")),
                          precision=precision)
    train = kind.endswith("train")
    n = size(32, (256 if train else 448) if dtype == "fp32" else (512 if train else 768))
    b = 2 if n <= 128 and rng.random() < 0.5 else 1
    if kind.startswith("attention"):
        h, d = rng.choice(((4, 32), (4, 32), (4, 32), (8, 16), (4, 24), (4, 48), (2, 64)))
        return _attention(None, n, dtype, train=train, h=h, d=d, b=b, mask=rng.choice(("none", "tail", "ragged")),
                          layout=rng.choice(("start", "start", "end", "cueq")), precision=precision,
                          bias_scale=rng.choice((1.0, 2.0)))
    c, ch = rng.choice(((128, 128), (128, 128), (128, 128), (64, 64), (64, 32), (128, 64), (256, 128)))
    return _trimul(None, n, dtype, train=train, c=c, ch=ch, b=b, mask=rng.choice(("none", "tail")),
                   direction=rng.choice(("outgoing", "incoming")), precision=precision, biases=rng.random() < 0.5)


# ------------------------------------------------------------------------------------ inputs
class _Random:
    def __init__(self, seed, dtype):
        self.g = torch.Generator(device="cuda").manual_seed(seed)
        self.dtype = dtype

    def normal(self, *shape, scale=1.0, shift=0.0):
        t = torch.randn(*shape, generator=self.g, device="cuda")
        return t.mul_(scale).add_(shift).to(self.dtype)

    def lengths(self, lo, hi, shape):
        return torch.randint(lo, hi + 1, shape, generator=self.g, device="cuda")


def _trimul_weights(r, c, ch, biases):
    w = {
        "norm_in_weight": r.normal(c, scale=0.1, shift=1.0), "norm_in_bias": r.normal(c, scale=0.1),
        "p_in_weight": r.normal(2 * ch, c, scale=c ** -0.5), "g_in_weight": r.normal(2 * ch, c, scale=c ** -0.5),
        "norm_out_weight": r.normal(ch, scale=0.1, shift=1.0), "norm_out_bias": r.normal(ch, scale=0.1),
        "p_out_weight": r.normal(c, ch, scale=ch ** -0.5), "g_out_weight": r.normal(c, c, scale=c ** -0.5),
    }
    if biases:
        w.update(p_in_bias=r.normal(2 * ch, scale=0.1), g_in_bias=r.normal(2 * ch, scale=0.1, shift=0.5),
                 p_out_bias=r.normal(c, scale=0.1), g_out_bias=r.normal(c, scale=0.1, shift=0.5))
    return w


def _live(n, mask):
    return torch.arange(n, device="cuda") < (n - max(1, n // 8) if mask == "tail" else n)


def _attention_inputs(case, r):
    """q, k, v and bias in the layout the caller holds them in, and the key mask."""
    b, n, h, d = (case[k] for k in ("b", "n", "h", "d"))
    shape = (b, n, h, n, d) if case["layout"] == "cueq" else (b, n, n, h, d)
    q, k, v = (r.normal(*shape) for _ in range(3))
    bias = r.normal(b, 1, h, n, n, scale=case["bias_scale"])
    mask = None
    if case["mask"] == "tail":
        mask = _live(n, "tail").expand(b, n, 1, 1, n).contiguous()
    elif case["mask"] == "ragged":
        mask = torch.arange(n, device="cuda") < r.lengths((n + 1) // 2, n, (b, n, 1, 1, 1))
    return q, k, v, bias, mask


def _inputs(case, seed):
    r = _Random(seed, DTYPES[case["dtype"]])
    b, n = case["b"], case["n"]
    if case["op"] == "attention":
        q, k, v, bias, mask = _attention_inputs(case, r)
        dout = r.normal(*q.shape) if case["train"] else None
        return {"leaves": [q, k, v, bias], "mask": mask, "dout": dout}
    if case["op"] == "trimul":
        x = r.normal(b, n, n, case["c"])
        w = _trimul_weights(r, case["c"], case["ch"], case["biases"])
        mask = None
        if case["mask"] == "tail":
            live = _live(n, "tail")
            mask = (live[:, None] & live[None, :]).to(x.dtype).expand(b, n, n).contiguous()
        dout = r.normal(*x.shape) if case["train"] else None
        return {"leaves": [x, *w.values()], "names": list(w), "mask": mask, "dout": dout}
    if case["op"] == "pair_bias":
        bm, h, d, cs, cz = b * case["m"], case["h"], case["d"], case["cs"], case["cz"]
        width = h * d
        s = r.normal(bm, n, cs)
        q, k, v = (r.normal(bm, h, n, d) for _ in range(3))
        z = r.normal(b, n, n, cz)
        w = {"proj_g_weight": r.normal(width, cs, scale=cs ** -0.5),
             "proj_o_weight": r.normal(cs, width, scale=width ** -0.5),
             "proj_z_weight": r.normal(h, cz, scale=cz ** -0.5), "ln_z_weight": r.normal(cz, scale=0.1, shift=1.0),
             "proj_g_bias": r.normal(width, scale=0.1)}
        mask = _live(n, case["mask"]).to(s.dtype).expand(b, n).contiguous() if case["mask"] == "tail" else None
        return {"tensors": (s, q, k, v, z), "weights": w, "mask": mask}
    c, ch, h, d = case["c"], case["ch"], case["h"], case["d"]
    return {"z": r.normal(b, n, n, c), "trimul": [_trimul_weights(r, c, ch, False) for _ in range(2)],
            "attention": [{"qkv": r.normal(3 * h * d, c, scale=c ** -0.5), "b": r.normal(h, c, scale=c ** -0.5),
                           "o": r.normal(c, h * d, scale=(h * d) ** -0.5)} for _ in range(2)]}


def prepare(case, seed):
    torch.backends.cuda.matmul.fp32_precision = case["precision"]
    state = _inputs(case, seed)
    if case["train"]:
        for t in state["leaves"]:
            t.requires_grad_()
    return dict(state, case=case)


# --------------------------------------------------------------------------------------- run
def _call(state, leaves):
    case = state["case"]
    if case["op"] == "attention":
        q, k, v, bias = leaves
        if case["layout"] == "cueq":
            return cueq.triangle_attention(q, k, v, bias, state["mask"])
        if case["layout"] == "end":
            q, k, v = (t.transpose(1, 2) for t in (q, k, v))
            return triangle_attention(q, k, v, bias.transpose(-1, -2), state["mask"])
        return triangle_attention(q, k, v, bias, state["mask"])
    return triangle_multiplicative_update(leaves[0], case["direction"], state["mask"],
                                          **dict(zip(state["names"], leaves[1:])))


def _block(state):
    case, z = state["case"], state["z"]
    b, n, h, d = (case[k] for k in ("b", "n", "h", "d"))
    for direction, w in zip(("outgoing", "incoming"), state["trimul"]):
        z = z + triangle_multiplicative_update(z, direction, None, **w)
    for ending, w in zip((False, True), state["attention"]):
        q, k, v = F.linear(z, w["qkv"]).view(b, n, n, 3, h, d).unbind(3)
        bias = F.linear(z, w["b"]).permute(0, 3, 1, 2).unsqueeze(1)
        if ending:
            q, k, v = (t.transpose(1, 2) for t in (q, k, v))
            bias = bias.transpose(-1, -2)
        o = F.linear(triangle_attention(q, k, v, bias).reshape(b, n, n, h * d), w["o"])
        z = z + (o.transpose(1, 2) if ending else o)
    return z


def run(state):
    case = state["case"]
    if case["train"]:
        out = _call(state, state["leaves"])
        dout = state["dout"].transpose(1, 2) if case.get("layout") == "end" else state["dout"]
        return (out, *torch.autograd.grad(out, state["leaves"], dout))
    with torch.inference_mode():
        if case["op"] == "block":
            return _block(state)
        if case["op"] == "pair_bias":
            out, _ = attention_pair_bias(*state["tensors"], **state["weights"], mask=state["mask"])
            return out
        return _call(state, state["leaves"])


# -------------------------------------------------------------------------------------- work
def _attention_work(b, n, h, d, e):
    return e * (4 * b * n * n * h * d + b * h * n * n), 4 * b * n * h * n * n * d


def _trimul_work(b, n, c, ch, e):
    weights = e * (4 * ch * c + c * ch + c * c + 2 * c + 2 * ch)
    return 2 * e * b * n * n * c + weights, 2 * b * n ** 3 * ch + b * n * n * (10 * c * ch + 2 * c * c)


def work(case):
    b, n, e = case["b"], case["n"], SIZE[case["dtype"]]
    if case["op"] == "attention":
        by, fl = _attention_work(b, n, case["h"], case["d"], e)
        by += b * n * n if case["mask"] != "none" else 0
        # the backward's own tensors (dout in, dq / dk / dv / dbias out), and its five products
        # (the logits once more, dP, dV, dQ, dK) to the forward's two
        return {"bytes": 2 * by if case["train"] else by, "flops": 3.5 * fl if case["train"] else fl}
    if case["op"] == "trimul":
        by, fl = _trimul_work(b, n, case["c"], case["ch"], e)
        by += e * b * n * n if case["mask"] != "none" else 0
        return {"bytes": 2 * by if case["train"] else by, "flops": 3 * fl if case["train"] else fl}
    if case["op"] == "pair_bias":
        bm, h, d, cs, cz = b * case["m"], case["h"], case["d"], case["cs"], case["cz"]
        by = e * (2 * bm * n * cs + 3 * bm * n * h * d + b * n * n * cz + 2 * cs * h * d)
        return {"bytes": by, "flops": 4 * bm * h * n * n * d + 2 * b * n * n * h * cz + 4 * bm * n * cs * h * d}
    c, ch, h, d = case["c"], case["ch"], case["h"], case["d"]
    flops = 2 * _trimul_work(b, n, c, ch, e)[1] + 2 * _attention_work(b, n, h, d, e)[1]
    flops += 2 * 2 * b * n * n * c * (4 * h * d + h)
    return {"bytes": 2 * e * b * n * n * c, "flops": flops}


# ------------------------------------------------------------------------- tolerance and exact
def tolerance(case):
    """About four times the relative error against exact(): fp32 sums 2e-6 (its three-term bf16 split
    1e-5), attention in bf16 2.8e-3, where the multiplicative update, the gated output and every
    gradient round more than once 5e-3 to 6.5e-3; fp16 has three bits more."""
    if case["dtype"] == "fp32":
        return {"rel": 5e-5 if case["precision"] == "tf32" else 1e-5}
    rel = 1e-2 if case["op"] == "attention" and not case["train"] else 2e-2
    return {"rel": rel if case["dtype"] == "bf16" else rel / 5}


def _exact_attention(q, k, v, bias, mask):
    """[B, S, N, H, D] float64, a few rows of S at a time; masked keys get no weight."""
    b, s, n, h, d = q.shape
    rows = max(1, (1 << 27) // (h * n * n))
    outs = []
    for i in range(b):
        for r in range(0, s, rows):
            qr, kr, vr = (t[i, r:r + rows].transpose(1, 2) for t in (q, k, v))
            logits = torch.matmul(qr * d ** -0.5, kr.transpose(-1, -2).contiguous()) + bias[i]
            if mask is not None:
                logits = logits.masked_fill(~mask[i, r:r + rows], float("-inf"))
            outs.append(torch.matmul(torch.softmax(logits, -1), vr.contiguous()).transpose(1, 2))
    return torch.cat(outs).view(b, s, n, h, d)


def _exact_attention_grads(q, k, v, bias, mask, dout):
    """The output and (dq, dk, dv, dbias), a few rows of S at a time."""
    grads = [torch.zeros_like(t) for t in (q, k, v, bias)]
    out = torch.zeros_like(q)
    rows = max(1, (1 << 26) // (q.shape[3] * q.shape[2] ** 2))
    for i in range(q.shape[0]):
        for r in range(0, q.shape[1], rows):
            part = [t[i:i + 1, r:r + rows].detach().requires_grad_() for t in (q, k, v)]
            part.append(bias[i:i + 1].detach().requires_grad_())
            o = _exact_attention(*part, None if mask is None else mask[i:i + 1, r:r + rows])
            for g, got, whole in zip(grads, torch.autograd.grad(o, part, dout[i:i + 1, r:r + rows]), (1, 1, 1, 0)):
                if whole:
                    g[i:i + 1, r:r + rows] = got
                else:
                    g[i:i + 1] += got
            out[i:i + 1, r:r + rows] = o.detach()
    return (out, *grads)


def _exact_trimul(x, direction, mask, w):
    ch = w["p_in_weight"].shape[0] // 2
    z = F.layer_norm(x, x.shape[-1:], w["norm_in_weight"], w["norm_in_bias"])
    p = F.linear(z, w["p_in_weight"], w.get("p_in_bias"))
    p = p * torch.sigmoid(F.linear(z, w["g_in_weight"], w.get("g_in_bias")))
    if mask is not None:
        p = p * mask[..., None]
    p = p.permute(0, 3, 1, 2).contiguous()  # [B, 2 Ch, N, N]
    a, b = p[:, :ch], p[:, ch:]
    if direction == "incoming":
        a, b = a.transpose(-1, -2), b.transpose(-1, -2)
    o = torch.matmul(a.contiguous(), b.transpose(-1, -2).contiguous()).permute(0, 2, 3, 1)
    o = F.layer_norm(o, (ch,), w["norm_out_weight"], w["norm_out_bias"])
    return F.linear(o, w["p_out_weight"], w.get("p_out_bias")) * torch.sigmoid(
        F.linear(z, w["g_out_weight"], w.get("g_out_bias")))


def _exact_block(case, s):
    z = s["z"].double()
    b, n, h, d = (case[k] for k in ("b", "n", "h", "d"))
    for direction, w in zip(("outgoing", "incoming"), s["trimul"]):
        z = z + _exact_trimul(z, direction, None, {k: v.double() for k, v in w.items()})
    for ending, w in zip((False, True), s["attention"]):
        t = z.transpose(1, 2) if ending else z
        q, k, v = F.linear(t, w["qkv"].double()).view(b, n, n, 3, h, d).unbind(3)
        bias = F.linear(t, w["b"].double()).permute(0, 3, 1, 2).unsqueeze(1)
        o = F.linear(_exact_attention(q, k, v, bias, None).reshape(b, n, n, h * d), w["o"].double())
        z = z + (o.transpose(1, 2) if ending else o)
    return z


def exact(case, seed):
    s = _inputs(case, seed)
    if case["op"] == "block":
        with torch.no_grad():
            return _exact_block(case, s)
    if case["op"] == "pair_bias":
        sr, q, k, v, z = (t.double() for t in s["tensors"])
        w = {k_: t.double() for k_, t in s["weights"].items()}
        bm, h, n, d = q.shape
        b, m = case["b"], case["m"]
        zn = F.layer_norm(z, z.shape[-1:], w["ln_z_weight"])
        bias = F.linear(zn, w["proj_z_weight"]).permute(0, 3, 1, 2).unsqueeze(1)
        q, k, v = (t.view(b, m, h, n, d).transpose(2, 3) for t in (q, k, v))
        mask = None if s["mask"] is None else (s["mask"] != 0).view(b, 1, 1, 1, n).expand(b, m, 1, 1, n)
        o = _exact_attention(q, k, v, bias, mask).reshape(bm, n, h * d)
        return F.linear(o * torch.sigmoid(F.linear(sr, w["proj_g_weight"], w["proj_g_bias"])), w["proj_o_weight"])
    leaves = [t.double() for t in s["leaves"]]
    if case["op"] == "trimul":
        mask = None if s["mask"] is None else s["mask"].double()
        if case["train"]:
            leaves = [t.requires_grad_() for t in leaves]
        out = _exact_trimul(leaves[0], case["direction"], mask, dict(zip(s["names"], leaves[1:])))
        return (out.detach(), *torch.autograd.grad(out, leaves, s["dout"].double())) if case["train"] else out
    mask = s["mask"]
    q, k, v, bias = leaves
    if case["layout"] != "start":
        axes = (2, 3) if case["layout"] == "cueq" else (1, 2)
        q, k, v = (t.transpose(*axes) for t in (q, k, v))
        bias = bias.transpose(-1, -2) if case["layout"] == "end" else bias
    if not case["train"]:
        o = _exact_attention(q, k, v, bias, mask)
        return o.transpose(2, 3) if case["layout"] == "cueq" else o
    dout = s["dout"].double()
    if case["layout"] == "start":
        return _exact_attention_grads(q, k, v, bias, mask, dout)
    out, dq, dk, dv, dbias = _exact_attention_grads(q, k, v, bias, mask, dout.transpose(*axes))
    out = out.transpose(2, 3) if case["layout"] == "cueq" else out
    return (out, *(t.transpose(*axes) for t in (dq, dk, dv)),
            dbias.transpose(-1, -2) if case["layout"] == "end" else dbias)
