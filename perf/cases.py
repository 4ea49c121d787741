"""The attention path's work, as cases that a timing program can run.

A case is a dict of plain values; `kind` says which public entry points it
goes through:

  self         attention(q, k, v) of one layer's self-attention, no grad
  cross_trim   head_norm(x) + cross_attention_trimmed over a zero-padded text
               context with key lengths, no grad
  layer        one layer's whole attention path, no grad: qkv_norm_rope,
               self-attention, head_norm, cross-attention over the 512
               untrimmed text keys
  train        qkv_norm_rope + attention, forward and backward (LoRA training)
  train_cross  head_norm + attention over the 512-key text context, forward
               and backward
  proj         one of the fused input projections (op: qkv, xq or kv), no grad
  vae          the VAE mid-block's head_dim-384 attention, no grad

Sizes are the model's: 16 heads of 128, width 2048, 512 text tokens of width
1024, one token per 16 x 16 pixels (a grid of h x w tokens, 4 h w positions in
the VAE). Images go from 256 x 256 to 1536 x 1536 pixels in any aspect ratio;
batch 2 is classifier-free guidance's two branches.
"""

from __future__ import annotations

import math

import torch

import __graft_entry__

H, HD = 16, 128
D = H * HD
TEXT, TEXT_DIM = 512, 1024
VAE_HD = 384
EPS = 1e-6
BF = torch.bfloat16
F64 = torch.float64


def listed():
    return [
        # Self-attention at 512 x 512, one branch: the smallest usual image,
        # where a launch's fixed cost weighs most.
        {"name": "self_512", "kind": "self", "B": 1, "h": 32, "w": 32},
        # ... at 768 x 768: a usual size that is no power of two.
        {"name": "self_768", "kind": "self", "B": 1, "h": 48, "w": 48},
        # ... at 1024 x 1024: the model's native size, the benchmark's headline.
        {"name": "self_1024", "kind": "self", "B": 1, "h": 64, "w": 64},
        # ... at 1536 x 1536, the largest image.
        {"name": "self_1536", "kind": "self", "B": 1, "h": 96, "w": 96},
        # Cross-attention of a guided step at 1024 x 1024 with a trimmed text
        # context: a short negative prompt and a long prompt.
        {"name": "cross_trim_1024", "kind": "cross_trim", "B": 2, "h": 64, "w": 64, "len0": 58, "len1": 322},
        # One layer's attention of a guided step at 832 x 1216, the usual
        # portrait size: 3952 tokens, ragged in every tile size.
        {"name": "layer_832x1216", "kind": "layer", "B": 2, "h": 76, "w": 52, "len0": 58, "len1": 322},
        # LoRA training on 512 x 512 images: self-attention of one item.
        {"name": "train_512", "kind": "train", "B": 1, "h": 32, "w": 32},
        # LoRA training on 1024 x 1024 images.
        {"name": "train_1024", "kind": "train", "B": 1, "h": 64, "w": 64},
        # LoRA training's cross-attention, two items at 1024 x 1024 (the text
        # context is not trimmed under autograd).
        {"name": "train_cross_1024", "kind": "train_cross", "B": 2, "h": 64, "w": 64, "len0": 58, "len1": 322},
        # The QKV projection with its normalisation and rotation, guided step
        # at 1024 x 1024.
        {"name": "proj_qkv_1024", "kind": "proj", "op": "qkv", "B": 2, "h": 64, "w": 64},
        # One layer's text keys and values, both prompts (28 such calls per image).
        {"name": "proj_kv_text", "kind": "proj", "op": "kv", "B": 2, "h": 0, "w": 0},
        # The VAE decoder's attention at 1024 x 1024: 16384 positions.
        {"name": "vae_1024", "kind": "vae", "B": 1, "h": 64, "w": 64},
    ]


def _side(rng):
    """One side of the image in tokens, 16 to 96, spread over its logarithm."""
    return int(round(math.exp(rng.uniform(math.log(16), math.log(96)))))


def draw(rng):
    most = {}
    for c in listed():
        most[c["kind"]] = max(most.get(c["kind"], 0.0), work(c)["flops"])
    kind = rng.choice(("self", "self", "cross_trim", "layer", "train", "train_cross", "proj", "vae"))
    while True:
        c = {"kind": kind, "B": rng.choice((1, 2)), "h": _side(rng), "w": _side(rng)}
        if kind in ("cross_trim", "layer", "train_cross"):
            c["len0"], c["len1"] = rng.randint(32, TEXT), rng.randint(32, TEXT)
        if kind == "proj":
            c["op"] = rng.choice(("qkv", "xq", "kv"))
        if work(c)["flops"] <= most[kind]:
            return c


# ------------------------------------------------------------------ inputs --


def _tokens(case):
    return case["h"] * case["w"]


def _lens(case):
    return [case["len0"], case["len1"]][: case["B"]]


def _inputs(case, seed):
    """The case's tensors on the GPU, from the seed alone: activations N(0, 1)
    in bf16, RMSNorm weights 1 + 0.02 N(0, 1) in fp32, projection weights
    N(0, 1 / K), a text context whose rows past each prompt are zero."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    pkg = __graft_entry__.load_package()

    def n(*shape, scale=1.0):
        return (torch.randn(*shape, generator=g, device="cuda") * scale).to(BF)

    def w():
        return 1 + 0.02 * torch.randn(HD, generator=g, device="cuda")

    kind, B, S = case["kind"], case["B"], _tokens(case)
    t = {}
    if kind == "vae":
        for name in ("q", "k", "v"):
            t[name] = n(B, 1, 4 * S, VAE_HD)
        return t
    if kind == "proj":
        op = case["op"]
        if op == "kv":
            t["x"], rows, width = n(B, TEXT, TEXT_DIM), 2 * D, TEXT_DIM
        else:
            t["x"], rows, width = n(B, S, D), 3 * D if op == "qkv" else D, D
        t["weight"] = n(rows, width, scale=width**-0.5)
        t["qw"], t["kw"] = w(), w()
        if op == "qkv":
            t["cos"], t["sin"] = pkg.rope_tables(case["h"], case["w"], HD, "cuda")
        return t
    if kind in ("self", "layer", "train"):
        t["qkv"], t["qw"], t["kw"] = n(B, S, 3 * D), w(), w()
        t["cos"], t["sin"] = pkg.rope_tables(case["h"], case["w"], HD, "cuda")
    if kind in ("cross_trim", "layer", "train_cross"):
        t["x"], t["xw"] = n(B, S, D), w()
        t["k"], t["v"] = n(B, TEXT, H, HD), n(B, TEXT, H, HD)
        for b, ln in enumerate(_lens(case)):
            t["k"][b, ln:] = 0
            t["v"][b, ln:] = 0
        lens = torch.tensor(_lens(case), dtype=torch.int32, device="cuda")
        t["lens"], t["ln_pad"] = lens, torch.log((TEXT - lens).float())
    if kind == "train":
        t["dout"] = n(B, S, D)
    if kind == "train_cross":
        t["dout"] = n(B, S, D)
    return t


def prepare(case, seed):
    pkg = __graft_entry__.load_package()
    t = _inputs(case, seed)
    t["kind"], t["pkg"], t["op"] = case["kind"], pkg, case.get("op")
    if case["kind"] == "self":
        # What the prologue leaves: q and k of their own, v a view of qkv.
        with torch.no_grad():
            t["q"], t["k"], t["v"] = pkg.qkv_norm_rope(t["qkv"], t["qw"], t["kw"], t["cos"], t["sin"], H, EPS)
    if case["kind"] == "proj":
        from anima_flat_amd.kernels import proj

        t["proj"] = proj
        t["kw16"] = t["kw"].to(BF)
    if case["kind"] == "train":
        for name in ("qkv", "qw", "kw"):
            t[name].requires_grad_(True)
    if case["kind"] == "train_cross":
        for name in ("x", "xw", "k", "v"):
            t[name].requires_grad_(True)
    return t


def run(state):
    t, pkg, kind = state, state["pkg"], state["kind"]
    if kind == "train":
        q, k, v = pkg.qkv_norm_rope(t["qkv"], t["qw"], t["kw"], t["cos"], t["sin"], H, EPS)
        out = pkg.attention(q, k, v)
        return (out.detach(), *torch.autograd.grad(out, (t["qkv"], t["qw"], t["kw"]), t["dout"]))
    if kind == "train_cross":
        out = pkg.attention(pkg.head_norm(t["x"], t["xw"], H, EPS), t["k"], t["v"])
        return (out.detach(), *torch.autograd.grad(out, (t["x"], t["xw"], t["k"], t["v"]), t["dout"]))
    with torch.no_grad():
        if kind == "self":
            return pkg.attention(t["q"], t["k"], t["v"])
        if kind == "cross_trim":
            q = pkg.head_norm(t["x"], t["xw"], H, EPS)
            return pkg.cross_attention_trimmed(q, t["k"], t["v"], t["lens"], t["ln_pad"])
        if kind == "layer":
            q, k, v = pkg.qkv_norm_rope(t["qkv"], t["qw"], t["kw"], t["cos"], t["sin"], H, EPS)
            a = pkg.attention(q, k, v)
            return a, pkg.attention(pkg.head_norm(t["x"], t["xw"], H, EPS), t["k"], t["v"])
        if kind == "vae":
            return pkg.vae.attend(t["q"], t["k"], t["v"])
        if t["op"] == "qkv":
            return t["proj"].qkv_proj_norm_rope(
                t["x"], t["weight"], t["qw"], t["kw"], t["cos"], t["sin"], H, EPS)
        if t["op"] == "xq":
            return t["proj"].proj_head_norm(t["x"], t["weight"], t["qw"], H, EPS)
        return t["proj"].kv_proj_norm(t["x"], t["weight"], t["kw16"], H, EPS)


# -------------------------------------------------------------------- work --


def work(case):
    """Bytes: each input read once, each output written once (bf16; the text
    K/V of a masked call up to each prompt's length). Flops: the matrix
    products (backward: 5 products where the forward has 2)."""
    kind, B, S = case["kind"], case["B"], _tokens(case)
    if kind == "vae":
        n = 4 * S
        return {"bytes": 8.0 * B * n * VAE_HD, "flops": 4.0 * B * n * n * VAE_HD}
    if kind == "proj":
        rows, width, cols = {
            "qkv": (B * S, D, 3 * D), "xq": (B * S, D, D), "kv": (B * TEXT, TEXT_DIM, 2 * D)}[case["op"]]
        return {"bytes": 2.0 * (rows * width + width * cols + rows * cols), "flops": 2.0 * rows * width * cols}
    act = 2.0 * B * S * D  # one [B, S, 16, 128] tensor
    text = 2.0 * B * TEXT * D
    tables = 8.0 * S * (HD // 2)
    self_flops = 4.0 * B * S * S * D
    cross_flops = 4.0 * B * S * TEXT * D
    if kind == "self":
        return {"bytes": 4 * act, "flops": self_flops}
    if kind == "cross_trim":
        used = float(sum(_lens(case)))
        return {"bytes": 2 * act + 4.0 * used * D, "flops": 4.0 * S * used * D}
    if kind == "layer":
        return {"bytes": 3 * act + tables + act + 2 * act + 2 * text, "flops": self_flops + cross_flops}
    if kind == "train":
        # qkv, dout in; out, dqkv out.
        return {"bytes": 8 * act + tables, "flops": 3.5 * self_flops}
    # x, dout, k, v in; out, dx, dk, dv out.
    return {"bytes": 4 * act + 4 * text, "flops": 3.5 * cross_flops}


def tolerance(case):
    # bf16 results of fp32 sums, with bf16 probabilities (in training also bf16
    # score gradients) between two products, and in `layer` and `train` bf16
    # q and k between the rotation and the attention. About four times the
    # largest distance from the 64-bit results measured on one run of the
    # listed and some drawn cases: rel 2.9e-3 and max 0.03 for one attention
    # or projection, 3.9e-3 behind the prologue, 4.9e-3 and 0.04 for gradients.
    if case["kind"] in ("train", "train_cross"):
        return {"rel": 2e-2, "max": 0.16}
    return {"rel": 1.6e-2 if case["kind"] == "layer" else 1.2e-2, "max": 0.12}


# ------------------------------------------------------------------- exact --


def _norm64(x, weight):
    x = x.to(F64)
    return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + EPS) * weight.to(F64)


def _rope64(x, cos, sin):
    c, s = cos.to(F64)[None, :, None], sin.to(F64)[None, :, None]
    a, b = x[..., : HD // 2], x[..., HD // 2 :]
    return torch.cat((a * c - b * s, b * c + a * s), -1)


def _qkv64(qkv, t):
    B, S, _ = qkv.shape
    q, k, v = qkv.to(F64).view(B, S, 3, H, HD).unbind(2)
    return _rope64(_norm64(q, t["qw"]), t["cos"], t["sin"]), _rope64(_norm64(k, t["kw"]), t["cos"], t["sin"]), v


def _attend64(q, k, v, dout=None):
    """softmax(q k^T / sqrt(d)) v of [B, S, heads, d] tensors one head and up
    to 4096 queries at a time; with dout also the gradients of q, k and v."""
    B, Sq, heads, d = q.shape
    out = torch.empty(q.shape, dtype=F64, device=q.device)
    grads = None if dout is None else tuple(torch.zeros(x.shape, dtype=F64, device=x.device) for x in (q, k, v))
    for b in range(B):
        for h in range(heads):
            kh, vh = k[b, :, h].to(F64).contiguous(), v[b, :, h].to(F64).contiguous()
            for s in range(0, Sq, 4096):
                qh = q[b, s : s + 4096, h].to(F64).contiguous()
                p = torch.softmax(qh @ kh.T / math.sqrt(d), -1)
                out[b, s : s + 4096, h] = p @ vh
                if dout is not None:
                    do = dout[b, s : s + 4096, h].to(F64).contiguous()
                    ds = p * (do @ vh.T - (do * out[b, s : s + 4096, h]).sum(-1, keepdim=True)) / math.sqrt(d)
                    grads[0][b, s : s + 4096, h] = ds @ kh
                    grads[1][b, :, h] += ds.T @ qh
                    grads[2][b, :, h] += p.T @ do
    return out if dout is None else (out, grads)


def exact(case, seed):
    t = _inputs(case, seed)
    kind, B, S = case["kind"], case["B"], _tokens(case)
    if kind == "vae":
        q, k, v = (t[n].transpose(1, 2) for n in ("q", "k", "v"))
        return _attend64(q, k, v).transpose(1, 2)
    if kind == "proj":
        y = t["x"].to(F64) @ t["weight"].to(F64).T
        if case["op"] == "qkv":
            return _qkv64(y, t)
        if case["op"] == "xq":
            return _norm64(y.view(B, S, H, HD), t["qw"])
        k, v = y.view(B, TEXT, 2, H, HD).unbind(2)
        return _norm64(k, t["kw"].to(BF)), v
    if kind == "self":
        # The call's inputs are the prologue's bf16 q and k.
        t = prepare(case, seed)
        return _attend64(t["q"], t["k"], t["v"]).flatten(2)
    if kind == "cross_trim":
        # Zero keys and values past each length: the padded softmax itself.
        return _attend64(_norm64(t["x"].view(B, S, H, HD), t["xw"]), t["k"], t["v"]).flatten(2)
    if kind == "layer":
        a = _attend64(*_qkv64(t["qkv"], t)).flatten(2)
        return a, _attend64(_norm64(t["x"].view(B, S, H, HD), t["xw"]), t["k"], t["v"]).flatten(2)
    dout = t["dout"].view(B, S, H, HD)
    if kind == "train":
        leaves = [t[n].to(F64).requires_grad_(True) for n in ("qkv", "qw", "kw")]
        q, k, v = _qkv64(leaves[0], {**t, "qw": leaves[1], "kw": leaves[2]})
        out, grads = _attend64(q.detach(), k.detach(), v.detach(), dout)
        return (out.flatten(2), *torch.autograd.grad((q, k, v), leaves, grads))
    x, xw = t["x"].to(F64).requires_grad_(True), t["xw"].to(F64).requires_grad_(True)
    q = _norm64(x.view(B, S, H, HD), xw)
    out, (dq, dk, dv) = _attend64(q.detach(), t["k"], t["v"], dout)
    return (out.flatten(2), *torch.autograd.grad(q, (x, xw), dq), dk, dv)
