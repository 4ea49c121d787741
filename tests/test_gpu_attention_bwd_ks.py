"""GPU parity of the backward's key-split dQ kernel (one workgroup per 64 queries, 32-key
blocks dealt to its four waves) and of the tails that the dQ and dK/dV kernels treat
apart, against the CPU oracle at the edges of their tiles."""

from __future__ import annotations

import pytest
import torch

from conftest import parity
from oracle import attn_oracle as ref

pytestmark = pytest.mark.gpu

BF = torch.bfloat16


def _inputs(B, Sq, Sk, H, seed):
    g = torch.Generator().manual_seed(seed)
    return [ref.bf16_normal((B, s, H, 128), g) for s in (Sq, Sk, Sk, Sq)]


def _gpu_backward(q, k, v, dout):
    q, k, v, dout = (t.to("cuda", BF) for t in (q, k, v, dout))
    out, lse = torch.ops.anima_flat.fa_fwd(q, k, v)
    grads = torch.ops.anima_flat.fa_bwd(dout, q, k, v, out, lse)
    again = torch.ops.anima_flat.fa_bwd(dout, q, k, v, out, lse)
    assert all(torch.equal(a, b) for a, b in zip(grads, again))  # fixed summation order
    return grads


@pytest.mark.parametrize(
    "B,Sq,Sk,H",
    [
        (1, 1, 2, 1),
        (1, 63, 31, 2),  # less than one key block: rows re-read, keys masked
        (2, 64, 32, 3),  # one block: three waves hold no keys
        (1, 65, 33, 2),  # two blocks, the second moved back over 31 keys
        (1, 100, 127, 2),  # every wave one block
        (1, 128, 129, 2),  # a second round of blocks for wave 0 only
        (2, 257, 160, 2),  # queries past the last whole item of 256
        (1, 300, 1000, 4),
    ],
)
def test_key_split_dq(pkg, monkeypatch, B, Sq, Sk, H):
    q, k, v, dout = _inputs(B, Sq, Sk, H, 500 + Sq + Sk)
    monkeypatch.setenv("AA_DQ_KERNEL", "ks")
    grads = _gpu_backward(q, k, v, dout)
    monkeypatch.setenv("AA_DQ_KERNEL", "2g")
    other = _gpu_backward(q, k, v, dout)
    for name, got, want in zip(("dq", "dk", "dv"), grads, ref.attention_backward(q, k, v, dout)):
        parity(got, want, name=name)
    # dK and dV come from the stats records the dQ kernel writes: the same bits.
    assert torch.equal(grads[1], other[1]) and torch.equal(grads[2], other[2])


@pytest.mark.parametrize("kernel", ["1w", "2role"])
@pytest.mark.parametrize(
    "Sq,Sk,H",
    [
        # 260 key blocks: the last 4 of them split over query ranges. 1560 dQ
        # items: the last 24 key-split.
        (1400, 100, 260),
        # 260 dQ items, 4 of them key-split; too few query tiles to split dK/dV.
        (70, 128, 260),
    ],
)
def test_tails_behind_whole_rounds(pkg, monkeypatch, kernel, Sq, Sk, H):
    q, k, v, dout = _inputs(1, Sq, Sk, H, 900 + Sq)
    monkeypatch.setenv("AA_DKDV_KERNEL", kernel)
    grads = _gpu_backward(q, k, v, dout)
    heads = [0, 128, 255, 256, 258, 259]
    want = ref.attention_backward(*(t[:, :, heads] for t in (q, k, v, dout)))
    for name, got, w in zip(("dq", "dk", "dv"), grads, want):
        parity(got[:, :, heads], w, name=f"{name} (sampled heads)")


def test_dq_kernel_env_rejects_unknown_value(pkg, monkeypatch):
    q, k, v, dout = (t.to("cuda", BF) for t in _inputs(1, 8, 8, 1, 1))
    out, lse = torch.ops.anima_flat.fa_fwd(q, k, v)
    monkeypatch.setenv("AA_DQ_KERNEL", "zz")
    with pytest.raises(ValueError, match="AA_DQ_KERNEL"):
        torch.ops.anima_flat.fa_bwd(dout, q, k, v, out, lse)


@pytest.mark.parametrize(
    "Sq,Sk,H,kernel",
    [
        (128, 64, 16, "2g"),
        (129, 64, 16, "ks"),
        (128, 65, 16, "ks"),
        (20, 60, 16, "2g"),
        (200, 64, 260, "2g"),  # a tail of 4 items behind a whole round
    ],
)
def test_dq_kernel_by_size(pkg, monkeypatch, Sq, Sk, H, kernel):
    """Short calls and tails of one key tile keep the two-group kernel: dQ has its bits, not the other's
    (with up to 32 keys the two sum the same products in the same order: no such case here)."""
    q, k, v, dout = _inputs(1, Sq, Sk, H, 70)
    dq = _gpu_backward(q, k, v, dout)[0]
    forced = {}
    for name in ("2g", "ks"):
        monkeypatch.setenv("AA_DQ_KERNEL", name)
        forced[name] = torch.equal(_gpu_backward(q, k, v, dout)[0], dq)
    assert forced == {name: name == kernel for name in forced}
