"""The fused projections' four-stage tile (128 x 1 section, three stages in flight) against
the two-stage ones, bit for bit (same accumulation order), where its ring can go wrong: fewer
K stages than it holds, a last stage of 32, more stages than one turn; and its epilogues. Every
tile gives the same bits, so nothing here tells which one a call takes by default."""

from __future__ import annotations

import pytest
import torch

from oracle import attn_oracle as ref

pytestmark = pytest.mark.gpu

BF = torch.bfloat16


@pytest.mark.parametrize("K", [32, 64, 96, 128, 192, 224, 256, 320, 1568])
def test_four_stage_ring(pkg, proj, monkeypatch, K):
    g = torch.Generator().manual_seed(K)
    x = ref.bf16_normal((1, 133, K), g).to("cuda", BF)
    w = (ref.bf16_normal((2 * 3 * 128, K), g) * K**-0.5).to("cuda", BF)
    nw = (1 + 0.02 * ref.bf16_normal((128,), g)).to("cuda", BF)
    outs = {}
    for tile in "acd":
        monkeypatch.setenv("AA_PROJ_TILE", tile)
        outs[tile] = proj.kv_proj_norm(x, w, nw, 3, 1e-6)
    for tile, (k, v) in outs.items():
        assert torch.equal(k, outs["a"][0]) and torch.equal(v, outs["a"][1]), tile


@pytest.mark.parametrize("H", [1, 2, 3])
def test_four_stage_epilogues(pkg, proj, monkeypatch, H):
    """Norm and rotation (sections of q and k), copy (v) and norm alone, at a ragged last tile."""
    g = torch.Generator().manual_seed(H)
    D = 128 * H
    x = ref.bf16_normal((2, 67, D), g).to("cuda", BF)
    w = (ref.bf16_normal((3 * D, D), g) * D**-0.5).to("cuda", BF)
    qw, kw = (1 + 0.02 * ref.bf16_normal((2, 128), g)).cuda()
    cos, sin = ref.bf16_normal((2, 67, 64), g).cuda()
    outs = {}
    for tile in "abcd":
        monkeypatch.setenv("AA_PROJ_TILE", tile)
        outs[tile] = (*proj.qkv_proj_norm_rope(x, w, qw, kw, cos, sin, H, 1e-6), proj.proj_head_norm(x, w[:D], qw, H, 1e-6))
    for tile in "bcd":
        assert all(torch.equal(a, b) for a, b in zip(outs["a"], outs[tile])), tile
