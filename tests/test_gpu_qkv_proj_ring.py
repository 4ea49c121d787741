"""The fused projections' four-stage tile (128 x 1 section, three stages in flight) against
the two-stage one, bit for bit (same accumulation order), where its ring can go wrong: fewer
K stages than it holds, a last stage of 32, more stages than one turn; and its default route."""

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
    if K >= 1536:
        monkeypatch.delenv("AA_PROJ_TILE")
        outs["default"] = proj.kv_proj_norm(x, w, nw, 3, 1e-6)
    for tile, (k, v) in outs.items():
        assert torch.equal(k, outs["a"][0]) and torch.equal(v, outs["a"][1]), tile
