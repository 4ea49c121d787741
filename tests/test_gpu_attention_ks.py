"""GPU parity of the key-split forward (one workgroup per 64 queries, the keys
split over its four waves and merged in LDS) against the CPU oracle, at the
edges of its tiles: query blocks of 64, key tiles of 64 dealt to 4 waves, a last
tile that re-reads its last row, waves without keys."""

from __future__ import annotations

import pytest
import torch

from conftest import parity
from oracle import attn_oracle as ref

pytestmark = pytest.mark.gpu

BF = torch.bfloat16
# LSE: the log of a sum of fp32 probabilities. Relative errors of the sum: its
# exp2 arguments s c - m c (2^-24 of up to ~300) and the device's exp2 and log2
# (1 ulp each), together below 5e-5.
LSE_TOL = {"max_abs": 1e-4, "rel_l2": 1e-5}


def _inputs(B, Sq, Sk, H, seed):
    g = torch.Generator().manual_seed(seed)
    return [ref.bf16_normal(s, g) for s in ((B, Sq, H, 128), (B, Sk, H, 128), (B, Sk, H, 128))]


@pytest.mark.parametrize(
    "B,Sq,Sk,H,lens",
    [
        (1, 1, 1, 1, None),
        (1, 63, 64, 2, None),  # one key tile: three waves hold no keys
        (2, 64, 65, 3, None),  # two tiles, the second of one key
        (1, 65, 255, 2, None),  # every wave one tile, the last partial
        (1, 100, 256, 1, None),
        (1, 129, 257, 2, None),  # a second round of tiles for wave 0 only
        (2, 70, 513, 2, [513, 1]),  # one key
        (3, 33, 300, 2, [63, 64, 192]),  # shorter than a tile, whole tiles
        (1, 300, 1000, 8, None),
        (1, 128, 4100, 2, None),  # many tiles per wave (lazy rescale)
    ],
)
def test_key_split_forward(pkg, monkeypatch, B, Sq, Sk, H, lens):
    q, k, v = _inputs(B, Sq, Sk, H, 100 + Sq + Sk)
    seq = torch.tensor(lens if lens is not None else [Sk] * B, dtype=torch.int32)
    kd, vd = k.to("cuda", BF), v.to("cuda", BF)
    for b, n in enumerate(seq.tolist()):  # rows past a key length hold anything
        kd[b, n:] = float("nan")
        vd[b, n:] = float("inf")
    monkeypatch.setenv("AA_FWD_KERNEL", "ks")
    qd = q.to("cuda", BF)
    if lens is None:
        out, lse = torch.ops.anima_flat.fa_fwd(qd, kd, vd)
    else:
        out, lse = torch.ops.anima_flat.fa_fwd_k(qd, kd, vd, seq.to("cuda"))
    pad = torch.log((Sk + 5 - seq).float())
    fused = pkg.cross_attention_trimmed(qd, kd, vd, seq.to("cuda"), pad.to("cuda"))
    torch.cuda.synchronize()
    eo, el = ref.attention_lse(q, k, v, seq)
    parity(out, eo, name="out")
    if lens is None:  # the instance that leaves the LSE out
        assert torch.equal(torch.ops.anima_flat.fa_fwd_nolse(qd, kd, vd), out)
    parity(lse, el, **LSE_TOL, name="lse")
    parity(fused.view(B, Sq, H, 128), ref.cross_attention_trimmed(q, k, v, seq, pad), name="fused")


def test_key_split_strides_and_route(pkg, monkeypatch):
    """The default rule takes it for 512 queries of 16 heads, with the same bits as when
    forced, and it reads strided views (v inside a fused projection) in place."""
    g = torch.Generator().manual_seed(7)
    qkv = ref.bf16_normal((1, 512, 3, 16, 128), g).to("cuda", BF)
    q, k, v = (qkv[:, :, i] for i in range(3))
    a = pkg.attention(q, k, v)
    monkeypatch.setenv("AA_FWD_KERNEL", "ks")
    b = pkg.attention(q, k, v)
    assert torch.equal(a, b)
    e = ref.attention_sdpa(*(t.float().cpu() for t in (q, k, v)))
    parity(a.view(1, 512, 16, 128), e, name="strided")


def test_key_split_growing_scores(pkg, monkeypatch):
    """Scores that grow along the keys by ~28 log2 units per tile: every wave raises its
    maximum at each of its tiles, and most of the waves' partial results weigh nothing."""
    g = torch.Generator().manual_seed(8)
    q, k, v = _inputs(1, 64, 700, 1, 9)
    u = torch.randn(128, generator=g)
    u = u / u.norm()
    q = (q + 60.0 * u).to(BF).float()
    k = (k + torch.linspace(0.0, 40.0, 700)[None, :, None, None] * u).to(BF).float()
    monkeypatch.setenv("AA_FWD_KERNEL", "ks")
    out, lse = torch.ops.anima_flat.fa_fwd(*(t.to("cuda", BF) for t in (q, k, v)))
    eo, el = ref.attention_lse(q, k, v, None)
    parity(out, eo, name="out")
    parity(lse, el, **LSE_TOL, name="lse")


@pytest.mark.parametrize("S,kernel", [(2049, "pp"), (2560, "pp"), (2561, "1w")])
def test_kernel_by_key_length(pkg, monkeypatch, S, kernel):
    """The default rule's kernel on both sides of the two-group kernel's longest key range:
    the bits of that kernel when forced, and the oracle's values on some rows."""
    g = torch.Generator().manual_seed(S)
    q, k, v = (ref.bf16_normal((1, S, 16, 128), g) for _ in range(3))
    d = [t.to("cuda", BF) for t in (q, k, v)]
    out = pkg.attention(*d).view(1, S, 16, 128)
    monkeypatch.setenv("AA_FWD_KERNEL", kernel)
    assert torch.equal(pkg.attention(*d).view(1, S, 16, 128), out)
    rows = [0, S // 2, S - 1]
    parity(out[:, rows], ref.attention_sdpa(q[:, rows], k, v), name="rows")


@pytest.mark.parametrize("first,last", [(0, 64), (64, 128), (192, 256), (0, 256), (320, 500), (448, 500), (0, 500)])
def test_key_split_infinite_scores(pkg, monkeypatch, first, last):
    """Keys first .. last - 1 at a score of -inf, in steps of the 64-key tiles dealt to the
    waves: a wave's first tile, its last, every wave's first, all. They weigh nothing; with no
    other key the output is 0 and the LSE -inf, as for an empty key range."""
    q, k, v = _inputs(1, 70, 500, 2, 40)
    q[..., 0], k[..., 0] = 1.0, 0.0  # column 0 of a key: added to each of its scores
    k[:, first:last] = 0.0
    k[:, first:last, :, 0] = float("-inf")
    monkeypatch.setenv("AA_FWD_KERNEL", "ks")
    d = [t.to("cuda", BF) for t in (q, k, v)]
    out, lse = torch.ops.anima_flat.fa_fwd(*d)
    assert torch.equal(torch.ops.anima_flat.fa_fwd_nolse(*d), out)
    if last - first == 500:
        assert not out.any() and torch.isneginf(lse).all()
        return
    keep = [j for j in range(500) if not first <= j < last]
    eo, el = ref.attention_lse(q, k[:, keep], v[:, keep], None)
    parity(out, eo, name="out")
    parity(lse, el, **LSE_TOL, name="lse")


@pytest.mark.parametrize("value", [float("nan"), float("inf")])
def test_key_split_rows_stay_apart(pkg, monkeypatch, value):
    """Query rows that hold no finite number give NaN, every other row what it gives without
    them (32 queries share an MFMA's columns)."""
    q, k, v = _inputs(1, 100, 300, 2, 50)
    monkeypatch.setenv("AA_FWD_KERNEL", "ks")
    d = [t.to("cuda", BF) for t in (q, k, v)]
    want, want_lse = torch.ops.anima_flat.fa_fwd(*d)
    rows = [3, 40, 62, 99]
    d[0][:, rows] = value
    others = [j for j in range(100) if j not in rows]
    out, lse = torch.ops.anima_flat.fa_fwd(*d)
    nolse = torch.ops.anima_flat.fa_fwd_nolse(*d)
    assert torch.equal(nolse.isnan(), out.isnan()) and torch.equal(nolse[:, others], out[:, others])
    # Their row sums are taken again from scores summed in another order: O within a bf16 step.
    assert torch.allclose(out[:, others].float(), want[:, others].float(), rtol=2.0**-7, atol=0)
    assert torch.equal(lse[..., others], want_lse[..., others])
    assert out[:, rows].isnan().all() and lse[..., rows].isnan().all()


@pytest.mark.parametrize("Sk,key", [(130, 120), (130, 3), (700, 638), (50, 20)])
def test_key_split_infinite_value(pkg, monkeypatch, Sk, key):
    """An infinite value makes its column infinite, not NaN, also near the end of a key range
    that is no whole number of tiles."""
    q, k, v = (t.to("cuda", BF) for t in _inputs(1, 70, Sk, 2, 60))
    monkeypatch.setenv("AA_FWD_KERNEL", "ks")
    want = torch.ops.anima_flat.fa_fwd_nolse(q, k, v)
    v[:, key, :, 5] = float("inf")
    out = torch.ops.anima_flat.fa_fwd_nolse(q, k, v)
    assert torch.isposinf(out[..., 5]).all()
    out[..., 5] = want[..., 5]
    assert torch.equal(out, want)


@pytest.mark.parametrize(
    "B,Sk,kernel",
    [
        (27, 2304, "pp"),  # 432 work items of 256 queries: 1.69 rounds of 256
        (28, 2304, "1w"),  # 1.75
        (16, 2304, "1w"),  # one whole round
        (16, 2048, "pp"),
        (32, 2049, "1w"),  # two
    ],
)
def test_kernel_by_rounds(pkg, monkeypatch, B, Sk, kernel):
    """Beyond 2048 keys the two-group kernel takes only calls that fill their last round in
    part: the bits of the named kernel, not of the other."""
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("rounds are counted for 256 CUs")
    g = torch.Generator(device="cuda").manual_seed(B)
    q, k, v = (torch.randn(B, s, 16, 128, generator=g, device="cuda").to(BF) for s in (256, Sk, Sk))
    out = pkg.attention(q, k, v)
    forced = {}
    for name in ("pp", "1w"):
        monkeypatch.setenv("AA_FWD_KERNEL", name)
        forced[name] = torch.equal(pkg.attention(q, k, v), out)
    assert forced == {name: name == kernel for name in forced}
