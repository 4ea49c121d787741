"""The ops' native dispatcher kernels against their Python functions: the same
results, autograd behaviour and errors, whichever of the two a call reaches."""

from __future__ import annotations

import importlib
import re
import shutil
import subprocess
import sys
import types
import warnings

import pytest
import torch
import torch._dynamo.compiled_autograd

import __graft_entry__
from oracle import attn_oracle as ref

BF = torch.bfloat16


def _qkv(device="cuda", Sq=70, Sk=90, H=2):
    g = torch.Generator().manual_seed(3)
    return [ref.bf16_normal((1, s, H, 128), g).to(device, BF) for s in (Sq, Sk, Sk)]


def _fake_forward(pkg):
    q, k, v = (torch.empty(2, s, 3, 128, dtype=BF, device="cuda", requires_grad=True) for s in (5, 7, 7))
    out = pkg.attention(q, k, v)
    assert out.shape == (2, 5, 384) and out.device.type == "cuda" and out.requires_grad
    return out, (q, k, v)


def test_fake_forward(pkg):
    """Fake CUDA tensors reach the fake implementations through the native autograd kernels
    (no GPU is touched)."""
    from torch._subclasses.fake_tensor import FakeTensorMode

    with FakeTensorMode():
        _fake_forward(pkg)


@pytest.mark.gpu
def test_fake_backward(pkg):
    from torch._subclasses.fake_tensor import FakeTensorMode

    with FakeTensorMode():
        out, leaves = _fake_forward(pkg)
        grads = torch.autograd.grad(out, leaves, torch.empty_like(out))
        assert [g.shape for g in grads] == [t.shape for t in leaves]


@pytest.mark.gpu
@pytest.mark.parametrize("form", ["plain", "head_major", "misaligned", "last_dim_strided"])
def test_same_result_from_both_paths(pkg, form):
    """Views the native kernel reads in place and views that go to the Python function (which
    copies them) give the bits of a plain call."""
    q, k, v = _qkv()
    if form == "head_major":
        kx = k.transpose(1, 2).contiguous().transpose(1, 2)
    elif form == "misaligned":
        kx = torch.empty(k.numel() + 4, dtype=BF, device="cuda")[4:].view(k.shape).copy_(k)
    elif form == "last_dim_strided":
        kx = torch.stack((k, k), -1)[..., 0]
    else:
        kx = k.clone()
    want = torch.ops.anima_flat.fa_fwd(q, k, v)
    got = torch.ops.anima_flat.fa_fwd(q, kx, v)
    direct = importlib.import_module("anima_flat_amd.attention")._launch_fwd(q, kx, v, want_lse=True)
    assert all(torch.equal(a, b) for a, b in zip(want, got))
    assert all(torch.equal(a, b) for a, b in zip(want, direct))


@pytest.mark.gpu
def test_autograd_behaviour(pkg):
    """Saved tensors pass the saved-tensor hooks, a second backward needs retain_graph, ops
    without a backward raise on it and not before, and so does a double backward."""
    leaves = [t.requires_grad_(True) for t in _qkv()]
    seen = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: (seen.append(tuple(t.shape)), t.clone())[1], lambda t: t):
        out = pkg.attention(*leaves)
    assert len(seen) == 5  # q, k, v, out, lse
    grads = torch.autograd.grad(out.float().pow(2).sum(), leaves, retain_graph=True)
    again = torch.autograd.grad(out.float().pow(2).sum(), leaves)
    assert all(torch.equal(a, b) for a, b in zip(grads, again))
    with pytest.raises(RuntimeError, match="second time"):
        torch.autograd.grad(out.float().pow(2).sum(), leaves)

    nolse = torch.ops.anima_flat.fa_fwd_nolse(*leaves)
    assert nolse.requires_grad
    with pytest.raises(RuntimeError, match="fa_fwd_nolse.default but no autograd formula"):
        nolse.sum().backward()

    first = torch.autograd.grad(pkg.attention(*leaves).float().pow(2).sum(), leaves, create_graph=True)
    with pytest.raises(RuntimeError, match="fa_bwd.default but no autograd formula"):
        torch.autograd.grad(first[0].float().sum(), leaves)


@pytest.mark.gpu
def test_errors_are_the_python_functions(pkg):
    q, k, v = _qkv()
    with pytest.raises(ValueError, match="only bfloat16"):
        torch.ops.anima_flat.fa_fwd(q.half(), k.half(), v.half())
    with pytest.raises(ValueError, match="same shape"):
        torch.ops.anima_flat.fa_fwd(q, k, v[:, :5])
    with pytest.raises(ValueError, match="seqused_k must be"):
        torch.ops.anima_flat.fa_fwd_k(q, k, v, torch.ones(2, dtype=torch.int32, device="cuda"))
    with pytest.raises(ValueError, match="CUDA tensors required"):
        pkg.attention(q.cpu(), k.cpu(), v.cpu())


def _op_cases():
    """Arguments of every op with native kernels, by qualified name: fp32 norm weights and
    tables whose values bf16 holds exactly."""
    q, k, v = _qkv()
    g = torch.Generator().manual_seed(5)

    def n(*shape):
        return ref.bf16_normal(shape, g).cuda()

    dout, x, dy = n(1, 70, 2, 128).to(BF), n(1, 40, 256).to(BF), n(1, 40, 2, 128).to(BF)
    qkv, grads = n(1, 40, 768).to(BF), [n(1, 40, 2, 128).to(BF) for _ in range(3)]
    qw, kw, cos, sin = n(128), n(128), n(40, 64), n(40, 64)
    q384, k384, v384 = (n(1, 50, 2, 384).to(BF) for _ in range(3))
    lens = torch.tensor([33], dtype=torch.int32, device="cuda")
    out, lse = torch.ops.anima_flat.fa_fwd(q, k, v)
    eps = 1e-6
    return {
        "anima_flat::fa_fwd": (q, k, v),
        "anima_flat::fa_fwd_nolse": (q, k, v),
        "anima_flat::fa_fwd_k": (q, k, v, lens),
        "anima_flat::fa_bwd": (dout, q, k, v, out, lse),
        "anima_flat_amd::fa_fwd_k_ctx": (q, k, v, lens, torch.log(90.0 - lens)),
        "anima_flat_amd::attend_d384": (q384, k384, v384),
        "anima_flat::qkv_norm_rope": (qkv, qw, kw, cos, sin, 2, eps),
        "anima_flat::qkv_norm_rope_v": (qkv, qw, kw, cos, sin, 2, eps),
        "anima_flat::qkv_norm_rope_bwd": (qkv, *grads, qw, kw, cos, sin, 2, eps),
        "anima_flat::head_norm": (x, qw, 2, eps),
        "anima_flat::head_norm_bwd": (x, dy, qw, 2, eps),
        "anima_flat_amd::qkv_proj_norm_rope": (x, n(768, 256).to(BF), qw, kw, cos, sin, 2, eps),
        "anima_flat_amd::proj_head_norm": (x, n(256, 256).to(BF), qw, 2, eps),
        "anima_flat_amd::kv_proj_norm": (x, n(512, 256).to(BF), kw, 2, eps),
    }


def _python_function(qualname):
    """The function that op `qualname` was registered with."""
    for name in ("attention", "vae", "kernels.rope", "kernels.proj"):
        for op in vars(importlib.import_module(f"anima_flat_amd.{name}")).values():
            if isinstance(op, torch.library.CustomOpDef) and op._qualname == qualname:
                return op._init_fn
    raise AssertionError(qualname)


@pytest.mark.gpu
@pytest.mark.parametrize("weights", [torch.float32, BF])
def test_python_functions_give_the_same_bits(pkg, proj, weights):
    """What a call gets without the extension, for every op it serves, also where the Python
    function converts norm weights and tables (each to a tensor that lives until the launch:
    their values are the same, so are all bits but those of the weights' own gradients)."""
    cases = _op_cases()
    assert set(cases) == importlib.import_module("anima_flat_amd._native").NATIVE_OPS
    for name, args in cases.items():
        ns, op = name.split("::")
        want = getattr(getattr(torch.ops, ns), op)(*args)
        cast = args if name.split("::")[1].startswith("fa_") else [
            a.to(weights) if isinstance(a, torch.Tensor) and a.dtype == torch.float32 else a for a in args]
        got = _python_function(name)(*cast)
        want, got = ([t] if isinstance(t, torch.Tensor) else list(t) for t in (want, got))
        assert len(want) == len(got)
        assert all(torch.equal(a.to(b.dtype), b) for a, b in zip(want, got)), name


@pytest.mark.gpu
def test_functional_transforms(pkg):
    """vmap batches a call without gradients; functorch's derivatives and forward mode, which
    no op here has, are refused and give no wrong result."""
    import torch.autograd.forward_ad as fwad

    q, k, v = _qkv()
    want = pkg.attention(q, k, v)
    assert torch.equal(torch.func.vmap(pkg.attention)(q[None], k[None], v[None])[0], want)
    leaf = q.clone().requires_grad_()
    scale = torch.arange(1.0, 3.0, device="cuda").to(BF)
    batched = torch.func.vmap(lambda x: pkg.attention(leaf, k, v) * x)(scale)  # of a constant
    assert batched.requires_grad and torch.equal(batched[1], 2 * want)
    with pytest.raises(RuntimeError, match="functorch transforms"):
        torch.func.grad(lambda a: pkg.attention(a, k, v).float().sum())(q)
    with pytest.raises(RuntimeError, match="functorch transforms"):
        torch.func.vjp(lambda a: pkg.head_norm(a, torch.ones(128, device="cuda"), 2), q.flatten(2))
    with fwad.dual_level(), pytest.raises(NotImplementedError, match="forward mode AD"):
        pkg.attention(fwad.make_dual(leaf, torch.ones_like(q)), k, v)


@pytest.mark.gpu
@pytest.mark.parametrize("path", ["attention", "head_norm", "prologue"])
def test_compiled_autograd(pkg, path):
    """torch.compile's tracing of the backward goes through the ops' autograd nodes."""
    q, k, v = _qkv()
    w, cos, sin = torch.ones(128, device="cuda"), *torch.randn(2, 70, 64, device="cuda")

    def run(a):
        if path == "attention":
            return pkg.attention(a, k, v)
        if path == "head_norm":
            return pkg.head_norm(a.flatten(2), w, 2)
        qkv = torch.cat([t.flatten(2) for t in (a, k[:, :70], v[:, :70])], -1)
        return pkg.qkv_norm_rope(qkv, w, w, cos, sin, 2)[0]  # two outputs without a gradient

    leaf = q.clone().requires_grad_()
    run(leaf).float().pow(2).sum().backward()
    want, leaf.grad = leaf.grad, None
    with torch._dynamo.compiled_autograd._enable(torch.compile(backend="eager")):
        run(leaf).float().pow(2).sum().backward()
    assert torch.equal(leaf.grad, want)


@pytest.mark.gpu
def test_streams_and_threads(pkg):
    """Calls from several threads, each on its own stream, forward and backward, with their
    temporaries (converted weights, workspaces) in use at once: the bits of a call alone."""
    import threading

    g = torch.Generator().manual_seed(6)
    qw, cos, sin = (ref.bf16_normal(s, g).to("cuda", BF) for s in ((128,), (300, 64), (300, 64)))
    inputs = [ref.bf16_normal((1, 300, 3 * 512), g).to("cuda", BF) for _ in range(4)]

    def step(x):
        x = x.detach().requires_grad_()
        q, k, v = pkg.qkv_norm_rope(x, qw, qw, cos, sin, 4, 1e-6)
        out = pkg.attention(q, k, v)
        return out, torch.autograd.grad(out.float().pow(2).sum(), x)[0]

    want = [step(x) for x in inputs]
    torch.cuda.synchronize()
    got = [None] * len(inputs)

    def work(i):
        stream = torch.cuda.Stream()
        with torch.cuda.stream(stream):
            for _ in range(10):
                got[i] = step(inputs[i])
        stream.synchronize()

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(inputs))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for a, b in zip(want, got):
        assert torch.equal(a[0], b[0]) and torch.equal(a[1], b[1])


@pytest.mark.gpu
def test_weights_in_another_dtype(pkg):
    """bf16 norm weights and tables are converted, each to a tensor of its own that lives
    until the launch (test_python_functions_give_the_same_bits: on the Python path)."""
    g = torch.Generator().manual_seed(4)
    qkv = ref.bf16_normal((1, 40, 3 * 256), g).to("cuda", BF)
    qw, kw = (ref.bf16_normal((128,), g).cuda() for _ in range(2))
    cos, sin = (ref.bf16_normal((40, 64), g).cuda() for _ in range(2))
    want = pkg.qkv_norm_rope(qkv, qw, kw, cos, sin, 2, 1e-6)
    got = pkg.qkv_norm_rope(qkv, *(t.to(BF) for t in (qw, kw, cos, sin)), 2, 1e-6)
    assert all(torch.equal(a, b) for a, b in zip(want, got))


# ------------------------------------------------- loading the extension --


@pytest.fixture
def native(pkg, monkeypatch):
    """anima_flat_amd._native as at its import, to be loaded again."""
    module = importlib.import_module("anima_flat_amd._native")
    if not (module.EXT_PATH.exists() and pkg._lib.LIB_PATH.exists()):
        pytest.skip("not built (run __graft_entry__.build())")
    monkeypatch.setattr(module, "_ext", None)
    monkeypatch.setattr(module, "_missing", False)
    monkeypatch.setattr(pkg._lib, "on_load", [])
    return module


def test_extension_version_is_the_headers(native):
    text = (__graft_entry__.ROOT / "include" / "anima_attn.h").read_text()
    ext = native._load()
    assert ext.abi_version() == int(re.search(r"#define AA_ABI_VERSION (\d+)", text)[1])
    assert ext.abi_version() == ext.library_abi_version()


@pytest.mark.parametrize("compiled,library", [(2, 3), (3, 4), (4, 4)])
def test_another_versions_extension_is_refused(native, compiled, library):
    """Structs of another layout than the library's, also where library and package agree."""
    module = types.SimpleNamespace(abi_version=lambda: compiled, library_abi_version=lambda: library)
    assert f"compiled for ABI version {compiled}" in native._version_error(module)


def test_missing_extension_is_reported_once(native, monkeypatch, tmp_path):
    monkeypatch.setattr(native, "EXT_PATH", tmp_path / "_anima_torch.so")
    with pytest.warns(RuntimeWarning, match="is not built"):
        assert native._load() is None
    with warnings.catch_warnings():
        warnings.simplefilter("error")
        assert native._load() is None


def test_library_built_after_the_import(pkg, native, monkeypatch, tmp_path):
    """With nothing built there is nothing to report, until the library is there."""
    built = pkg._lib.LIB_PATH
    monkeypatch.setattr(pkg._lib, "LIB_PATH", tmp_path / "libanima_attn.so")
    with warnings.catch_warnings():
        warnings.simplefilter("error")
        assert native._load() is None
    monkeypatch.setattr(pkg._lib, "LIB_PATH", built)
    monkeypatch.setattr(pkg._lib, "_lib", None)
    with pytest.warns(RuntimeWarning, match="was not built when the package was imported"):
        pkg._lib.lib()


def test_import_with_an_extension_that_does_not_load(native, tmp_path):
    """The package imports, says so and keeps its Python ops (an extension of another torch)."""
    copy = tmp_path / "anima-flat_amd"
    shutil.copytree(__graft_entry__.PKG_DIR, copy, ignore=shutil.ignore_patterns("_build", "csrc", "__pycache__"))
    (copy / "_anima_torch.so").write_bytes(b"no shared object")
    code = f"""
import pathlib, sys, warnings
sys.path.insert(0, {str(__graft_entry__.ROOT)!r})
import torch, __graft_entry__ as g
g.PKG_DIR = pathlib.Path({str(copy)!r})
with warnings.catch_warnings(record=True) as seen:
    warnings.simplefilter("always")
    pkg = g.load_package()
assert pkg.__file__.startswith({str(copy)!r})
assert [w for w in seen if "does not load" in str(w.message)] and len(seen) == 1, [str(w.message) for w in seen]
assert pkg._lib.available() and not pkg.use_fa4(torch.empty(1, dtype=torch.bfloat16))
assert torch.ops.anima_flat.fa_fwd(*[torch.empty(1, 2, 1, 128, dtype=torch.bfloat16, device="meta")] * 3)[0].is_meta
"""
    proc = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=300)
    assert proc.returncode == 0, proc.stderr
