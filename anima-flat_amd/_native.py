"""Native dispatcher kernels of the package's torch ops (csrc/torch_ops.cpp).

`attach(qualname, impl)` gives a registered op CUDA and AutogradCUDA kernels
that call libanima_attn.so straight from C++; `impl`, the op's Python function,
stays the kernel of every other dispatch key and takes the calls the native
kernels hand back (copies, other dtypes, errors). The extension is built with
the library (build.py); without it the ops run the same HIP kernels through
Python, which is reported once; so they do if it does not load.
"""

from __future__ import annotations

import importlib.util
import warnings
from pathlib import Path

import torch  # noqa: F401  (the extension binds to torch's libraries)

from . import _lib

EXT_PATH = Path(__file__).resolve().with_name("_anima_torch.so")

NATIVE_OPS = frozenset({
    "anima_flat::fa_fwd", "anima_flat::fa_fwd_nolse", "anima_flat::fa_fwd_k", "anima_flat::fa_bwd",
    "anima_flat_amd::fa_fwd_k_ctx", "anima_flat_amd::attend_d384",
    "anima_flat::qkv_norm_rope", "anima_flat::qkv_norm_rope_v", "anima_flat::qkv_norm_rope_bwd",
    "anima_flat::head_norm", "anima_flat::head_norm_bwd",
    "anima_flat_amd::qkv_proj_norm_rope", "anima_flat_amd::proj_head_norm",
    "anima_flat_amd::kv_proj_norm",
})

_ext = None
_missing = False


def _unusable(why: str) -> None:
    """Say once that this process calls every op through Python, and why."""
    global _missing
    _missing = True
    warnings.warn(f"{EXT_PATH.name} {why}: every op call of this process goes through Python "
                  "(`python anima-flat_amd/build.py` builds it)", RuntimeWarning, stacklevel=5)


def _version_error(module) -> str | None:
    """Why the extension must not be used: the argument structs it was compiled with, the
    library it is linked to and this package have to agree on the ABI version."""
    versions = module.abi_version(), module.library_abi_version(), _lib.ABI_VERSION
    if len(set(versions)) == 1:
        return None
    return "was compiled for ABI version {}, runs on a library of {} and is called by a package of {}".format(*versions)


def _load():
    """The extension module, or None (reported once) when it is not built or does not load
    (another torch's, a library it cannot find)."""
    global _ext, _missing
    if _ext is None and not _missing:
        if not _lib.LIB_PATH.exists():
            # Nothing to call either: said when the library is there in the end.
            _missing = True
            _lib.on_load.append(lambda: _unusable("was not built when the package was imported"))
            return None
        if not EXT_PATH.exists():
            _unusable("is not built")
            return None
        try:
            spec = importlib.util.spec_from_file_location("_anima_torch", EXT_PATH)
            module = importlib.util.module_from_spec(spec)
            spec.loader.exec_module(module)
            error = _version_error(module)
        except (ImportError, OSError, AttributeError) as e:
            error = f"does not load ({e})"
        if error is not None:
            _unusable(error)
            return None
        _ext = module
    return _ext


def attach(qualname: str, impl) -> None:
    """Give op `qualname` its native kernels, if it has any."""
    if qualname in NATIVE_OPS:
        ext = _load()
        if ext is not None:
            ext.attach(qualname, impl)
