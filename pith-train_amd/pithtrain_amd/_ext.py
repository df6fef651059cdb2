"""Loads the native host path (csrc/host/torch_ops.cpp, built in-tree as lib/_pith_torch.so): the torch.library ops
`torch.ops.pithtrain_amd.*` and the fast form of the *_into calls. Like the kernel library it has no fallback: if it has
not been built, importing the operators raises.

Every native function returns False (None) when a call is not of ordinary layout or the library rejected it; nothing has
been launched then, and the caller runs the operator's Python body, which takes every layout and words the errors. A launch
that failed raises PithError at once."""

import importlib.util
import os

import torch  # noqa: F401  (libtorch and the HIP runtime must be in the process first)

from pithtrain_amd import _C

EXT_PATH = os.path.join(os.path.dirname(os.path.abspath(__file__)), "lib", "_pith_torch.so")


def _load():
    if not os.path.exists(EXT_PATH):
        raise ImportError(
            f"{EXT_PATH} is missing: build it with `python -m pithtrain_amd.build` (there is no non-HIP fallback for these operators)"
        )
    spec = importlib.util.spec_from_file_location("_pith_torch", EXT_PATH)
    module = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(module)
    return module


native = _load()
native.set_bodies({"check": _C.check})


def define_op(name: str, body, fake):
    """Attaches the Python body and the fake (shape) implementation of the native op `name`; returns the op."""
    native.set_bodies({name: body})
    torch.library.register_fake(f"pithtrain_amd::{name}", fake)
    return getattr(torch.ops.pithtrain_amd, name).default
