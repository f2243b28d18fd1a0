"""Loads the native host side (recml_amd/lib/_native.so, built from recml_amd/csrc/native.cpp).

Its functions take a call whose arguments are ready for the kernels as they are, and return None for any other, which
the Python side then checks, converts or reports.
"""

from __future__ import annotations

import importlib.util
import os

import torch
from torch.autograd import forward_ad

from recml_amd import _lib, _lib_block

PATH = os.path.join(os.path.dirname(os.path.abspath(__file__)), "lib", "_native.so")


def has_tangent(*tensors) -> bool:
  """Whether one of the tensors carries a forward-mode tangent: the kernels' results have none, so such a call goes through the
  autograd functions, which refuse it."""
  return any(isinstance(t, torch.Tensor) and forward_ad.unpack_dual(t).tangent is not None for t in tensors)


def _load():
  if not os.path.exists(PATH):
    raise RuntimeError(f"{PATH} is missing: build it with `python -m recml_amd.build`; this package has no CPU fallback")
  _lib.load()
  _lib_block.load()
  spec = importlib.util.spec_from_file_location("recml_amd.lib._native", PATH)
  module = importlib.util.module_from_spec(spec)
  spec.loader.exec_module(module)
  return module


def _other_library() -> bool:
  """Whether other libraries than the packaged ones are to run: every call then goes the Python way."""
  return bool(os.environ.get("RECML_AMD_LIB") or os.environ.get("RECML_AMD_BLOCK_LIB"))


def _decline(*args):
  return None


def _first_call(name):
  """A stand-in that loads the module when it is first called and is replaced by the module's function."""

  def call(*args):
    module = None if _other_library() else _load()
    for n in _FUNCTIONS:
      globals()[n] = _decline if module is None else getattr(module, n)
    return globals()[name](*args)

  return call


_FUNCTIONS = ("attention", "block", "blocks", "embed", "final_norm", "linear", "pack", "mask_lengths", "raised", "norm_gate_bwd", "has_room")
attention, block, blocks, embed, final_norm, linear, pack, mask_lengths, raised, norm_gate_bwd, has_room = (_first_call(n) for n in _FUNCTIONS)
