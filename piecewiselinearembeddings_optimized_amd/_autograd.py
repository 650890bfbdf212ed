"""Autograd formulas of the PLE operators.

The contract is the reference's (``src/rtdl_num_embeddings_cuda/_autograd.py:9-96``).
The formulas are registered with the operators by the extension module
(``csrc/ple_autograd.cpp``); this module keeps the reference's submodule name
and checks that they are there.
"""

from __future__ import annotations

import torch

from . import _C as _C  # noqa: F401

for _name in ("forward", "forward_with_bias", "forward_epilogue", "encode"):
    if not torch._C._dispatch_has_kernel_for_dispatch_key(f"rtdl_num_embeddings_cuda::{_name}", "Autograd"):
        raise ImportError(f"the extension module registers no autograd formula for {_name}")
