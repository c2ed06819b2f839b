"""The native host layer, `lib/mq_host.so` (csrc/host/mq_host.cpp): outputs, job records and straight-through nodes without
Python in between.

`native` is the extension module.  It is built with the kernels (`python -m miles_amd.build`); where it is missing, the first
use raises like a missing kernel library does.
"""

from __future__ import annotations

import importlib.machinery
import importlib.util
import os

import torch  # noqa: F401  (the module links against torch's libraries, which this loads)

from miles_amd import _lib

_PATH = os.path.join(os.path.dirname(os.path.abspath(__file__)), "lib", "mq_host.so")


class _Missing:
    def __getattr__(self, name):
        raise _lib.MilesQuantError(f"{_PATH} is missing: build it with `python -m miles_amd.build` (g++, against this torch).")


def _load():
    if not os.path.exists(_PATH):
        return _Missing()
    loader = importlib.machinery.ExtensionFileLoader("mq_host", _PATH)
    module = importlib.util.module_from_spec(importlib.util.spec_from_loader("mq_host", loader))
    loader.exec_module(module)
    module.set_error(_lib.MilesQuantError)
    return module


native = _load()
