"""The native host layer, `lib/mq_host.so` (csrc/host/mq_host.cpp): outputs, job records and straight-through nodes without
Python in between.

`native` is the extension module.  It is built with the kernels (`python -m miles_amd.build`); where it is missing or does not
load (another torch, no kernel library beside it), the package is still imported and the first quantizer raises, as it does
for a missing kernel library.
"""

from __future__ import annotations

import importlib.machinery
import importlib.util
import os

import torch  # noqa: F401  (the module links against torch's libraries, which this loads)

from miles_amd import _lib

_PATH = os.path.join(os.path.dirname(os.path.abspath(__file__)), "lib", "mq_host.so")


class _Missing:
    """In the module's place where there is none: blocks of jobs are entered and left, everything else raises."""

    def __init__(self, why: str) -> None:
        self._why = why

    def __getattr__(self, name):
        raise _lib.MilesQuantError(f"{_PATH} {self._why}: build it with `python -m miles_amd.build` (g++, against this torch).")

    def Recorder(self) -> None:       # (jobs are recorded from Python)
        return None

    def enter(self, recorder) -> None:
        pass

    def leave(self) -> None:
        pass


def _load():
    if not os.path.exists(_PATH):
        return _Missing("is missing")
    loader = importlib.machinery.ExtensionFileLoader("mq_host", _PATH)
    try:
        module = importlib.util.module_from_spec(importlib.util.spec_from_loader("mq_host", loader))
        loader.exec_module(module)
    except ImportError as e:
        return _Missing(f"does not load ({e})")
    module.set_error(_lib.MilesQuantError)
    return module


native = _load()
