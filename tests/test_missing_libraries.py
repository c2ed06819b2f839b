"""A package whose libraries are missing or do not load: it is imported and its blocks of jobs are entered and left, and the
first quantizer says what is wrong."""

import os
import shutil
import subprocess
import sys

import pytest

import miles_amd
from miles_amd import _lib

PACKAGE = os.path.dirname(os.path.abspath(miles_amd.__file__))

USE = """
import torch
from miles_amd import _lib, launch
from miles_amd.utils import mxfp4, nvfp4
with launch.deferred() as batch:
    assert len(batch) == 0
with launch.recording() as batch:
    assert batch.records == [] and launch.active_batch() is batch
assert launch.active_batch() is None
x = torch.zeros(4, 32, dtype=torch.bfloat16)
for block in (launch.deferred, launch.recording, None):
    try:
        if block is None:
            launch.submit(_lib.JOB_MXFP8, x, x, x, None, None, 4, 32, 32)
        else:
            with block():
                launch.produce(_lib.JOB_MXFP8, x, 4, 32, 32, 0, 0, (torch.uint8, 4, 32), (torch.uint8, 4, 1))
    except _lib.MilesQuantError as e:
        assert "python -m miles_amd.build" in str(e) and "mq_host.so" in str(e), e
        print("refused")
    assert launch.active_batch() is None
"""


@pytest.mark.parametrize("libraries", ["none", "host_only", "kernels_only", "host_damaged"])
def test_first_use_says_what_is_missing(libraries, tmp_path):
    copy = tmp_path / "miles_amd"
    shutil.copytree(PACKAGE, copy, ignore=shutil.ignore_patterns("lib", "__pycache__", "csrc"))
    os.mkdir(copy / "lib")
    built = os.path.dirname(_lib.lib_path())
    for name, kinds in (("mq_host.so", ("host_only",)), ("libmiles_quant.so", ("kernels_only", "host_damaged"))):
        if libraries in kinds:
            shutil.copy(os.path.join(built, name), copy / "lib" / name)
    if libraries == "host_damaged":
        (copy / "lib" / "mq_host.so").write_bytes(b"\x7fELF, cut short")
    done = subprocess.run([sys.executable, "-c", USE], cwd=tmp_path, env=dict(os.environ, PYTHONPATH=str(tmp_path)),
                          stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=300)
    assert done.returncode == 0, done.stdout
    assert done.stdout.split() == ["refused"] * 3
