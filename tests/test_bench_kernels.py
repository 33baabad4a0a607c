"""The kernels that bench.py looks up in the counter summaries exist under
those names in the library built here, and the committed summaries hold them."""

import json
import os
import re
import shutil
import subprocess

import pytest

import bench
from azplugins_amd import build

ROOT = os.path.dirname(os.path.abspath(bench.__file__))


def _names():
    with open(os.path.join(ROOT, "bench.py")) as fh:
        text = fh.read()
    return sorted(set(re.findall(r'"(void azp::k_\w+<[^"]*>\(azp::\w+\))"', text)) | {bench.HEADLINE_KERNEL})


def test_kernel_names_are_in_the_library():
    nm = shutil.which("nm")
    if nm is None:
        pytest.skip("no nm")
    text = subprocess.run([nm, "-C", build.LIB], capture_output=True, text=True, check=True).stdout
    symbols = {line.split(" ", 2)[2] for line in text.splitlines() if line[:1] != " "}
    names = _names()
    assert len(names) >= 4
    for name in names:
        assert name in symbols, name


def test_summaries_hold_the_kernels():
    held = set()
    for fname in bench.KERNEL_SOURCES:
        with open(os.path.join(ROOT, "profiles", fname)) as fh:
            held |= set(json.load(fh)["kernels"])
    for name in _names():
        assert name in held, name
