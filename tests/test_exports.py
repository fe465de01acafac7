"""Every C symbol that libyas.so exports is one that include/yas.h declares:
nothing can be called that the header does not document."""
import os
import re
import shutil
import subprocess

import pytest

from yetanotherslam_amd import native

HEADER = os.path.join(os.path.dirname(__file__), "..", "include", "yas.h")


def test_every_exported_c_symbol_is_declared():
    nm = shutil.which("nm")
    if not nm:
        pytest.skip("nm not available")
    out = subprocess.run([nm, "-D", "--defined-only", native.LIB_PATH], check=True, capture_output=True, text=True).stdout
    exported = set(re.findall(r" T (yas_\w+)$", out, re.M))
    with open(HEADER) as fh:
        declared = set(re.findall(r"\b(yas_[a-z0-9_]+)\s*\(", fh.read()))
    assert len(exported) > 50 and exported <= declared, exported - declared
