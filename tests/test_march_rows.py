"""How many rays a ray cast puts in a wavefront (march_rows in
yetanotherslam_amd/csrc/yas_raycast_dev.hpp), compiled for the host here
(hipcc): as few as leave no wavefront waiting for a place on the CUs that there
are, of a whole device, of a partition or of a stream's mask."""
import ctypes
import os
import shutil
import subprocess

import pytest

HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
CSRC = os.path.join(os.path.dirname(__file__), "..", "yetanotherslam_amd", "csrc")
SRC = r'''
#include "yas_raycast_dev.hpp"
extern "C" int rows(int w, int h, int cus) { return yas::march_rows(w, h, cus); }
extern "C" int tiles(int w, int h, int r) { return yas::march_tiles(w, h, r); }
'''


def test_rows_fill_the_places_of_the_cus_there_are(tmp_path):
    if not os.path.exists(HIPCC):
        pytest.skip("hipcc not available")
    src, so = tmp_path / "s.hip", tmp_path / "s.so"
    src.write_text(SRC)
    subprocess.run([HIPCC, "-x", "hip", "--offload-arch=gfx950", "-std=c++17", "-O2", "-ffp-contract=off", "-shared",
                    "-fPIC", "-I", CSRC, "-I", os.path.join(CSRC, "..", "..", "include"), str(src), "-o", str(so)],
                   check=True, capture_output=True)
    L = ctypes.CDLL(str(so))
    whole = {(160, 120): 1, (320, 240): 2, (480, 360): 4, (640, 480): 8, (1280, 960): 8}
    for (w, h), r in whole.items():
        assert L.rows(w, h, 256) == r
    for cus in (256, 128, 64, 32, 1):
        for w in range(8, 2600, 72):
            h = w * 3 // 4 // 8 * 8 or 8
            r = L.rows(w, h, cus)
            assert r in (1, 2, 4, 8)
            # (w * h rays: tiles at the right and lower edges are partly empty)
            assert w * h <= 24 * cus * 8 * r or r == 8
            assert r == 1 or w * h > 24 * cus * 8 * (r // 2)
            assert L.tiles(w, h, r) * 4 * 8 * r >= w * h
