"""Fusion takes the same image sizes from uint16 depth as from float depth,
whether it converts the image or reads it in place."""
import ctypes

import numpy as np
import pytest

from yetanotherslam_amd import native
from yetanotherslam_amd import rgbdfusion as rf

pytestmark = pytest.mark.gpu


def test_u16_images_beyond_the_float_limit_are_refused(gpu):
    import torch
    m = rf.MapStruct(np.float32([500, 500, 320, 240]), 1 << 10, 1 << 8, 0.01, 0.04)
    buf = torch.zeros(16, dtype=torch.int16, device="cuda")  # never read: the call is refused first
    T = np.eye(4)
    for w, h, pitch in ((32768, 32768, 65536), (1 << 29, 2, 1 << 30), (32768, 32768, 1 << 32)):
        with pytest.raises(native.YasError) as e:
            native.call("yas_map_fuse_u16", m.h, ctypes.c_void_p(buf.data_ptr()), pitch, w, h, 1000.0, rf._ptr(T))
        assert e.value.code == 1 and "4 GiB" in str(e.value)
    assert m.stats().num_allocated == 0
