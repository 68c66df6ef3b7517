"""The renderer's correctly rounded device operations (gvv_math.hpp) against the IEEE operations over
every binary32 bit pattern: reciprocal, square root, quotients by a binary64 reciprocal, conversion to
int32 and the depth key.  Not one may differ."""
import ctypes

import pytest
import torch

from gvv_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("first,count", [(0, 1), (0x0D7FFFF0, 0x20), (0x71FFFFF0, 0x20), (0, 1 << 31), (1 << 31, 1 << 31)])
def test_rounding(device, first, count):
    bad = torch.zeros(5, dtype=torch.int64, device=device)
    _lib.check(_lib.load().gvv_check_rounding(first, count, ctypes.c_void_p(bad.data_ptr()),
                                              ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)), "gvv_check_rounding")
    assert bad.cpu().tolist() == [0] * 5
