"""The radix sort's workspace size, on the host: a workspace sized for n pairs
serves every smaller number of them."""
import ctypes

import numpy as np
import pytest

from wtet_amd import _core

BIG_FROM = 192 * 4096  # tiles of 1,024 pairs below, of 4,096 from here


@pytest.mark.parametrize("bits", [32, 64])
def test_workspace_grows_with_the_number_of_pairs(bits):
    # wtet::radix_temp_bytes_u32 / _u64 (uint32_t n, int end_bit)
    size = getattr(_core.lib(), "_ZN4wtet20radix_temp_bytes_u%dEji" % bits)
    size.argtypes, size.restype = [ctypes.c_uint32, ctypes.c_int], ctypes.c_size_t
    n = np.unique(np.concatenate([
        np.arange(0, 20000), BIG_FROM + np.arange(-6000, 6000), 4 * BIG_FROM + np.arange(-9000, 9000),
        np.geomspace(20000, 2 ** 31, 4000).astype(np.int64)]))
    bytes_ = np.array([size(int(k), bits) for k in n], np.uint64)
    down = np.nonzero(bytes_[1:] < bytes_[:-1])[0]
    assert len(down) == 0, [(int(n[i]), int(bytes_[i]), int(n[i + 1]), int(bytes_[i + 1])) for i in down[:3]]
