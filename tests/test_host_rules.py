"""Rules that the host and the kernels share, replayed on the CPU."""
import ctypes as C

import pytest

from parcompfin_amd import _native as N


def index32(items, block, ipt):
    blocks = C.c_int32()
    yes = N.load().pcf_debug_index32(items, block, ipt, C.byref(blocks))
    return bool(yes), blocks.value


# ---------------------------------------------------------------- 32-bit loops over paths
@pytest.mark.parametrize("block", list(range(64, 1025, 64)))
def test_index32_never_wraps(block):
    """For every block size and items per thread that a call may ask for: a
    32-bit count is taken only if the item after any thread's last one is still
    a 32-bit number, and it is taken for every count far from the bound."""
    for ipt in range(1, 4097):
        for items in (1, 10**8, 1 << 30, 2**32 - 2**30 - 1, 2**32 - 2**30, 2**32 - 2**30 + 1, 0xF0000000 - 1, 0xF0000000,
                      0xF0000000 + 1, 2**32 - block, 2**32 - 1, 2**32, 2**34):
            yes, blocks = index32(items, block, ipt)
            assert 1 <= blocks <= 1 << 20
            fits = items - 1 + blocks * block < 2**32
            assert yes == fits, (items, block, ipt, blocks)
            if items <= 2**32 - 2**30:
                assert yes


@pytest.mark.parametrize("paths,block,ipt", [(13 * 10**9, 1024, 1), (16 * 10**9, 1024, 3), (16 * 10**9, 512, 1),
                                             (16 * 10**9, 512, 4), (12 * 10**9, 1024, 1), (4 * 10**9, 256, 1)])
def test_index32_loops_end(paths, block, ipt):
    """The loop of the first and the last thread in the launch's arithmetic."""
    groups = (paths + 3) // 4
    yes, blocks = index32(groups, block, ipt)
    stride = blocks * block
    mask = 2**32 - 1 if yes else 2**64 - 1
    for g in (0, min(stride, groups) - 1):
        turns = -(-(groups - g) // stride)
        for _ in range(turns):
            assert g < groups
            g = (g + stride) & mask
        assert g >= groups
