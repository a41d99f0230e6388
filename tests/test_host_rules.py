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


# ---------------------------------------------------------------- results of a launch that has ended
def collect(words, njobs, nres):
    a = (C.c_uint64 * len(words))(*words)
    ms = C.c_double(-1.0)
    return N.load().pcf_debug_wait_results(a, njobs, nres, C.byref(ms)), ms.value


UNWRITTEN = 2**64 - 1


@pytest.mark.parametrize("njobs", [1, 3])
@pytest.mark.parametrize("nres", [1, 4, 8])
def test_results_of_an_ended_launch(njobs, nres):
    words = []
    for j in range(njobs):
        words += [17 + i if i < nres else UNWRITTEN for i in range(8)]
        words += [1000 if j == 0 else UNWRITTEN, 3000 + j] + [UNWRITTEN] * 6
    status, ms = collect(words, njobs, nres)
    assert status == N.PCF_OK and ms == (3000 + njobs - 1 - 1000) / 1e5
    # a result may be the marker's own NaN where the job says that it ended
    odd = list(words)
    odd[0] = UNWRITTEN
    assert collect(odd, njobs, nres)[0] == N.PCF_OK
    # a job that never wrote is an error, whichever it is, and so is a missing start
    for j in range(njobs):
        lost = list(words)
        lost[16 * j:16 * j + 8] = [UNWRITTEN] * 8
        lost[16 * j + 9] = UNWRITTEN
        assert collect(lost, njobs, nres)[0] != N.PCF_OK
    lost = list(words)
    lost[8] = UNWRITTEN
    assert collect(lost, njobs, nres)[0] != N.PCF_OK
