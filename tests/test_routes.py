"""CPU: the rules that choose a kernel's form by size, asked of the library without a device."""
import ctypes as C

import pytest


@pytest.fixture(scope="module")
def L():
    from booster_amd import build
    return C.CDLL(build.build())


def test_norm_blocks_hold_the_rows_they_can(L):
    """a thread holds two pieces of four floats: every row of up to 8192 floats that is a multiple of four fits its block, and no block has a wave more than that takes (or fewer than four); rows
    that are no multiple of four, which are read again for every sum, get all the threads unless there are blocks enough without"""
    for n in range(4, 8196, 4):
        t = L.bamd_op_norm_threads(n, 1)
        assert t == L.bamd_op_norm_threads(n, 4096)
        assert t % 64 == 0 and 256 <= t <= 1024
        assert 8 * t >= n or n > 8192, n
        assert t == 256 or 8 * (t - 64) < n, n
    assert {n: [L.bamd_op_norm_threads(n, rows) for rows in (1, 512, 513)] for n in (1, 1023, 1026, 2050, 4095, 9001)} == {
        1: [256] * 3, 1023: [256] * 3, 1026: [1024, 1024, 256], 2050: [1024, 1024, 320], 4095: [1024, 1024, 512], 9001: [1024] * 3}
