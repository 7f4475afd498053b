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


Q4_K, Q5_K, Q6_K = 12, 13, 14


def prefill(L, t, rows, k, T):
    """(token tiles of the few-token kernel or 0, dynamic LDS, the most the load-time probe asks for)"""
    v = [C.c_int(0) for _ in range(3)]
    assert L.bamd_op_prefill_route(t, rows, k, T, *map(C.byref, v)) == 0
    return tuple(x.value for x in v)


def test_the_launch_probe_covers_every_prompt_product(L):
    seen = set()
    for t in (Q4_K, Q5_K, Q6_K):
        for rows in (8, 4096, 6144, 14336, 28672):
            for T in (1, 32, 33, 48, 49, 64, 65, 512):
                tiles, lds, most = prefill(L, t, rows, 4096, T)
                assert lds <= most <= 160 * 1024
                seen.add((tiles, lds))
    assert {s[0] for s in seen} == {0, 2, 3, 4} and max(s[1] for s in seen) == 159328 == most
