"""CPU: the rules that choose a kernel's form by size, asked of the library without a device."""
import ctypes as C

import pytest


@pytest.fixture(scope="module")
def L():
    from booster_amd import build
    return C.CDLL(build.build())


def test_norm_blocks_hold_the_rows_they_can(L):
    """a thread holds two pieces of four floats: every row of up to 8192 floats that is a multiple of four fits its block, and no block has a wave more than that takes (or fewer than four); rows
    that are no multiple of four, which lie in registers one by one, get all the threads unless there are blocks enough without"""
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


# type, K, rows, tokens, measured us of the other kernel (64-row blocks up to 16384 rows) and of the few-token kernel
@pytest.mark.parametrize("t,k,rows,T,wide,few", [
    (Q4_K, 4096, 4096, 37, 24.7, 11.8), (Q4_K, 4096, 8192, 32, 25.0, 19.6), (Q4_K, 4096, 8192, 48, 25.4, 23.0), (Q4_K, 4096, 8192, 64, 26.0, 26.2), (Q4_K, 3840, 6144, 36, 23.5, 20.0), (Q4_K, 4096, 6144, 36, 24.8, 21.0),
    (Q4_K, 2048, 4352, 40, 14.4, 13.2), (Q4_K, 1536, 5120, 32, 11.8, 10.5), (Q4_K, 1536, 6144, 40, 11.9, 11.6), (Q4_K, 1024, 8192, 48, 9.5, 10.4), (Q4_K, 8960, 6144, 36, 49.4, 38.7), (Q4_K, 4096, 12288, 32, 25.4, 28.3),
    (Q4_K, 2048, 24576, 16, 15.2, 31.2), (Q4_K, 14336, 24576, 32, 75.4, 155.3), (Q5_K, 3072, 6144, 64, 20.9, 21.5), (Q5_K, 2048, 6144, 48, 14.9, 15.0), (Q5_K, 13312, 6144, 48, 74.9, 65.6), (Q5_K, 14336, 4352, 32, 74.1, 53.1),
    (Q5_K, 4096, 14336, 48, 27.4, 46.6), (Q6_K, 4096, 8192, 64, 30.9, 33.2), (Q6_K, 2048, 4352, 32, 13.8, 17.1), (Q6_K, 1024, 8192, 64, 11.4, 14.4), (Q6_K, 8192, 6144, 40, 50.0, 53.7), (Q6_K, 14336, 14336, 40, 84.7, 175.7),
    (Q6_K, 4096, 12288, 32, 24.2, 42.2), (Q6_K, 4096, 6144, 16, 23.3, 25.7), (Q6_K, 4096, 4352, 37, 27.1, 29.8), (Q6_K, 4096, 4096, 40, 27.2, 16.5), (Q6_K, 5120, 20480, 32, 38.8, 83.2)])
def test_few_token_products_take_the_faster_kernel(L, t, k, rows, T, wide, few):
    assert (prefill(L, t, rows, k, T)[0] > 0) == (few < wide)


def test_few_token_kernel_covers_its_tokens(L):
    for t in (Q4_K, Q5_K, Q6_K):
        for T in range(1, 130):
            tiles = prefill(L, t, 1024, 4096, T)[0]
            assert tiles == (0 if T > 64 else 2 if T <= 32 else 3 if T <= 48 else 4)


BF16, F32 = 0, 1
T256x256, T128x256, T128x128, T64x128, T64x64, T64x64_DEEP = range(6)
ROWS, POLY, GROUP, GLU = 0, 2, 3, 5


def dense(L, act, n, k, rows, pre=-1, most=2):
    share = C.c_int(0)
    tile = L.bamd_op_dense_route(act, n, k, rows, pre, most, C.byref(share))
    return tile, share.value


# activation rows, matrix rows, K, the shares of the faster form: where a second 64 x 64 block per CU would make halves slower than the whole, and around it
@pytest.mark.parametrize("rows,n,k,want", [(131, 4096, 14336, (T128x128, 2)), (131, 3072, 8192, (T128x128, 2)), (300, 2048, 8192, (T128x128, 2)), (192, 4096, 8192, (T128x128, 2)), (65, 6144, 8192, (T128x128, 2)),
                                           (300, 2048, 4096, (T64x64, 2)), (640, 1024, 4096, (T64x64, 2)), (131, 2048, 8192, (T64x64_DEEP, 2)), (412, 4096, 8192, (T128x128, 2)), (131, 8192, 2048, (T64x64, 1))])
def test_many_rows_are_halved_where_that_is_faster(L, rows, n, k, want):
    assert dense(L, BF16, n, k, rows) == want
    assert dense(L, BF16, n, k, rows, most=1)[1] == 1


def test_few_rows_are_halved_where_that_is_faster(L):
    share = lambda act, n, k, pre, rows=1: dense(L, act, n, k, rows, pre)[1]
    for pre in (POLY, GROUP, GLU):
        # measured, 2048 to 1040 outputs: slower in halves up to K = 4096, faster from 4128; 1024 and 512 outputs: never slower
        assert [share(BF16, n, k, pre) for n in (2048, 1536, 1040) for k in (2048, 4096, 4128, 14336)] == [1, 1, 2, 2] * 3
        assert [share(BF16, n, k, pre) for n in (1024, 512) for k in (2048, 4096, 5632, 14336)] == [2] * 8
        assert [share(F32, 2048, k, pre) for k in (2016, 2048, 14336)] == [1, 2, 2]
    for act in (BF16, F32):
        assert [share(act, n, k, ROWS, rows) for rows in (1, 64) for n, k in ((2048, 2048), (2049, 2048), (2048, 2016))] == [2, 1, 1] * 2
    assert [share(BF16, 512, 4096, pre) for pre in (1, 4, 6)] == [1, 1, 1]           # prologues that write state


# type, rank, heads, rows, positions, measured us of a step of eight layers with latent attention in three launches and in one (where both are level, either is right)
@pytest.mark.parametrize("act,rank,heads,rows,positions,three,one", [
    (BF16, 32, 8, 1, 2000, 267, 261), (BF16, 32, 8, 1, 4000, 264, 273), (BF16, 64, 8, 1, 1500, 265, 261), (BF16, 64, 8, 1, 3000, 266, 280), (BF16, 64, 16, 1, 1000, 378, 366), (BF16, 64, 16, 1, 2000, 381, 384),
    (BF16, 128, 8, 1, 1000, 277, 271), (BF16, 128, 8, 1, 1500, 279, 284), (BF16, 128, 16, 6, 1000, 490, 474), (BF16, 128, 16, 6, 2000, 494, 502), (BF16, 256, 16, 1, 520, 392, 384), (BF16, 256, 16, 1, 800, 432, 438),
    (BF16, 512, 32, 1, 155, 830, 809), (BF16, 512, 32, 1, 800, 827, 884), (BF16, 512, 32, 16, 216, 1280, 1253), (BF16, 512, 32, 16, 500, 1289, 1317), (BF16, 256, 16, 48, 100, 1200, 1223), (BF16, 64, 16, 16, 1000, 595, 550),
    (F32, 32, 8, 1, 1700, 272, 268), (F32, 32, 8, 1, 3000, 276, 284), (F32, 64, 8, 1, 1000, 274, 265), (F32, 64, 8, 1, 1700, 277, 281), (F32, 128, 8, 1, 500, 290, 267), (F32, 128, 8, 1, 1700, 287, 316),
    (F32, 256, 16, 1, 380, 460, 452), (F32, 256, 16, 1, 800, 461, 501), (F32, 512, 32, 1, 155, 907, 849)])
def test_latent_steps_take_the_faster_launches(L, act, rank, heads, rows, positions, three, one):
    assert L.bamd_op_latent_route(act, 128, rank, rows, heads, positions) == (one < three)


def test_latent_steps_of_shorter_sequences_are_no_slower_choice(L):
    """the layers that take one launch are told apart by their number: what takes it at some length takes it at every shorter one"""
    for act in (BF16, F32):
        for rank in (32, 96, 256, 512, 544):
            got = [L.bamd_op_latent_route(act, 128, rank, 1, 16, n) for n in range(1, 5000)]
            assert got == sorted(got, reverse=True) and got[0] == (rank <= 512)
