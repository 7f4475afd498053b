"""GPU: the configured layer stacks (Tupitar, Mafurax) against oracle/stack_oracle.py — every mechanism alone, whole models in both compute types, and what must not matter:
portions, batches, pages and sequences."""
import ctypes as C
import json
import os
import subprocess
import sys

import numpy as np
import pytest

from conftest import ROOT
from oracle import stack_oracle as so
import stack_cases
from stack_cases import CONFIGS, ROWS, SEEDS, attend, config, latent, mafurax, mamba, parallel, tokens

pytestmark = pytest.mark.gpu
TOL = {"float32": 3e-5, "bfloat16": 0.03}                 # of the reference's root mean square
DTYPES = ["float32", "bfloat16"]


def rel(a, b):
    a, b = np.asarray(a, np.float64), np.asarray(b, np.float64)
    return float(np.sqrt(np.mean((a - b) ** 2) / np.mean(b ** 2)))


def near(a, b, dtype, f=1.0):
    """every row (last axis) within the tolerance of the compute type"""
    a, b = np.asarray(a, np.float64), np.asarray(b, np.float64)
    assert a.shape == b.shape
    e = np.sqrt(((a - b) ** 2).mean(-1) / (b ** 2).mean(-1))
    assert np.isfinite(a).all() and e.max() < f * TOL[dtype], "worst row %s: %.3g" % (np.unravel_index(e.argmax(), e.shape), e.max())


def bamd_lib():
    import booster_amd
    return booster_amd.lib()


# ---- mechanisms alone --------------------------------------------------------------------------------------------------------------------------------------
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("n,k,rows", [(1, 1, 1), (17, 31, 3), (130, 33, 64), (300, 75, 16), (48, 600, 17), (513, 96, 33), (260, 288, 65), (1100, 320, 500), (2050, 160, 1500)])
def test_dense(bamd, dtype, n, k, rows):
    r = np.random.default_rng(n + k)
    w = so.f32_to_bf16(r.standard_normal((n, k)))
    x = so.round_bf16(r.standard_normal((rows, k)))
    want = x.astype(np.float64) @ so.bf16_to_f32(w).T.astype(np.float64)
    scale = np.sqrt(k)
    for impl in (0, 1, 2, 3):
        if impl == 1 and rows > 64:
            continue
        tol = 2e-6 if impl < 2 or dtype == "float32" else 0.02
        assert np.abs(bamd.op_dense(w, x, dtype, impl) - want).max() < tol * scale * 4, impl
    if dtype == "float32":                               # operands keep their 32 bits
        x = r.standard_normal((rows, k)).astype(np.float32)
        want = x.astype(np.float64) @ so.bf16_to_f32(w).T.astype(np.float64)
        for impl in (0, 1):
            if impl == 0 or rows <= 64:
                assert np.abs(bamd.op_dense(w, x, dtype, impl) - want).max() < 8e-6 * scale


TILES = {("bfloat16", 8170, 2045): 0, ("bfloat16", 8170, 1000): 1, ("bfloat16", 4090, 1000): 2, ("bfloat16", 4090, 1100): 3, ("bfloat16", 8190, 131): 4, ("bfloat16", 2047, 131): 5, ("float32", 2047, 131): 4}


# one size per tile of the many-row product (256 x 256, 128 x 256, 128 x 128, 64 x 128, 64 x 64 with four and with eight stages; 32-bit: 64 x 64), ragged in every dimension, fewer and more column blocks than stages
@pytest.mark.parametrize("dtype,n,rows", [("bfloat16", 8170, 2045), ("bfloat16", 8170, 1000), ("bfloat16", 4090, 1000), ("bfloat16", 4090, 1100), ("bfloat16", 8190, 131), ("bfloat16", 2047, 131), ("float32", 2047, 131)])
@pytest.mark.parametrize("k", [1, 70, 300])
def test_dense_tiles(bamd, dtype, n, rows, k):
    assert bamd.op_dense_route(n, k, rows, dtype, most=1) == (TILES[dtype, n, rows], 1)
    r = np.random.default_rng(n + k + rows)
    w = so.f32_to_bf16(r.standard_normal((n, k)).astype(np.float32))
    x = r.standard_normal((rows, k)).astype(np.float32)
    x = x if dtype == "float32" else so.round_bf16(x)
    want = x.astype(np.float64) @ so.bf16_to_f32(w).T.astype(np.float64)
    scale = np.sqrt(np.abs(x).astype(np.float64) ** 2 @ np.abs(so.bf16_to_f32(w)).T.astype(np.float64) ** 2) + 1e-30      # of a sum of k products with random signs
    for impl, tol in ((0, 8e-6), (2, 2.0 ** -8), (3, 2.0 ** -8)):                    # k <= 300 roundings of 2^-24 | the result rounded to bfloat16 (2^-9 of it)
        e = np.abs(bamd.op_dense(w, x, dtype, impl) - want)
        assert (e <= tol * (scale if impl == 0 else np.abs(want) + 0.01 * scale)).all(), impl


# 32-bit: one size per tile (128 x 256, 128 x 128, 64 x 128, 64 x 64), ragged, and halves of three of them.  Bound: a rounding per column block and share, and what a column block's three matrix
# instructions cut off (2^-23 each of sums that grow to it)
@pytest.mark.parametrize("n,rows,k,route", [(8180, 1000, 1, (1, 1)), (8180, 1000, 300, (1, 1)), (8170, 500, 70, (2, 1)), (12600, 250, 300, (2, 1)), (8170, 250, 70, (3, 1)), (2040, 1000, 300, (3, 1)), (2040, 131, 1, (4, 1)),
                                            (2040, 131, 230, (4, 1)), (4090, 500, 2100, (2, 2)), (2040, 500, 2100, (3, 2)), (500, 131, 2100, (4, 2))])
def test_dense_split(bamd, n, rows, k, route):
    assert bamd.op_dense_route(n, k, rows, "float32") == route
    r = np.random.default_rng(n + k + rows)
    w = so.f32_to_bf16(r.standard_normal((n, k), np.float32) + np.float32(0.5))
    x = r.standard_normal((rows, k), np.float32) * np.exp(2 * r.standard_normal((rows, 1), np.float32)) + np.float32(0.5)
    wf = so.bf16_to_f32(w).astype(np.float64)
    want, size = x.astype(np.float64) @ wf.T, np.abs(x).astype(np.float64) @ np.abs(wf).T
    for impl in (4,) if route[1] == 2 else (0, 2, 3):
        assert (np.abs(bamd.op_dense(w, x, "float32", impl) - want) <= (k / 32 + 8) * 2.0 ** -24 * size).all(), impl


# 32-bit numbers at the ends of their range: the parts a product is made of stay what they are together
def test_dense_split_values(bamd):
    k, r = 96, np.random.default_rng(5)
    w = so.f32_to_bf16(np.abs(r.standard_normal((40, k), np.float32)) * np.float32(1e-3) + np.float32(1e-4))
    x = np.abs(r.standard_normal((70, k), np.float32))
    nan_low = np.array([0x7f800001], np.uint32).view(np.float32)[0]
    for row, v in ((1, np.inf), (2, -np.inf), (3, nan_low), (4, np.nan), (5, np.finfo(np.float32).max), (6, -np.finfo(np.float32).max), (7, np.float32(1e-30)), (8, 0.0)):
        x[row, 10] = v
    x[9] = np.finfo(np.float32).max                                    # sums beyond the range
    with np.errstate(over="ignore", invalid="ignore"):
        want = (x.astype(np.float64) @ so.bf16_to_f32(w).T.astype(np.float64)).astype(np.float32)
    got = bamd.op_dense(w, x, "float32", 0)
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(np.isposinf(got), np.isposinf(want)) and np.array_equal(np.isneginf(got), np.isneginf(want))
    ok = np.isfinite(want)
    assert not np.isnan(got[1]).any() and np.isnan(got[3:5]).all() and np.allclose(got[ok], want[ok], rtol=2e-6, atol=0)


# and weights that are not finite: what 32-bit products give, whatever parts an activation has (numbers of eight bits, powers of two, zeros and infinities among them)
@pytest.mark.parametrize("rows,impl", [(70, 0), (70, 2), (70, 6), (5, 1), (17, 1), (64, 7)])
def test_dense_weights_that_are_not_finite(bamd, rows, impl):
    k, r = 160, np.random.default_rng(rows)
    x = r.standard_normal((rows, k), np.float32) + np.float32(5)
    x[:, 10:14] = [1, -2, 0.375, 1 + 2.0 ** -16]
    x[0, 20:24], x[1, 20], x[2, 21], x[3, 22] = [0, -0.0, 1e-28, -1e-28], np.inf, -np.inf, np.nan
    x[4] = so.round_bf16(x[4])
    w = r.standard_normal((60, k)).astype(np.float32)
    for row, col, v in ((0, 10, np.inf), (1, 11, np.inf), (2, 12, -np.inf), (3, 13, np.nan), (4, 10, np.inf), (4, 12, np.inf), (5, 10, np.inf), (5, 11, np.inf), (6, 20, np.inf), (7, 21, -np.inf), (8, 22, np.inf), (9, 23, np.inf), (10, 50, -np.inf)):
        w[row, col] = v
    w = so.f32_to_bf16(w)
    with np.errstate(invalid="ignore"):
        want = sum(x[:, i:i + 1].astype(np.float64) * so.bf16_to_f32(w[:, i]).astype(np.float64) for i in range(k)).astype(np.float32)      # (one by one: a matrix product may leave zeros out)
    got = bamd.op_dense(w, x, "float32", impl)
    assert np.isinf(want).sum() > 8 * rows and np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(np.isposinf(got), np.isposinf(want)) and np.array_equal(np.isneginf(got), np.isneginf(want))
    ok = np.isfinite(want)
    assert np.allclose(got[ok], want[ok], rtol=0, atol=160 * 2.0 ** -24 * 40)


# the widths between: 256 x 224, 256 x 192 and 256 x 160, ragged in every dimension; the gated unit on 256 x 192
@pytest.mark.parametrize("n,rows,tile", [(14330, 1000, 6), (11000, 900, 7), (12600, 1485, 8)])
@pytest.mark.parametrize("k", [1, 70, 300])
def test_dense_tiles_between(bamd, n, rows, tile, k):
    assert bamd.op_dense_route(n, k, rows, "bfloat16", most=1) == (tile, 1)
    r = np.random.default_rng(n + k + rows)
    w = so.f32_to_bf16(r.standard_normal((n, k), np.float32))
    x = so.round_bf16(r.standard_normal((rows, k), np.float32))
    wf = so.bf16_to_f32(w)
    want, scale = x.astype(np.float64) @ wf.T.astype(np.float64), np.sqrt((x * x) @ (wf * wf).T) + 1e-30
    for impl, tol in ((0, 8e-6), (6, 8e-6), (2, 2.0 ** -8), (3, 2.0 ** -8)):         # as test_dense_tiles
        e = np.abs(bamd.op_dense(w, x, "bfloat16", impl) - want)
        assert (e <= tol * (scale if impl in (0, 6) else np.abs(want) + 0.01 * scale)).all(), impl


@pytest.mark.parametrize("k", [1, 300])
def test_dense_gated_tile_between(bamd, k):
    gated(bamd, "bfloat16", 5490, 900, k)


# whole rounds of 256 x 256 and the rest apart: the same bits as the parts by themselves (a sum's order does not hang on the tile)
@pytest.mark.parametrize("n,rows,k,cut", [(16890, 2045, 1500, 16384), (16890, 1030, 1500, 0)])
def test_dense_whole_rounds(bamd, n, rows, k, cut):
    r = np.random.default_rng(n + k + rows)
    w = so.f32_to_bf16(r.standard_normal((n, k), np.float32))
    x = so.round_bf16(r.standard_normal((rows, k), np.float32))
    assert bamd.lib().bamd_op_dense_cut(n, k, rows, 0) == cut and not bamd.lib().bamd_op_dense_cut(cut or n, k, rows, 0)
    parts = [w[:cut], w[cut:]] if cut else [w[:8192], w[8192:]]
    want = np.concatenate([bamd.op_dense(p, x, "bfloat16", 0) for p in parts], 1)
    for impl in (0, 6):
        assert np.array_equal(bamd.op_dense(w, x, "bfloat16", impl).view(np.uint32), want.view(np.uint32)), impl


def test_dense_gated_whole_rounds(bamd):
    F, rows, k, cut = 14330, 2045, 2050, 12288                          # (rows of 1500 columns are not worth a second launch)
    r = np.random.default_rng(F + k + rows)
    gate, up = (so.f32_to_bf16(r.standard_normal((F, k), np.float32) * np.float32(0.03)) for _ in range(2))
    x = so.round_bf16(r.standard_normal((rows, k), np.float32))
    assert bamd.lib().bamd_op_dense_cut(2 * ((F + 31) // 32 * 32), k, rows, 1) == 2 * cut
    want = np.concatenate([bamd.op_dense_glu(gate[i:j], up[i:j], x, 7.0, "bfloat16") for i, j in ((0, cut), (cut, F))], 1)
    for blocks in (False, True):
        assert np.array_equal(bamd.op_dense_glu(gate, up, x, 7.0, "bfloat16", blocks).view(np.uint32), want.view(np.uint32)), blocks


# operand rows by blocks of 32 columns, as the passes have them, against the same rows by rows: every tile of many rows and every group of few, ragged
@pytest.mark.parametrize("n,rows,impl", [(8170, 2045, 0), (8170, 1000, 0), (4090, 1000, 0), (4090, 1100, 0), (8190, 131, 0), (2047, 131, 0), (2030, 1, 1), (2030, 16, 1), (4620, 3, 1), (11000, 15, 1), (4100, 17, 1), (4620, 32, 1), (4620, 33, 1),
                                         (12400, 33, 1), (520, 64, 1)])
@pytest.mark.parametrize("k", [1, 300, 2050])
def test_dense_rows_by_blocks(bamd, n, rows, impl, k):
    r = np.random.default_rng(n + k + rows)
    w = so.f32_to_bf16(r.standard_normal((n, k), np.float32))
    x = so.round_bf16(r.standard_normal((rows, k), np.float32))
    assert np.array_equal(bamd.op_dense(w, x, "bfloat16", impl + 6).view(np.uint32), bamd.op_dense(w, x, "bfloat16", impl).view(np.uint32))


# and in 32-bit, three planes to a block: 128 x 256, 128 x 128, 64 x 128 and 64 x 64, and groups of 16, 32 and 64 rows
@pytest.mark.parametrize("n,rows,impl", [(8180, 1000, 0), (8170, 500, 0), (8170, 250, 0), (2040, 131, 0), (2030, 1, 1), (4620, 2, 1), (2030, 16, 1), (4100, 17, 1), (4100, 32, 1), (4620, 33, 1), (520, 64, 1)])
@pytest.mark.parametrize("k", [1, 300, 2050])
def test_dense_rows_by_blocks_in_32_bit(bamd, n, rows, impl, k):
    if impl == 0:
        assert bamd.op_dense_route(n, k, rows, "float32", most=1)[0] == {1000: 1, 500: 2, 250: 3, 131: 4}[rows]
    r = np.random.default_rng(n + k + rows)
    w = so.f32_to_bf16(r.standard_normal((n, k), np.float32))
    x = r.standard_normal((rows, k), np.float32)
    assert np.array_equal(bamd.op_dense(w, x, "float32", impl + 6).view(np.uint32), bamd.op_dense(w, x, "float32", impl).view(np.uint32))


# the gated unit from operands by blocks to results by blocks, against rows: few rows, the tiles of many, and 32-bit results of three planes
@pytest.mark.parametrize("dtype,F,rows", [("bfloat16", 1001, 3), ("bfloat16", 1001, 17), ("bfloat16", 8210, 32), ("bfloat16", 7000, 33), ("bfloat16", 4085, 1000), ("bfloat16", 5490, 900), ("bfloat16", 1001, 131),
                                          ("float32", 4085, 1000), ("float32", 4085, 500), ("float32", 1001, 131)])
@pytest.mark.parametrize("k", [1, 300])
def test_dense_gated_by_blocks(bamd, dtype, F, rows, k):
    r = np.random.default_rng(F + k + rows)
    gate, up = (so.f32_to_bf16(r.standard_normal((F, k), np.float32)) for _ in range(2))
    x = r.standard_normal((rows, k), np.float32)
    assert np.array_equal(bamd.op_dense_glu(gate, up, x, 7.0, dtype, True).view(np.uint32), bamd.op_dense_glu(gate, up, x, 7.0, dtype).view(np.uint32))


# the same tiles where they write the clamped gated unit of their gate and up tiles in turn: widths that end inside a pair of tiles, on its edge and inside a group of four
@pytest.mark.parametrize("dtype,F,rows,tile", [("bfloat16", 4085, 2045, 0), ("bfloat16", 4085, 1000, 1), ("bfloat16", 2032, 1000, 2), ("bfloat16", 2046, 1100, 3), ("bfloat16", 4090, 131, 4), ("bfloat16", 1001, 131, 5), ("bfloat16", 35, 70, 5),
                                                ("float32", 1001, 131, 4)])
@pytest.mark.parametrize("k", [1, 70, 300])
def test_dense_gated_tiles(bamd, dtype, F, rows, tile, k):
    assert bamd.op_dense_route(2 * ((F + 31) // 32 * 32), k, rows, dtype, most=1) == (tile, 1)
    gated(bamd, dtype, F, rows, k)


# a unit alone, a remainder of a round of units, rows at the edges of their groups, and beyond 32 the tiles of prompts (7000: enough row tiles; 200: not enough, in the engine the unit has its own launch)
@pytest.mark.parametrize("F,rows", [(1, 2), (16, 16), (40, 17), (8210, 5), (8210, 32), (7000, 33), (200, 64)])
@pytest.mark.parametrize("k", [1, 230, 2050])
def test_dense_gated_few_rows(bamd, F, rows, k):
    gated(bamd, "bfloat16", F, rows, k)


def gated(bamd, dtype, F, rows, k):
    r = np.random.default_rng(F + k + rows)
    gate, up = (so.f32_to_bf16(r.standard_normal((F, k)).astype(np.float32)) for _ in range(2))
    x, limit = r.standard_normal((rows, k)).astype(np.float32), 7.0
    x = x if dtype == "float32" else so.round_bf16(x)
    both = [x.astype(np.float64) @ so.bf16_to_f32(w).T.astype(np.float64) for w in (gate, up)]
    scale = [np.sqrt(np.abs(x).astype(np.float64) ** 2 @ np.abs(so.bf16_to_f32(w)).T.astype(np.float64) ** 2) for w in (gate, up)]
    g, u = np.minimum(both[0], limit), np.clip(both[1], -limit, limit)
    want = g * so.sigmoid(1.702 * g) * (u + 1)
    # errors of the sums (test_dense_tiles) through slopes of at most 1.13 |u + 1| and |g sigmoid| <= limit, and the result's own rounding
    e = np.abs(bamd.op_dense_glu(gate, up, x, limit, dtype) - want)
    assert (e <= 8e-6 * (1.13 * (limit + 1) * scale[0] + limit * scale[1]) + (1e-5 if dtype == "float32" else 2.0 ** -8) * np.abs(want) + 1e-30).all()


# one, two and three row tiles per step with a remainder, every group of rows and its edges, fewer column blocks than waves and more than a ring holds
@pytest.mark.parametrize("n,rows", [(2030, 1), (2030, 16), (4620, 2), (11000, 15), (4100, 17), (4620, 32), (4620, 33), (12400, 33), (520, 64)])
@pytest.mark.parametrize("k", [1, 230, 2050])
def test_dense_few_rows(bamd, n, rows, k):
    r = np.random.default_rng(n + k + rows)
    w = so.f32_to_bf16(r.standard_normal((n, k)).astype(np.float32))
    x = so.round_bf16(r.standard_normal((rows, k)).astype(np.float32))
    want = x.astype(np.float64) @ so.bf16_to_f32(w).T.astype(np.float64)
    scale = np.sqrt(np.abs(x).astype(np.float64) ** 2 @ np.abs(so.bf16_to_f32(w)).T.astype(np.float64) ** 2) + 1e-30      # of a sum of k products with random signs
    assert (np.abs(bamd.op_dense(w, x, "bfloat16", 1) - want) <= 1e-5 * scale).all()                 # sqrt(k) <= 46 roundings of 2^-24 in a row, three times over


# rows in LDS: the first and last sizes (257 row tiles, more than two a CU, the shortest and the longest K), shares of K that differ by a column block, tiles that meet in two goes (K = 4600), a CU with a
# tile more than others, rows by rows and by blocks; sizes beside them for which dense_few_kernel stays
@pytest.mark.parametrize("n,rows,k", [(4097, 5, 3553), (4097, 16, 4096), (4640, 2, 3300), (4640, 16, 4100), (8192, 4, 4090), (8193, 1, 3041), (8193, 3, 3040), (8210, 16, 4600), (8210, 16, 4640), (12290, 9, 3300)])
def test_dense_rows_in_lds(bamd, n, rows, k):
    r = np.random.default_rng(n + k + rows)
    w = so.f32_to_bf16(r.standard_normal((n, k)).astype(np.float32))
    x = so.round_bf16(r.standard_normal((rows, k)).astype(np.float32))
    wf = so.bf16_to_f32(w)
    want = x.astype(np.float64) @ wf.T.astype(np.float64)
    scale = np.sqrt((x ** 2) @ (wf.T ** 2))
    for impl in (1, 7):
        assert (np.abs(bamd.op_dense(w, x, "bfloat16", impl) - want) <= 1.5e-5 * scale).all(), impl      # sqrt(k) <= 68 roundings of 2^-24 in a row, three times over (12e-6), and the scale's own


@pytest.mark.parametrize("F,rows,k", [(2060, 5, 3553), (2060, 16, 4096), (4096, 4, 4090), (4112, 2, 3041), (4112, 16, 4600), (4128, 16, 4640), (6200, 3, 3300)])
def test_dense_gated_rows_in_lds(bamd, F, rows, k):
    gated(bamd, "bfloat16", F, rows, k)


# K in two shares (few row tiles, many columns: an odd number of column blocks among them), and sizes just below that
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("n,k,rows", [(500, 2100, 131), (77, 2049, 300), (500, 1000, 70), (500, 2100, 1), (2048, 2080, 6), (2049, 2080, 6), (77, 2049, 20), (500, 2100, 45), (500, 2000, 6)])
def test_dense_halves(bamd, dtype, n, k, rows):
    halved = 2 if (n, k, rows) not in ((500, 1000, 70), (2049, 2080, 6), (500, 2000, 6)) else 1
    assert bamd.op_dense_route(n, k, rows, dtype, pre=-1 if rows > 64 else 0)[1] == (halved if k != 1000 or dtype == "bfloat16" else 2)
    r = np.random.default_rng(n + k + rows)
    w = so.f32_to_bf16(r.standard_normal((n, k)).astype(np.float32))
    x = so.round_bf16(r.standard_normal((rows, k)).astype(np.float32))
    want = x.astype(np.float64) @ so.bf16_to_f32(w).T.astype(np.float64)
    scale = np.sqrt(np.abs(x).astype(np.float64) ** 2 @ np.abs(so.bf16_to_f32(w)).T.astype(np.float64) ** 2)
    for impl in (4,) if rows > 64 else (4, 5):
        assert (np.abs(bamd.op_dense(w, x, dtype, impl) - want) <= 1e-5 * scale).all(), impl


# and of the larger tiles, whose halves need larger matrices
@pytest.mark.parametrize("n,k,rows,tile", [(4247, 8200, 65, 2), (8247, 4130, 131, 3), (2045, 4090, 300, 4), (8247, 8200, 513, 0)])
def test_dense_halves_of_large_tiles(bamd, n, k, rows, tile):
    assert bamd.op_dense_route(n, k, rows, "bfloat16") == (tile, 2)
    r = np.random.default_rng(n + k + rows)
    w = so.f32_to_bf16(r.standard_normal((n, k), np.float32))
    x = so.round_bf16(r.standard_normal((rows, k), np.float32))
    wf = so.bf16_to_f32(w)
    want = x.astype(np.float64) @ wf.T.astype(np.float64)
    scale = np.sqrt((x * x) @ (wf * wf).T)
    assert (np.abs(bamd.op_dense(w, x, "bfloat16", 4) - want) <= 1e-5 * scale).all()               # as above: sqrt(k) <= 91 roundings of 2^-24 in a row, twice over


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("E,rows,pos0,with_y,with_mu", [(75, 5, 0, True, True), (75, 5, 9, True, True), (33, 1, 4, True, True), (1, 3, 0, True, True), (300, 4, 0, False, True), (96, 3, 2, True, False), (2000, 2, 7, True, True)])
def test_residual_norm_and_token_shift(bamd, dtype, E, rows, pos0, with_y, with_mu):
    r = np.random.default_rng(E + rows)
    x, y, prev = r.standard_normal((rows, E)), r.standard_normal((rows, E)) * 3, r.standard_normal(E)
    mu = r.uniform(0, 1, E) if with_mu else None
    xo, h, last = bamd.op_residual_rows(x, y if with_y else None, 0.7, 1e-3, mu, prev, pos0, dtype)
    ref = np.stack([xi + so.scalar_norm(yi, 0.7, 1e-3) if with_y else xi for xi, yi in zip(x, y)])
    near(xo, ref, "float32")
    if with_mu:
        front = np.concatenate([(prev if pos0 else np.zeros(E))[None], ref[:-1]])
        near(h, np.stack([so.token_shift(a, b, mu) for a, b in zip(ref, front)]), dtype)
        near(last, ref[-1], "float32")
    else:
        near(h, ref, dtype)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("F", [1, 40, 333, 3000])
def test_poly_norm(bamd, dtype, F):
    r = np.random.default_rng(F)
    z, coef = r.standard_normal((6, F)) * np.array([1e-3, 0.1, 1, 3, 10, 50])[:, None], [0.8, -0.5, 0.6, 0.25]
    near(bamd.op_poly_norm(z, coef, 1e-4, dtype), np.stack([so.poly_norm(v, *coef, 1e-4) for v in z]), dtype)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("n,groups", [(60, 1), (60, 5), (120, 3), (256, 64), (20, 20), (4096, 8)])
def test_group_norm(bamd, dtype, n, groups):
    r = np.random.default_rng(n + groups)
    y, w = r.standard_normal((3, n)) * np.repeat(r.uniform(0.1, 10, groups), n // groups), 1 + r.standard_normal(n)
    near(bamd.op_group_norm(y, w, groups, 1e-5, dtype), np.stack([so.grouped_norm(v, groups, w, 1e-5) for v in y]), dtype)


def plain_ssm(rows, H, P, N, G, conv, cb, dtb, A, D, hist, S):
    inner, out = H * P, []
    for row in rows:
        z, xbc, dt = np.split(row, [inner, 2 * inner + 2 * G * N])
        xbc, hist = so.causal_conv(conv, cb, hist, xbc)
        x, B, C_ = np.split(so.silu(xbc), [inner, inner + G * N])
        dt = so.softplus(dt + dtb)
        y = np.zeros(inner)
        for i in range(H):
            g = i // (H // G)
            S[i], y[i * P:(i + 1) * P] = so.ssd_step(S[i], dt[i], A[i], D[i], B[g * N:(g + 1) * N], C_[g * N:(g + 1) * N], x[i * P:(i + 1) * P])
        out.append(y * so.silu(z))
    return np.array(out), hist, S


@pytest.mark.parametrize("H,P,N,G,taps", [(1, 1, 1, 1, 1), (3, 20, 24, 1, 4), (4, 10, 12, 4, 2), (4, 16, 40, 2, 3), (2, 130, 33, 1, 7), (1, 64, 256, 1, 4), (2, 24, 128, 2, 5)])
def test_ssm(bamd, H, P, N, G, taps):
    """portions from one token up, first tokens (taps reach before the start), state and convolution inputs handed from portion to portion, fast and slow decays"""
    r = np.random.default_rng(H * P + N)
    inner, ch = H * P, H * P + 2 * G * N
    conv, cb, dtb, A, D = r.standard_normal((ch, taps)), r.standard_normal(ch) * 0.3, r.uniform(-6, 1, H), r.uniform(-4, 2, H), r.standard_normal(H)
    f = lambda a: np.asarray(a, np.float32)
    rows = f(r.standard_normal((70, inner + ch + H)))
    rows[::9, -H:] -= 30                                  # a step size of almost zero: the state stays as it is
    rows[5::11, -H:] += 25                                # and a large one: it is forgotten
    conv, cb, dtb, A, D = map(f, (conv, cb, dtb, A, D))
    hist, S = np.zeros((taps - 1, ch)), np.zeros((H, N, P))
    gh, gs, pos = f(hist), f(S) + 7, 0                    # what a fresh sequence finds in its place must not matter
    gh = gh + 7
    for n in (1, 1, 2, 15, 16, 17, 18):
        part = rows[pos:pos + n]
        want, hist, S = plain_ssm(part.astype(np.float64), H, P, N, G, conv, cb, dtb, A, D, hist, S)
        got, gh, gs = bamd.op_ssm(part, pos, H, P, N, G, conv, cb, dtb, A, D, gh, gs)
        assert rel(got, want) < 2e-5, pos
        assert rel(gs, S) < 2e-5 and (taps == 1 or rel(gh, hist) < 1e-6)
        pos += n


@pytest.mark.parametrize("H,P,N,G", [(2, 40, 128, 1), (130, 33, 24, 2), (256, 64, 12, 1), (257, 20, 3, 1), (1, 64, 256, 1), (128, 64, 256, 1), (256, 64, 256, 4)])
def test_ssm_tokens_of_four_taps(bamd, H, P, N, G):
    """one token after the other, from a fresh state on: blocks of 16, 32 and 64 columns, with one, two and three channels per thread"""
    r = np.random.default_rng(H + P + N)
    inner, ch = H * P, H * P + 2 * G * N
    f = lambda a: np.asarray(a, np.float32)
    conv, cb, dtb, A, D = map(f, (r.standard_normal((ch, 4)), r.standard_normal(ch) * 0.3, r.uniform(-6, 1, H), r.uniform(-4, 3, H), r.standard_normal(H)))
    rows = f(r.standard_normal((6, inner + ch + H)))
    hist, S = np.zeros((3, ch)), np.zeros((H, N, P))
    gh, gs = f(hist) + 7, f(S) + 7
    for pos in range(6):
        want, hist, S = plain_ssm(rows[pos:pos + 1].astype(np.float64), H, P, N, G, conv, cb, dtb, A, D, hist, S)
        got, gh, gs = bamd.op_ssm(rows[pos:pos + 1], pos, H, P, N, G, conv, cb, dtb, A, D, gh, gs)
        assert rel(got, want) < 2e-5 and rel(gs, S) < 2e-5 and np.array_equal(gh, f(hist)), pos


@pytest.mark.parametrize("H,P,N,G", [(2, 32, 64, 1), (1, 33, 65, 1), (3, 64, 128, 3), (1, 31, 129, 1), (2, 100, 200, 2), (1, 16, 256, 1)])
def test_ssm_chunks(bamd, H, P, N, G):
    """prompts through every number of state tiles, around the width of a block and the sixteen tokens of a chunk, with decays down to zero and up to one; portions continue one another"""
    r = np.random.default_rng(H * P + N)
    inner, ch = H * P, H * P + 2 * G * N
    f = lambda a: np.asarray(a, np.float32)
    conv, cb, dtb, A, D = map(f, (r.standard_normal((ch, 4)), r.standard_normal(ch) * 0.3, r.uniform(-6, 1, H), r.uniform(-4, 3, H), r.standard_normal(H)))
    rows = f(r.standard_normal((200, inner + ch + H)))
    rows[::9, -H:] -= 30
    rows[5::11, -H:] += 90                                # exp(-exp(A) dt) is zero
    hist, S = np.zeros((3, ch)), np.zeros((H, N, P))
    gh, gs, pos = f(hist), f(S) + 7, 0
    for n in (31, 32, 33, 2, 48, 54):
        part = rows[pos:pos + n]
        want, hist, S = plain_ssm(part.astype(np.float64), H, P, N, G, conv, cb, dtb, A, D, hist, S)
        got, gh, gs = bamd.op_ssm(part, pos, H, P, N, G, conv, cb, dtb, A, D, gh, gs)
        assert rel(got, want) < 2e-5 and rel(gs, S) < 2e-5, pos      # as test_ssm
        pos += n


# a token of a prompt that is not finite leaves the tokens in front of it as they are (in B, C, x and the step size, at several places of a chunk), and so does a state handed over that is not;
# "far": finite values whose product with a token further back overflows
@pytest.mark.parametrize("N,at", [(40, 20), (128, 30), (200, 17)])
@pytest.mark.parametrize("what,value", [("x", np.inf), ("x", np.nan), ("B", np.inf), ("C", np.nan), ("dt", np.inf), ("far", 1e20), ("state", np.inf)])
def test_ssm_tokens_that_are_not_finite(bamd, N, at, what, value):
    H, P, n = 2, 40, 70
    r = np.random.default_rng(N)
    inner, ch = H * P, H * P + 2 * N
    f = lambda a: np.asarray(a, np.float32)
    conv, cb, dtb, A, D = map(f, (r.uniform(0.5, 2, (ch, 1)), np.zeros(ch), r.uniform(-2, 1, H), r.uniform(-2, 1, H), r.standard_normal(H)))
    rows, S = f(r.standard_normal((n, inner + ch + H))), f(r.standard_normal((H, N, P)))
    x, B, C = inner + P + 33, 2 * inner + N // 2, 2 * inner + N + 1                  # a column of the second head, a state row of both
    if what == "state":
        S[1, N - 1, 5] = value
    elif what == "far":
        rows[at, 2 * inner + N + N // 2] = rows[at + 1, B] = value
    else:
        rows[at, {"x": x, "B": B, "C": C, "dt": -1}[what]] = value
    with np.errstate(all="ignore"):
        want, _, _ = plain_ssm(rows.astype(np.float64), H, P, N, 1, conv, cb, dtb, A, D, np.zeros((0, ch)), S.astype(np.float64))
    got, _, _ = bamd.op_ssm(rows, 1, H, P, N, 1, conv, cb, dtb, A, D, np.zeros((0, ch)), S)
    assert np.isfinite(want[:at] if what != "state" else want[:, :P]).all() and (what == "far" or not np.isfinite(want).all())
    for t in range(n):
        ok = np.isfinite(want[t])
        assert (np.isfinite(got[t]) == ok).all(), t
        assert not ok.any() or rel(got[t][ok], want[t][ok]) < 2e-5, t                # as test_ssm


@pytest.mark.parametrize("H,P,N,G", [(2, 40, 40, 1), (1, 31, 200, 1), (80, 10, 12, 2), (43, 33, 65, 1), (65, 40, 8, 1)])
@pytest.mark.parametrize("n", [63, 64, 65, 100, 257])
def test_ssm_prompts_in_parts(bamd, H, P, N, G, n):
    """fresh prompts whose tokens are taken in four parts, three, two and one, last chunks of one token and of sixteen; a portion behind them starts from their state"""
    r = np.random.default_rng(H * P + N + n)
    inner, ch = H * P, H * P + 2 * G * N
    f = lambda a: np.asarray(a, np.float32)
    conv, cb, dtb, A, D = map(f, (r.standard_normal((ch, 4)), r.standard_normal(ch) * 0.3, r.uniform(-6, 1, H), r.uniform(-4, 3, H), r.standard_normal(H)))
    rows = f(r.standard_normal((n + 70, inner + ch + H)))
    rows[::9, -H:] -= 30
    hist, S = np.zeros((3, ch)), np.zeros((H, N, P))
    gh, gs = f(hist), f(S) + 7
    for pos, end in ((0, n), (n, n + 70)):
        want, hist, S = plain_ssm(rows[pos:end].astype(np.float64), H, P, N, G, conv, cb, dtb, A, D, hist, S)
        got, gh, gs = bamd.op_ssm(rows[pos:end], pos, H, P, N, G, conv, cb, dtb, A, D, gh, gs)
        assert rel(got, want) < 2e-5 and rel(gs, S) < 2e-5, pos      # as test_ssm


@pytest.mark.parametrize("H,P,N,more", [(2, 40, 40, 66), (1, 31, 200, 130), (43, 33, 65, 86), (70, 20, 12, 140), (2, 64, 128, 128)])
@pytest.mark.parametrize("n", [64, 81, 300])
def test_ssm_parts_give_the_bits_of_one(bamd, H, P, N, more, n):
    """the same heads in a launch that takes its tokens in four, three or two parts, and among so many that it takes one: outputs and state bit for bit"""
    r = np.random.default_rng(H * P + N + n)
    f = lambda a: np.asarray(a, np.float32)
    chan = lambda H: H * P + 2 * N
    cx, cbc, bx, bbc = r.standard_normal((H, P, 4)), r.standard_normal((2 * N, 4)), r.standard_normal((H, P)) * 0.3, r.standard_normal(2 * N) * 0.3
    dtb, A, D = r.uniform(-6, 1, H), r.uniform(-4, 3, H), r.standard_normal(H)
    z, x, bc, dt = r.standard_normal((n, H, P)), r.standard_normal((n, H, P)), r.standard_normal((n, 2 * N)), r.standard_normal((n, H))
    dt[::9] -= 30
    def go(heads):
        k = np.arange(heads) % H
        rows = np.concatenate([z[:, k].reshape(n, -1), x[:, k].reshape(n, -1), bc, dt[:, k]], 1)
        got, _, S = bamd.op_ssm(f(rows), 0, heads, P, N, 1, f(np.concatenate([cx[k].reshape(-1, 4), cbc])), f(np.concatenate([bx[k].ravel(), bbc])), f(dtb[k]), f(A[k]), f(D[k]), np.zeros((3, chan(heads)), np.float32), np.zeros((heads, N, P), np.float32))
        return got.reshape(n, heads, P), S
    y, S = go(H)
    ym, Sm = go(more)
    k = np.arange(more) % H
    assert (np.ascontiguousarray(ym).view(np.uint32) == np.ascontiguousarray(y[:, k]).view(np.uint32)).all() and (Sm.view(np.uint32) == np.ascontiguousarray(S[k]).view(np.uint32)).all()


@pytest.mark.parametrize("N,at", [(40, 0), (128, 3), (200, 17), (40, 47), (128, 60), (40, 110)])
@pytest.mark.parametrize("what,value", [("x", np.inf), ("x", np.nan), ("B", np.inf), ("C", np.nan), ("dt", np.inf), ("far", 1e20)])
def test_ssm_tokens_that_are_not_finite_in_parts(bamd, N, at, what, value):
    """a token that the parts behind it meet on their way to a state, or that no part does"""
    H, P, n = 2, 40, 130
    r = np.random.default_rng(N + at)
    inner, ch = H * P, H * P + 2 * N
    f = lambda a: np.asarray(a, np.float32)
    conv, cb, dtb, A, D = map(f, (r.uniform(0.5, 2, (ch, 1)), np.zeros(ch), r.uniform(-2, 1, H), r.uniform(-2, 1, H), r.standard_normal(H)))
    rows = f(r.standard_normal((n, inner + ch + H)))
    x, B, C = inner + P + 33, 2 * inner + N // 2, 2 * inner + N + 1                  # a column of the second head, a state row of both
    if what == "far":
        rows[at, 2 * inner + N + N // 2] = rows[at + 1, B] = value
    else:
        rows[at, {"x": x, "B": B, "C": C, "dt": -1}[what]] = value
    with np.errstate(all="ignore"):
        want, _, S = plain_ssm(rows.astype(np.float64), H, P, N, 1, conv, cb, dtb, A, D, np.zeros((0, ch)), np.zeros((H, N, P)))
    got, _, gs = bamd.op_ssm(rows, 0, H, P, N, 1, conv, cb, dtb, A, D, np.zeros((0, ch)), np.zeros((H, N, P), np.float32))
    assert np.isfinite(want[:at]).all() and (what == "far" or not np.isfinite(want).all())
    assert np.array_equal(np.isfinite(gs), np.isfinite(S))
    for t in range(n):
        ok = np.isfinite(want[t])
        assert (np.isfinite(got[t]) == ok).all(), t
        assert not ok.any() or rel(got[t][ok], want[t][ok]) < 2e-5, t                # as test_ssm


@pytest.mark.parametrize("N", [1, 64])
def test_ssm_scan_in_one_part_has_two_blocks_per_cu(N):
    """a block is eight waves, so that two need no more than 128 registers; what brings states along for parts of the tokens must not cost launches that fill the chip their second block"""
    assert bamd_lib().bamd_op_ssm_blocks(N, 1) == 2


def plain_attention(q, c, gate, past, uk, uv, c_norm, sink, scale, eps, H):
    T, _, d = q.shape
    lat = np.stack([so.rms(v, eps) * c_norm for v in c])
    every = lat if past is None else np.concatenate([past, lat])
    uk, uv = so.bf16_to_f32(uk).astype(np.float64), so.bf16_to_f32(uv).astype(np.float64)
    k, v = (every @ uk.T).reshape(len(every), H, d), (every @ uv.T).reshape(len(every), H, -1)
    out = np.zeros((T, H, v.shape[2]))
    for t in range(T):
        n = len(every) - T + t + 1
        for h in range(H):
            s = k[:n, h] @ q[t, h] * scale
            p = so.sink_softmax(s, sink[h]) if sink is not None else np.exp(s - s.max()) / np.exp(s - s.max()).sum()
            out[t, h] = p @ v[:n, h] * (so.sigmoid(gate[t, h]) if gate is not None else 1)
    return out


def attention_case(H, d, dv, R, T, pos0, seed, dtype):
    r = np.random.default_rng(seed)
    rd = so.round_bf16 if dtype == "bfloat16" else (lambda a: np.asarray(a, np.float32))
    return dict(q=rd(r.standard_normal((T, H, d))), c=rd(r.standard_normal((T, R))), gate=r.standard_normal((T, H)).astype(np.float32), past=rd(r.standard_normal((pos0, R))) if pos0 else None,
                uk=so.f32_to_bf16(r.standard_normal((H * d, R)) / np.sqrt(R)), uv=so.f32_to_bf16(r.standard_normal((H * dv, R)) / np.sqrt(R)), c_norm=rd(1 + 0.2 * r.standard_normal(R)),
                sink=r.standard_normal(H).astype(np.float32), scale=1.5 / np.sqrt(d), eps=1e-5)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("H,d,dv,R", [(1, 8, 8, 8), (3, 24, 40, 36), (5, 33, 12, 20), (17, 16, 32, 64), (2, 72, 130, 100), (2, 128, 64, 200), (1, 200, 16, 300), (2, 64, 128, 700)])
@pytest.mark.parametrize("T,pos0", [(1, 0), (3, 0), (63, 0), (130, 0), (2, 63), (2, 64), (66, 130), (1, 63), (1, 64), (1, 200), (1, 500)])
def test_latent_attention(bamd, dtype, H, d, dv, R, T, pos0):
    a = attention_case(H, d, dv, R, T, pos0, H * d + T + pos0, dtype)
    want = plain_attention(H=H, **a)
    for decode in ((False, True) if T == 1 else (False,)):
        got = bamd.op_latent_attention(dtype=dtype, decode=decode, **a)
        near(got.reshape(T, -1), want.reshape(T, -1), dtype)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("H,d,dv,R", [(1, 8, 8, 8), (3, 24, 40, 36), (17, 16, 32, 64), (2, 72, 128, 100), (2, 128, 64, 256), (3, 100, 96, 264), (2, 128, 128, 512)])
@pytest.mark.parametrize("pos0", [0, 1, 15, 63, 64, 127, 128, 191, 192, 255, 256, 257, 520, 1100])
def test_latent_attention_step_in_one_launch(bamd, dtype, H, d, dv, R, pos0):
    """the token's own latent alone, first and last of a chunk of cached ones (64 to 256, by the rank and the type), whole chunks and a part"""
    a = attention_case(H, d, dv, R, 1, pos0, H * d + pos0, dtype)
    near(bamd.op_latent_attention(dtype=dtype, decode=2, **a).reshape(1, -1), plain_attention(H=H, **a).reshape(1, -1), dtype)


def test_latent_attention_step_weighs_shares_in_32_bits():
    """scores that are whole numbers, a share for every key, and values that keep the keys apart: what is left of an output's error is its share's weight.  An exponential of a product rounded to 32 bits
    is off by up to 3e-6 here (half an ulp of 62 log2(e)); one to an ulp and a half, the sum, the quotient and the products are no more than eight roundings of 2^-24"""
    import booster_amd as bamd
    n, d = 32, 8
    scores = np.random.default_rng(2).permutation(np.arange(n) * 2 + 3).astype(np.float32)
    past = np.zeros((n, n), np.float32)
    past[:, 0] = scores
    past[np.arange(1, n), np.arange(1, n)] = 1
    uk, q, cn = np.zeros((d, n)), np.zeros((1, 1, d), np.float32), np.ones(n, np.float32)
    uk[0, 0], q[0, 0, 0], cn[0] = 1, 1, 0                 # (the token's own score: zero)
    c = np.zeros((1, n), np.float32)
    c[0, 0] = 1
    uv = np.eye(n)[1:]
    a = dict(q=q, c=c, gate=None, past=past, uk=so.f32_to_bf16(uk), uv=so.f32_to_bf16(uv), c_norm=cn, sink=None, scale=1.0, eps=1e-5)
    want = plain_attention(H=1, **a)
    got = bamd.op_latent_attention(dtype="float32", decode=2, **a)
    assert np.abs(got / want - 1).max() < 5e-7


@pytest.mark.parametrize("H,d,R,T,pos0", [(128, 24, 20, 257, 0), (128, 24, 20, 512, 70), (128, 24, 20, 513, 0), (85, 40, 36, 700, 130)])
def test_latent_attention_in_paired_blocks(bamd, H, d, R, T, pos0):
    """tiles of 128 queries: one block per CU and a part of a second, two (taken the other way round), two and a part of a third (plain order), and heads that do not divide the CUs"""
    a = attention_case(H, d, d, R, T, pos0, H + T, "bfloat16")
    want = plain_attention(H=H, **a)
    near(bamd.op_latent_attention(dtype="bfloat16", **a).reshape(T, -1), want.reshape(T, -1), "bfloat16")


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("T,pos0", [(3, 65600), (70, 65470)])
def test_latent_attention_behind_many_positions(bamd, dtype, T, pos0):
    """more cached rows than a grid's y axis may have blocks"""
    a = attention_case(2, 24, 40, 36, T, pos0, T, dtype)
    want = plain_attention(H=2, **a)
    near(bamd.op_latent_attention(dtype=dtype, **a).reshape(T, -1), want.reshape(T, -1), dtype, 3)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("pos0", [0, 127, 250])
def test_one_key_stands_out(bamd, dtype, pos0):
    """one score far above hundreds of others, at the first positions, on both sides of every page border, at the query itself, and just behind it (never seen)"""
    H, d, dv, R, n = 2, 24, 40, 36, 300
    T = n - pos0
    a = attention_case(H, d, dv, R, n, 0, 77, dtype)
    lat = np.stack([so.rms(v, a["eps"]) * a["c_norm"] for v in a["c"]])
    k = (lat @ so.bf16_to_f32(a["uk"]).T.astype(np.float64)).reshape(n, H, d)
    for key in (0, 1, 2, 62, 63, 64, 65, 127, 128, 191, 192, 250, 255, 256, 298, 299):
        q = np.zeros((n, H, d))
        q[:] = k[key] / (k[key] ** 2).sum(-1, keepdims=True)
        rd = so.round_bf16 if dtype == "bfloat16" else (lambda v: np.asarray(v, np.float32))
        case = dict(a, q=rd(q[pos0:]), c=a["c"][pos0:], gate=a["gate"][pos0:], past=rd(lat[:pos0]) if pos0 else None, scale=24.0)
        want = plain_attention(H=H, **case)
        near(bamd.op_latent_attention(dtype=dtype, **case).reshape(T, -1), want.reshape(T, -1), dtype, 3)
    # the same, decoded: the query is the last position
    for key in (0, 63, 64, 191, 298, 299):
        case = dict(a, q=rd(k[key][None] / (k[key] ** 2).sum(-1)[None, :, None]), c=a["c"][-1:], gate=a["gate"][-1:], past=rd(lat[:-1]), scale=24.0)
        want = plain_attention(H=H, **case)
        for decode in (True, 2):
            near(bamd.op_latent_attention(dtype=dtype, decode=decode, **case).reshape(1, -1), want.reshape(1, -1), dtype, 3)


@pytest.mark.parametrize("scale", [0.125, 0.13])
def test_scores_far_from_zero(bamd, scale):
    """whole numbers that 32 bits hold exactly, thousands from zero and a few from one another, beside a sink among them and one far below: what a score or a maximum is rounded by (2^-13 of the
    exponent here, 1e-4 of a weight) must not show in the weights"""
    H, d, R, n, T = 2, 64, 32, 200, 70
    a = attention_case(H, d, 16, R, T, n, 3, "float32")
    r = np.random.default_rng(4)
    past = r.integers(-3, 4, (n, R)).astype(np.float32)
    past[:, 0] = 200
    q = np.zeros((T, H, d), np.float32)
    q[:, :, 1:R] = r.integers(-2, 3, (T, H, R - 1))
    q[:, :, 0] = 160
    uk = np.zeros((H, d, R), np.float32)
    uk[:, np.arange(R), np.arange(R)] = 1
    uv = a["uv"].copy()
    uv[:, 0] = 0
    a = dict(a, q=q, past=past, uk=so.f32_to_bf16(uk.reshape(H * d, R)), uv=uv, sink=np.array([32005 * scale, -5], np.float32), scale=scale)
    want = plain_attention(H=H, **dict(a, scale=float(np.float32(scale))))
    near(bamd.op_latent_attention(dtype="float32", **a).reshape(T, -1), want.reshape(T, -1), "float32")


@pytest.mark.parametrize("decode", [False, True, 2])
@pytest.mark.parametrize("dtype", DTYPES)
def test_sinks_and_gates(bamd, dtype, decode):
    """sinks from nothing to almost everything, none at all, gates open, shut and absent"""
    H, d, dv, R = 4, 16, 16, 24
    a = attention_case(H, d, dv, R, 1, 150, 5, dtype)
    for sink in ([-60, -2, 4, 9], [80, 0, 30, -80], None):
        for gate in (np.array([[-30, -1, 2, 30.]], np.float32), None):
            case = dict(a, sink=None if sink is None else np.array(sink, np.float32), gate=gate)
            want, got = plain_attention(H=H, **case), bamd.op_latent_attention(dtype=dtype, decode=decode, **case)
            live = np.abs(want).max(-1) > 1e-6
            near(got[live], want[live], dtype)
            assert np.abs(got[~live]).max(initial=0) < 1e-6


# ---- whole models ------------------------------------------------------------------------------------------------------------------------------------------
class Case:
    def __init__(self, folder, cfg, seed, rows=None):
        self.folder, self.cfg = folder, cfg
        w = so.random_model(cfg, seed, rows)
        so.write_model(folder, cfg, w)
        self.oracle = so.StackModel(cfg, w)
        self.known = {}

    def logits(self, toks):
        key = tuple(toks)
        if key not in self.known:
            self.known[key] = self.oracle.forward(toks)
        return self.known[key]


@pytest.fixture(scope="module")
def cases(tmp_path_factory):
    d = tmp_path_factory.mktemp("stack")
    return {n: Case(str(d / n), c, SEEDS[n], ROWS.get(n)) for n, c in sorted(CONFIGS.items())}


# a rank of 512: one launch for the latent attention of up to 324 positions in bfloat16, 252 in 32-bit, three behind them; a rank that takes three throughout.
# Weights by their condition: the oracle with every product's operands rounded to bfloat16 moves no row behind position 150 of the tests' tokens by more than 0.0112 (weights 5: 0.051)
LONG_LATENT = config(64, 97, [latent(3, 24, 40, 512, 0.31, ff=70), mamba(3, 20, 24, 1, 5, 3), latent(2, 33, 12, 600, 0.2, ff=50)])


@pytest.fixture(scope="module")
def long_latent(tmp_path_factory):
    return Case(str(tmp_path_factory.mktemp("long_latent") / "m"), LONG_LATENT, 13)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("rows", [1, 3])
def test_latent_steps_that_outgrow_one_launch(bamd, long_latent, dtype, rows):
    """sequences of different lengths decoded across the most positions that one launch takes"""
    m = bamd.Model(long_latent.folder, dtype=dtype)
    c = bamd.Context(m, 448 * rows, rows)
    for most in ((318,) if dtype == "bfloat16" else (246,)):
        t = [tokens(LONG_LATENT, most + 12, 30 + i) for i in range(rows)]
        want = [long_latent.logits(x) for x in t]
        at = [most - 40 * s for s in range(rows)]
        for s in range(rows): c.seq_free(s)
        c.decode_batch([(s, t[s][:at[s]], [at[s] - 1]) for s in range(rows)])
        for _ in range(12):
            got = c.decode_batch([(s, [t[s][at[s]]], [0]) for s in range(rows)])
            near(got, np.stack([want[s][at[s]] for s in range(rows)]), dtype)
            at = [a + 1 for a in at]
    c.close(); m.close()


@pytest.mark.parametrize("dtype", DTYPES)
def test_generating_across_the_limit_of_one_launch_is_stepping_across_it(bamd, long_latent, dtype):
    """the logits behind steps enqueued at once are those, bit for bit, of the same steps one call each, however many of them run behind the limit"""
    m = bamd.Model(long_latent.folder, dtype=dtype)
    c = bamd.Context(m, 512, 1)
    at = 318 if dtype == "bfloat16" else 246
    p = tokens(LONG_LATENT, at, 7)
    for steps in (4, 36):
        c.seq_free(0)
        c.decode(p, 0)
        out, _ = c.generate_greedy(at, steps)
        last = c.last_logits()
        c.seq_free(0)
        c.decode(p, 0)
        for i in range(steps): one = c.decode([out[i]], at + i)
        assert np.array_equal(last.view(np.uint32), one.view(np.uint32)), steps
    c.close(); m.close()


@pytest.fixture(params=[(n, t) for n in sorted(CONFIGS) for t in DTYPES], ids=lambda p: "-".join(p))
def run(request, bamd, cases):
    name, dtype = request.param
    m = bamd.Model(cases[name].folder, dtype=dtype)
    c = bamd.Context(m, 512, 4)
    yield cases[name], c, dtype
    c.close(); m.close()


def everywhere(toks):
    return list(range(len(toks)))


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("width", [75, 76])
@pytest.mark.parametrize("design", ["Tupitar", "Mafurax"])
def test_models_whose_products_are_halved(bamd, dtype, width, design, tmp_path):
    """output and down projections of 5 row tiles and 66 column blocks: their halves meet in the residual sum behind them, of prompts, of a few sequences and of one, in rows that are kept in
    registers and in rows that are not"""
    if design == "Tupitar":
        cfg = stack_cases.config(width, 131, [stack_cases.mamba(33, 64, 8, 1, 1, 2, ff=2100), stack_cases.latent(9, 24, 250, 36, 0.31, ff=2100)])
    else:
        cfg = stack_cases.mafurax(width, 131, [stack_cases.parallel(stack_cases.attend(17, 1, 24, 120, 0.4, 6.0, 50, 19, 3), 0.7, (3, 10, 14, 8.0), 1.3, ff=2100, limit=0.8)])
    case = Case(str(tmp_path / "m"), cfg, 3, dict(rel=8, rank=5))
    m = bamd.Model(case.folder, dtype=dtype)
    c = bamd.Context(m, 512, 3)
    t = [tokens(cfg, 76, 30 + i) for i in range(3)]
    for n in (70, 9, 1):
        near(c.decode_batch([(0, t[0][:n], everywhere(t[0][:n]))]), case.logits(t[0])[:n], dtype)
        c.seq_free(0)
    got = c.decode_batch([(i, t[i][:70 - i], [69 - i]) for i in range(3)])
    near(got, np.stack([case.logits(t[i])[69 - i] for i in range(3)]), dtype)
    for k in range(3):
        got = c.decode_batch([(i, [t[i][70 - i + k]], [0]) for i in range(3)])
        near(got, np.stack([case.logits(t[i])[70 - i + k] for i in range(3)]), dtype)
    near(c.decode_batch([(1, [t[1][72]], [0])])[0], case.logits(t[1])[72], dtype)
    c.close(); m.close()


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("design", ["Tupitar", "Mafurax"])
def test_a_context_that_is_just_large_enough_gives_the_same_bits(bamd, dtype, design, tmp_path):
    """products of 5 row tiles and 66 column blocks, which are halved: with every row of the context's scratch in use as with a fraction of it"""
    if design == "Tupitar":
        cfg = stack_cases.config(76, 131, [stack_cases.mamba(33, 64, 8, 1, 1, 2, ff=2100), stack_cases.latent(9, 24, 250, 36, 0.31, ff=2100)], max_positions=1024)
    else:
        cfg = stack_cases.mafurax(76, 131, [stack_cases.parallel(stack_cases.attend(17, 1, 24, 120, 0.4, 6.0, 50, 19, 3), 0.7, (3, 10, 14, 8.0), 1.3, ff=2100, limit=0.8)])
    m = bamd.Model(Case(str(tmp_path / "m"), cfg, 3, dict(rel=8, rank=5)).folder, dtype=dtype)
    for n in (64, 320):
        got = []
        for n_ctx in (n, 1024):
            c = bamd.Context(m, n_ctx, 1)
            got.append(c.decode(tokens(cfg, n, 30), 0))
            c.close()
        assert np.array_equal(got[0].view(np.uint32), got[1].view(np.uint32)), n
    m.close()


@pytest.mark.parametrize("n", [1, 2, 3, 5, 64, 65, 150])
def test_prompt(run, n):
    case, c, dtype = run
    t = tokens(case.cfg, 150, 1)[:n]
    near(c.decode_batch([(0, t, everywhere(t))]), case.logits(tokens(case.cfg, 150, 1))[:n], dtype)


def test_prompt_against_decoding(run):
    """token by token from the first one, over two page borders"""
    case, c, dtype = run
    t = tokens(case.cfg, 150, 1)
    got = np.concatenate([c.decode_batch([(2, [x], [0])]) for x in t])
    near(got, case.logits(t), dtype)


@pytest.mark.parametrize("size", [2, 3, 7, 33, 64, 65, 100])
def test_portions(run, size):
    case, c, dtype = run
    t = tokens(case.cfg, 150, 1)
    got = np.concatenate([c.decode_batch([(1, t[i:i + size], everywhere(t[i:i + size]))]) for i in range(0, len(t), size)])
    near(got, case.logits(t), dtype)
    assert c.seq_len(1) == 150


def test_unequal_batch_against_each_alone(run):
    case, c, dtype = run
    lens = [1, 70, 23, 129]
    t = [tokens(case.cfg, n + 10, 20 + n) for n in lens]
    got = c.decode_batch([(s, t[s][:n], everywhere(t[s][:n])) for s, n in enumerate(lens)])
    at = 0
    for s, n in enumerate(lens):
        near(got[at:at + n], case.logits(t[s])[:n], dtype)
        at += n
    for k in range(10):                                   # decoded together; the shorter ones stop earlier
        live = [s for s in range(4) if k < 4 + 2 * s]
        got = c.decode_batch([(s, [t[s][lens[s] + k]], [0]) for s in live])
        for g, s in zip(got, live):
            near(g, case.logits(t[s])[lens[s] + k], dtype)
        for s in range(4):
            if k == 3 + 2 * s:
                c.seq_free(s)


def test_mixed_batch(run):
    """a decoding sequence, a continued prompt and a fresh one in the same batch; places wanted in one of them only"""
    case, c, dtype = run
    t = tokens(case.cfg, 150, 1)
    c.decode_batch([(0, t[:80], []), (1, t[:5], [])])
    got = c.decode_batch([(1, t[5:71], [0, 65]), (0, t[80:81], [0]), (3, t[:9], [])])
    near(got, case.logits(t)[[5, 70, 80]], dtype)
    got = c.decode_batch([(0, t[81:82], [0]), (1, t[71:72], []), (3, t[9:10], [0])])
    near(got, case.logits(t)[[81, 9]], dtype)


def test_pages_and_sequences_used_again(run):
    case, c, dtype = run
    t, u = tokens(case.cfg, 150, 1), tokens(case.cfg, 140, 9)
    for s in range(4):
        c.decode_batch([(s, u[:100 + s], [])])
    for s in (2, 0):
        c.seq_free(s)
    near(c.decode_batch([(2, t[:70], everywhere(t[:70]))]), case.logits(t)[:70], dtype)
    near(c.decode_batch([(0, t[:3], [0, 1, 2])]), case.logits(t)[:3], dtype)
    got = c.decode_batch([(1, u[101:102], [0]), (3, u[103:104], [0]), (2, t[70:71], [0]), (0, t[3:4], [0])])
    near(got[2:], case.logits(t)[[70, 3]], dtype)
    near(got[:2], case.logits(u)[[101, 103]], dtype)
    for s in range(4):
        c.seq_free(s)
    near(c.decode_batch([(3, t, everywhere(t))]), case.logits(t), dtype)


def test_decode_interface(run):
    """bamd_decode on sequence 0: a new prompt at position 0 replaces it, positions cannot be taken back"""
    import booster_amd
    case, c, dtype = run
    t = tokens(case.cfg, 150, 1)
    c.decode(t[:30], 0)
    near(c.decode(t[:40], 0), case.logits(t)[39], dtype)
    near(c.decode(t[40:41], 40), case.logits(t)[40], dtype)
    near(c.last_logits(), case.logits(t)[40], dtype)
    with pytest.raises(booster_amd.BamdError, match="41 tokens"):
        c.decode(t[:5], 30)
    with pytest.raises(booster_amd.BamdError):
        c.kv_seq_add(0, 10, 1)
    with pytest.raises(booster_amd.BamdError):
        c.kv_seq_rm(10, -1)
    c.kv_seq_rm(0, -1)
    assert c.seq_len(0) == 0


@pytest.mark.parametrize("read_every", [1, 2, 5])
def test_decoding_steps_read_or_not(run, read_every):
    """decoding steps whose logits go to the host, and steps that nobody waits for in between (descriptors by way of pinned memory): the same bits, whoever reads when"""
    case, c, dtype = run
    t = tokens(case.cfg, 100, 1)
    L = bamd_lib()
    rows = []
    c.decode(t[:60], 0)
    want = {k: c.decode(t[k:k + 1], k) for k in range(60, 80)}
    c.decode(t[:60], 0)
    try:
        for n_past in range(60, 80):
            L.bamd_set_logits_readback(c.h, 0)
            tok = np.ascontiguousarray(t[n_past:n_past + 1], np.int32)
            if (n_past + 1) % read_every:
                assert L.bamd_decode(c.h, tok.ctypes.data, 1, n_past) == 0
                continue
            L.bamd_set_logits_readback(c.h, n_past % 2)
            rows.append((n_past, c.decode(tok, n_past), c.last_logits()))
    finally:
        L.bamd_set_logits_readback(c.h, 1)
    for k, a, b in rows:
        assert np.array_equal(a.view(np.uint32), want[k].view(np.uint32)) and np.array_equal(a.view(np.uint32), b.view(np.uint32)), k
    near(rows[-1][1], case.logits(t)[rows[-1][0]], dtype)
    c.seq_free(0)


def test_greedy_generation(run):
    """the device loop, the same in a batch of unequal sequences, and the scheduler over more requests than sequences: the same tokens; in 32-bit the plain statement's"""
    from booster_amd.scheduler import Scheduler
    case, c, dtype = run
    prompts = [tokens(case.cfg, n, 40 + n) for n in (1, 63, 20, 40, 7, 64)]
    n_new = 12
    alone, first = [], []
    for p in prompts:
        first.append(int(np.argmax(c.decode(p, 0))))
        out, _ = c.generate_greedy(len(p), n_new - 1)
        assert out[0] == first[-1]
        last = c.last_logits()
        alone.append([int(x) for x in out])
        assert int(np.argmax(last)) == alone[-1][-1]
        c.seq_free(0)
    if dtype == "float32":
        for p, a in zip(prompts[:4], alone):
            st = case.oracle.new_state()
            l = case.oracle.forward(p, st)[-1]
            for tok in a:
                top = np.sort(l)[-2:]
                assert int(np.argmax(l)) == tok or top[1] - top[0] < 1e-4 * np.abs(l).max()
                l = case.oracle.forward([tok], st)[-1]
    for s in range(4):
        c.decode_batch([(s, prompts[s], [])])
    out, _ = c.generate_greedy_seqs([0, 1, 2, 3], first[:4], n_new - 1)
    for s in range(4):
        c.seq_free(s)
    sched = Scheduler(c).generate(prompts, n_new)
    if dtype == "float32":
        assert [[int(x) for x in o] for o in out] == alone[:4] and sched == alone
    else:                                                 # rounding may pick another of two near equals: the first tokens agree
        assert [int(o[0]) for o in out] == first[:4] and [o[0] for o in sched] == first


@pytest.mark.parametrize("name", ["odd", "side", "side_long"])
def test_long_decoding(bamd, cases, name):
    """hundreds of decoded tokens behind a short prompt: in one device loop, then token by token, over page borders; the state of a sequence beside it stays"""
    case = cases[name]
    m = bamd.Model(case.folder, dtype="float32"); c = bamd.Context(m, 704, 2)
    p = tokens(case.cfg, 6, 3)
    c.decode_batch([(1, tokens(case.cfg, 9, 4), [])])
    c.decode(p, 0)
    out, _ = c.generate_greedy(len(p), 301)
    seq = p + [int(x) for x in out[:-1]]
    want = case.logits(seq)
    near(c.last_logits(), want[-1], "float32")
    assert all(int(np.argmax(l)) == int(t) for l, t in zip(want[len(p) - 1:], out))
    more = tokens(case.cfg, 30, 5)
    st = case.oracle.new_state(); case.oracle.forward(seq, st)
    ref = case.oracle.forward(more, st)
    near(np.stack([c.decode([t], len(seq) + i) for i, t in enumerate(more)]), ref, "float32")
    near(c.decode_batch([(1, [1], [0])])[0], case.logits(tokens(case.cfg, 9, 4) + [1])[-1], "float32")
    c.close(); m.close()


@pytest.mark.parametrize("design", ["Tupitar", "Mafurax"])
@pytest.mark.parametrize("dtype", DTYPES)
def test_many_wanted_places_and_passes(bamd, dtype, design, tmp_path):
    """more rows than one pass holds (2048), more wanted places than the logits buffer, a prompt cut between passes, a wide latent and larger matrices; scans in segments, a window and kept
    tokens far behind the queries"""
    cfg = config(128, 97, [latent(2, 16, 24, 40, 0.3, ff=64), mamba(2, 12, 10, 1, 1, 4, ff=48)], max_positions=1600)
    if design == "Mafurax":
        cfg = mafurax(128, 97, [parallel(attend(4, 2, 16, 24, 0.5, 10.0, 120, 200, 9), 0.8, (2, 20, 24, 16.0), 1.0, ff=64, limit=1.0),
                                parallel(attend(2, 1, 24, 16, 0.4, 12.0, 800, 900, 0), 0.8, (3, 12, 16, 16.0), 1.0, ff=48, limit=1.0)])
    case = Case(str(tmp_path / "m"), cfg, 3)
    m = bamd.Model(case.folder, dtype=dtype); c = bamd.Context(m, 3200, 3)
    t = [tokens(cfg, n, n) for n in (900, 1500, 40)]
    want = [[0, 899], list(range(1200, 1400)) + [1499], everywhere(t[2])]
    got = c.decode_batch([(s, t[s], want[s]) for s in range(3)])
    at = 0
    for s in range(3):
        near(got[at:at + len(want[s])], case.logits(t[s])[want[s]], dtype, 2)      # the worst of some 240 rows
        at += len(want[s])
    c.close(); m.close()


def test_limits(bamd, cases):
    import booster_amd
    case = cases["odd"]
    m = bamd.Model(case.folder, dtype="bfloat16"); c = bamd.Context(m, 1024, 2)
    t = tokens(case.cfg, 700, 1)
    c.decode_batch([(0, t, [])])
    for bad in ([(0, [1], [0])],                          # behind the last learned position
                [(2, [1], [0])], [(1, [], [])], [(1, [case.cfg["vocab"]], [0])], [(1, [-1], [0])], [(1, [1, 2], [2])], [(1, [1, 2], [1, 0])], [(1, [1], []), (1, [2], [])],
                [(1, t[:480], [])]):                      # 700 + 480 positions do not fit
        with pytest.raises(booster_amd.BamdError):
            c.decode_batch(bad)
    assert c.seq_len(0) == 700 and c.seq_len(1) == 0      # refused batches leave the sequences alone
    with pytest.raises(booster_amd.BamdError):
        c.generate_greedy(700, 1)
    near(c.decode_batch([(1, t[:50], [49])]), case.logits(t[:50])[-1:], "bfloat16")
    c.close(); m.close()
    broken = dict(case.cfg, layers=[dict(case.cfg["layers"][0], type="nope")])
    os.makedirs(case.folder + "_b", exist_ok=True)
    json.dump(broken, open(case.folder + "_b/config.json", "w"))
    if not os.path.exists(case.folder + "_b/model.safetensors"):
        os.symlink(case.folder + "/model.safetensors", case.folder + "_b/model.safetensors")
    with pytest.raises(booster_amd.BamdError, match="nope"):
        bamd.Model(case.folder + "_b")
    json.dump(dict(case.cfg, width=76), open(case.folder + "_b/config.json", "w"))
    with pytest.raises(booster_amd.BamdError, match="expected shape"):
        bamd.Model(case.folder + "_b")


@pytest.mark.parametrize("name", ["odd", "side"])
@pytest.mark.parametrize("dtype", DTYPES)
def test_layer_split_stages(bamd, cases, dtype, name):
    """the layers over two stages with the hidden state handed over: prompt, portions and single tokens"""
    import torch
    case = cases[name]
    t = tokens(case.cfg, 150, 1)
    E = case.cfg["width"]
    a = bamd.Model(case.folder, layer_first=0, layer_last=1, with_output=False, dtype=dtype)
    b = bamd.Model(case.folder, layer_first=1, layer_last=-1, with_embd=False, dtype=dtype)
    ca, cb = bamd.Context(a, 256), bamd.Context(b, 256)
    hid = torch.zeros((128, E), device="cuda", dtype=torch.float32)
    tok = torch.zeros(1, device="cuda", dtype=torch.int32)
    s = torch.cuda.current_stream().cuda_stream
    pos = 0
    for n in (70, 2, 33):
        assert ca.stage_prefill(t[pos:pos + n], n, pos, None, hid.data_ptr(), False, s)
        assert cb.stage_prefill(None, n, pos, hid.data_ptr(), None, True, s)
        pos += n
        near(cb.stage_logits(s), case.logits(t)[pos - 1], dtype)
    for _ in range(6):
        tok.fill_(t[pos])
        ca.stage_step(0, pos, None, hid.data_ptr(), 0, 0, s, token_dev_ptr=tok.data_ptr())
        cb.stage_step(0, pos, hid.data_ptr(), None, 1, 0, s)
        pos += 1
        near(cb.stage_logits(s), case.logits(t)[pos - 1], dtype)
        assert cb.stage_argmax(s) == int(np.argmax(cb.stage_logits(s)))
        cb.stage_token_to(tok.data_ptr(), s); torch.cuda.synchronize()
        assert int(tok[0]) == int(np.argmax(cb.stage_logits(s)))
    for x in (ca, cb, a, b):
        x.close()


@pytest.mark.parametrize("name", ["wide", "side_wide"])
def test_replays_with_other_work_between(bamd, cases, name):
    """the decoding graph, replayed with prompts, other sequences and eager work between its replays, gives what a fresh context gives"""
    case = cases[name]
    t = tokens(case.cfg, 80, 6)
    m = bamd.Model(case.folder, dtype="float32"); c = bamd.Context(m, 512, 3)
    c.decode_batch([(0, t[:40], [])])
    for k in range(40, 60):
        got = c.decode_batch([(0, [t[k]], [0])])
        near(got, case.logits(t)[k:k + 1], "float32")
        if k % 3 == 0:
            c.decode_batch([(1, t[:k], [k - 1])]); c.decode_batch([(1, [t[k]], [])]); c.seq_free(1)
        if k % 4 == 0:
            near(bamd.op_poly_norm(np.ones((2, 40)), [1, 1, 1, 1], 0.0, "float32"), np.full((2, 40), 4.0), "float32")
        if k % 5 == 0:
            c.decode_batch([(2, [t[0]], [0])]); c.seq_free(2)
    c.close(); m.close()


@pytest.mark.parametrize("design", ["Tupitar", "Mafurax"])
def test_bridge_serves_a_model_folder(bamd, design, tmp_path):
    """initContext / doInference on a folder with tokenizer.gguf: prompt, Janus sampling on the device's logits, text out; without a tokenizer the request is refused"""
    from booster_amd import gguf
    from test_gpu_bridge import bind, ctx_args
    L = bind(bamd)
    vocab = gguf.synthetic_spm_vocab()
    cfg = config(60, len(vocab["tokens"]), [mamba(2, 12, 16, 1, 2, 4, ff=50), latent(3, 16, 20, 24, 0.3, ff=64)], max_positions=192)
    if design == "Mafurax":
        cfg = mafurax(60, len(vocab["tokens"]), [parallel(attend(4, 2, 16, 20, 0.4, 7.0, 30, 9, 2), 0.9, (2, 12, 16, 4.0), 0.8, ff=50, limit=0.9)])
    jobs = [(design + n).encode() for n in ("-none", "-a", "-b")]
    d = str(tmp_path / "m")
    so.write_model(d, cfg, so.random_model(cfg, 8))
    ctx = L.initContext(*ctx_args(6, d, (100, 0, 0, 0), 128, 24))
    assert ctx and L.doInference(6, ctx, jobs[0], b"s", b"the cat sat") == 1
    gguf.write_synthetic_llama(d + "/tokenizer.gguf", E=256, H=2, Hkv=1, L=1, F=256, V=len(vocab["tokens"]), seed=2, vocab=vocab)
    ctx = L.initContext(*ctx_args(6, d, (100, 0, 0, 0), 128, 24))
    assert ctx
    for job in jobs[1:]:                  # the second request starts over in the same context
        n = L.doInference(6, ctx, job, b"s", b"the cat sat on the hat")
        prompt = L.getPromptTokenCount(job)
        assert prompt > 4 and prompt <= n <= prompt + 23
        text = L.status(job)
        assert b"the cat sat on the hat" in text
    # hi = lo = 1: only the top candidate survives, the draw is the arg-max of the penalised logits and both requests agree
    assert L.status(jobs[1]) == L.status(jobs[2])


@pytest.mark.parametrize("name", ["odd", "side"])
def test_trace_run(bamd, cases, name, tmp_path):
    """bin/trace_run replays requests step by step and writes the wanted logits"""
    case = cases[name]
    t = tokens(case.cfg, 150, 1)
    steps = [{"step": 0, "entries": [{"id": "x", "tokens": t[:70], "want": [69, 3]}, {"id": "y", "tokens": t[:5], "want": []}], "end": []},
             {"step": 1, "entries": [{"id": "y", "tokens": [t[5]], "want": [0]}, {"id": "x", "tokens": [t[70]], "want": [0]}], "end": ["y"]},
             {"step": 2, "entries": [{"id": "x", "tokens": [t[71]], "want": []}], "end": ["x"]},
             {"step": 3, "entries": [{"id": "y", "tokens": t[:9], "want": [8]}], "end": ["y"]}]
    for dtype in DTYPES:
        out = tmp_path / dtype
        out.mkdir()
        p = subprocess.run([sys.executable, os.path.join(ROOT, "bin", "trace_run"), "--model", case.folder, "--dtype", dtype, "--out", str(out), "--max-tokens", "256"],
                           input="".join(json.dumps(s) + "\n" for s in steps), capture_output=True, text=True, timeout=100)
        assert p.returncode == 0, p.stderr[-2000:]
        assert [l for l in p.stdout.splitlines() if l.startswith("done")] == ["done %d" % i for i in range(4)]
        want = case.logits(t)
        for step, rows in ((0, [69, 3]), (1, [5, 70]), (3, [8])):
            got = np.fromfile(str(out / ("%d.f32" % step)), "<f4").reshape(len(rows), -1)
            near(got, want[rows], dtype)
        assert not (out / "2.f32").exists()


@pytest.mark.parametrize("name", ["odd", "side"])
def test_command_line(bamd, cases, name, capsys):
    """python -m booster_amd: several requests of a folder together; a GGUF model through the same scheduler, one request after the other"""
    from booster_amd.__main__ import main
    from conftest import GOLDEN
    case = cases[name]
    prompts = [tokens(case.cfg, n, n) for n in (5, 70, 33)]
    assert main(["--model", case.folder, "--dtype", "float32", "-n", "6"] + [x for p in prompts for x in ("--tokens", ",".join(map(str, p)))]) == 0
    got = [[int(t) for t in l.split(",")] for l in capsys.readouterr().out.split()]
    m = bamd.Model(case.folder, dtype="float32"); c = bamd.Context(m, 128)
    for p, g in zip(prompts, got):
        first = int(np.argmax(c.decode(p, 0)))
        assert g == [int(x) for x in c.generate_greedy(len(p), 5)[0]] and g[0] == first
    c.close(); m.close()
    path = os.path.join(GOLDEN, "tiny_a.gguf")
    assert main(["--model", path, "-n", "6", "--tokens", "1,5,9,2", "--tokens", "3,4"]) == 0
    got = [[int(t) for t in l.split(",")] for l in capsys.readouterr().out.split()]
    m = bamd.Model(path); c = bamd.Context(m, 128)
    for p, g in zip(([1, 5, 9, 2], [3, 4]), got):
        c.decode(p, 0)
        assert g == [int(x) for x in c.generate_greedy(len(p), 5)[0]]
    c.close(); m.close()
