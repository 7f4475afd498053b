"""GPU: the mechanisms of the Mafurax design alone, against oracle/stack_oracle.py — attention over cached keys and values, gated linear attention, layer norms around a
sublayer, the clamped gated unit.  Whole models: test_gpu_stack.py."""
import functools

import numpy as np
import pytest

from oracle import stack_oracle as so
import stack_cases
from stack_cases import tokens
from test_gpu_stack import Case, DTYPES, near, rel
from test_gpu_stack import test_poly_norm as poly_norm_case

pytestmark = pytest.mark.gpu


def rounder(dtype):
    return so.round_bf16 if dtype == "bfloat16" else (lambda a: np.asarray(a, np.float32))


# ---- rows --------------------------------------------------------------------------------------------------------------------------------------------------
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("E,rows,with_y,with_pre", [(75, 5, True, True), (2, 3, True, True), (96, 4, False, True), (96, 4, True, False), (300, 70, True, True), (1028, 2, True, True), (3000, 3, True, True), (9001, 2, True, True)])
def test_layer_norms_around_a_sublayer(bamd, dtype, E, rows, with_y, with_pre):
    """rows with means far from zero, and small and large spreads"""
    r = np.random.default_rng(E + rows)
    spread = 10.0 ** r.uniform(-1, 1, (rows, 1))
    x, y = r.standard_normal((rows, E)) * spread + 3, r.standard_normal((rows, E)) * spread[::-1] - 20 * spread[::-1]
    g, gi = r.standard_normal(E), 1 + 0.3 * r.standard_normal(E)
    xo, h = bamd.op_layer_rows(x, y if with_y else None, g, gi if with_pre else None, 1e-4, dtype)
    f = lambda a: np.asarray(a, np.float32).astype(np.float64)
    x, y = f(x), f(y)
    ref = np.stack([a + so.layer_norm(b, g, 1e-4) if with_y else a for a, b in zip(x, y)])
    near(xo, ref, "float32")
    near(h, np.stack([so.layer_norm(a, gi, 1e-4) for a in ref]) if with_pre else ref, dtype)


# The order of a layer norm's sums is fixed, to the bit: rows of whole pieces of four, and odd ones, which lie in registers one by one and are summed as longer ones are.  Lengths whose waves hold a
# power of two of the row, so that a wave's mean times its count is exact
@pytest.mark.parametrize("E", [4, 8, 256, 1024, 2048, 4096, 3, 587, 1023, 2050, 4095])
def test_sums_of_a_layer_norm_keep_their_order(bamd, E):
    f, rows = np.float32, 64
    t = bamd.lib().bamd_op_norm_threads(E, rows)
    def tree(a):                                                           # neighbours first; 64 lanes of a wave, sixteen waves
        while a.shape[-1] > 1:
            a = a[..., 0::2] + a[..., 1::2]
        return a[..., 0]
    def fma(a, b, c):
        return (a.astype(np.longdouble) * b + c).astype(f)
    def over_waves(a):
        return tree(np.concatenate([a, np.zeros((16 - a.shape[0]), f)]))
    def sum_of(a):
        return over_waves(tree(a.reshape(-1, 64)))
    def norm(y):
        if E % 4:                                                          # thread i: y[i], y[i + t], ...
            v = np.zeros(-(-E // t) * t, f); v[:E] = y
            v, there = v.reshape(-1, t), (np.arange(v.size) < E).reshape(-1, t)
            s = q = np.zeros(t, f)
            for a in v: s = s + a
            mean = sum_of(s) / f(E)
            for a, b in zip(v, there): q = np.where(b, fma(a - mean, a - mean, q), q)
            return mean, sum_of(q) / f(E)
        n = -(-E // (4 * t))                                               # thread i: pieces i, i + t, ...
        v = np.zeros(n * 4 * t, f); v[:E] = y
        v, there = v.reshape(n, t, 4), np.arange(n * t).reshape(n, t) < E // 4
        s = q = c = np.zeros(t, f)
        for a, b in zip(v, there): s, c = s + ((a[:, 0] + a[:, 1]) + (a[:, 2] + a[:, 3])), c + f(4) * b
        s, c = tree(s.reshape(-1, 64)), tree(c.reshape(-1, 64))
        m = np.where(c > 0, s / np.maximum(c, f(1)), f(0))
        for i, (a, b) in enumerate(zip(v, there)):
            d = a - np.repeat(m, 64)[:, None]
            p = fma(d[:, 0], d[:, 0], d[:, 1] * d[:, 1]) if i == 0 else fma(d[:, 1], d[:, 1], fma(d[:, 0], d[:, 0], q))
            q = np.where(b, fma(d[:, 3], d[:, 3], fma(d[:, 2], d[:, 2], p)), q)
        mean = over_waves(m * c) / f(E)
        return mean, over_waves(fma(c * (m - mean), m - mean, tree(q.reshape(-1, 64)))) / f(E)
    r = np.random.default_rng(E)
    x, y, g = (r.standard_normal(s, f) for s in ((rows, E), (rows, E), (E,)))
    y = y + f(0.3)
    want = np.stack([fma((b - mean) * (f(1) / np.sqrt(var + f(1e-6))), g, a) for a, b in zip(x, y) for mean, var in (norm(b),)])
    assert np.array_equal(bamd.op_layer_rows(x, y, g, None, 1e-6, "float32")[0].view(np.uint32), want.view(np.uint32))


# What a 32-bit row of operands holds is the rounded number, also where the last step in front of it is a product: factors that are known to the bit (means of zero, a root of 2^40, a single key)
@pytest.mark.parametrize("n", [64, 96, 5000, 301])
def test_operand_rows_hold_rounded_products(bamd, n):
    f = np.float32
    r = np.random.default_rng(n)
    y, w = r.standard_normal((3, n), f), r.standard_normal(n, f)
    same = lambda got, want: np.array_equal(got.view(np.uint32), want.view(np.uint32))
    assert same(bamd.op_group_norm(y, w, 1, 2.0 ** 40, "float32"), y * f(2.0 ** -20) * w)
    x = np.zeros((3, n), f)
    x[:, 0:n - 1:2], x[:, 1:n:2] = y[:, :n // 2], -y[:, :n // 2]                  # sums of zero, whatever their order
    xo, h = bamd.op_layer_rows(x, None, None, w, 2.0 ** 40, "float32")
    assert same(xo, x) and np.array_equal(h, x * f(2.0 ** -20) * w)
    q, k, v = (r.standard_normal((1, h, 64), f) for h in (6, 2, 2))
    for splits in (0, 1):
        got = bamd.op_kv_attention(q, k, v, None, None, None, 0.125, 30.0, 1e-6, False, None, 0, 100, 0, "float32", out_scale=0.7, splits=splits)
        assert same(got, np.repeat(v, 3, 1) * f(0.7)), splits


# widths just inside and outside of what a block of four or five waves keeps in registers, and widths that no block keeps
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("E", [1030, 2044, 2048, 2050, 2052, 2560, 2564, 4100])
def test_norms_of_rows_at_the_edge_of_a_block(bamd, dtype, E):
    r = np.random.default_rng(E)
    f = lambda a: np.asarray(a, np.float32).astype(np.float64)
    x, y, g, gi, mu, prev = f(r.standard_normal((3, E))), f(r.standard_normal((3, E)) - 2), f(r.standard_normal(E)), f(1 + 0.3 * r.standard_normal(E)), f(r.uniform(0, 1, E)), f(r.standard_normal(E))
    xo, h = bamd.op_layer_rows(x, y, g, gi, 1e-4, dtype)
    ref = np.stack([a + so.layer_norm(b, g, 1e-4) for a, b in zip(x, y)])
    near(xo, ref, "float32")
    near(h, np.stack([so.layer_norm(a, gi, 1e-4) for a in ref]), dtype)
    xo, h, last = bamd.op_residual_rows(x, y, 0.7, 1e-3, mu, prev, 5, dtype)
    ref = np.stack([a + so.scalar_norm(b, 0.7, 1e-3) for a, b in zip(x, y)])
    near(xo, ref, "float32")
    near(h, np.stack([so.token_shift(a, b, mu) for a, b in zip(ref, np.concatenate([prev[None], ref[:-1]]))]), dtype)
    near(last, ref[-1], "float32")


# odd lengths, which lie in registers one by one: the longest that a block holds, and one more
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("E,F", [(1023, 2047), (4095, 8191), (8191, 32767), (8193, 32769)])
def test_norms_of_rows_of_odd_lengths(bamd, dtype, E, F):
    test_norms_of_rows_at_the_edge_of_a_block(bamd, dtype, E)
    poly_norm_case(bamd, dtype, F)


# a step's logits, which the head brings to the host itself or leaves to a kernel behind it (33 to 64 bfloat16 rows of more than 768 row tiles and of whole pieces of four): vocabularies around the
# tiles and the rule, every form of the few-row product, a step after the other; against the prompt
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("V", [83, 4100, 12288, 12290, 12292])
def test_logits_of_steps(bamd, tmp_path, dtype, V):
    from booster_amd import synthetic
    layer = {"type": "mamba2", "mixer": dict(heads=2, vdim=32, state=32, groups=1, norm_groups=1, conv=4), "mlp": {"kind": "dense", "ff": 96}}
    cfg = {"architecture": "Tupitar", "vocab": V, "width": 64, "max_positions": 64, "embedding": {"scale": 1.0}, "norm": {"eps": 1e-6}, "layers": [layer]}
    synthetic.write_synthetic_stack(str(tmp_path / "m"), cfg)
    m = bamd.Model(str(tmp_path / "m"), dtype=dtype)
    for n in (1, 2, 16, 17, 32, 33, 64):
        a, b = bamd.Context(m, 64, n), bamd.Context(m, 64, n)
        t = np.random.default_rng(n).integers(0, V, (n, 3)).astype(np.int32)
        whole = a.decode_batch([(i, t[i], [0, 1, 2]) for i in range(n)]).reshape(n, 3, V)
        for k in range(3):
            near(b.decode_batch([(i, t[i, k:k + 1], [0]) for i in range(n)]), np.ascontiguousarray(whole[:, k]), dtype, 2.0)
        a.close(); b.close()
    m.close()


# and in front of the product of one row: blocks of 512 threads hold 4095 and not 4097, whatever the kind of norm; token by token against the prompt
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("kind,E", [("tupitar", 2047), ("tupitar", 4097), ("mafurax", 4095), ("mafurax", 4097)])
def test_odd_widths_token_by_token(bamd, tmp_path, dtype, kind, E):
    from booster_amd import synthetic
    mlp = {"kind": "dense", "ff": 3001}
    if kind == "tupitar":
        layers = [{"type": "latent_attention", "mixer": dict(heads=2, dim=32, vdim=32, kv_rank=40, scale=32 ** -0.5), "mlp": mlp},
                  {"type": "mamba2", "mixer": dict(heads=3, vdim=32, state=32, groups=1, norm_groups=1, conv=4), "mlp": mlp}]
        cfg = {"architecture": "Tupitar", "vocab": 80, "width": E, "max_positions": 64, "embedding": {"scale": 1.0}, "norm": {"eps": 1e-6}, "layers": layers}
    else:
        left = dict(heads=2, kv_heads=1, dim=32, vdim=32, scale=32 ** -0.5, softcap=30.0, bias_max=512, mask=dict(size=16, keep_first=2))
        layers = [{"type": "parallel", "mixer": dict(left=left, left_scale=0.5, right=dict(heads=2, dim=32, vdim=32, tau=16.0), right_scale=0.8), "mlp": dict(mlp, limit=7.0)}] * 2
        cfg = {"architecture": "Mafurax", "vocab": 80, "width": E, "logit_scale": E ** -0.5, "norm": {"eps": 1e-6}, "layers": layers}
    synthetic.write_synthetic_stack(str(tmp_path / "m"), cfg)
    m = bamd.Model(str(tmp_path / "m"), dtype=dtype)
    a, b = bamd.Context(m, 64, 1), bamd.Context(m, 64, 1)
    t = np.random.default_rng(E).integers(0, 80, 9).astype(np.int32)
    whole = a.decode_batch([(0, t, list(range(9)))])
    each = np.concatenate([b.decode_batch([(0, t[i:i + 1], [0])]) for i in range(9)])
    near(each, whole, dtype, 2.0)                                  # (either is off by its own rounding)
    a.close(); b.close(); m.close()


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("F,rows,limit", [(1, 1, 1.0), (40, 3, 0.5), (333, 2, 2.0), (3000, 2, 7.0)])
def test_clamped_glu(bamd, dtype, F, rows, limit):
    """values inside, at and far beyond the limits, on both sides"""
    r = np.random.default_rng(F)
    g, u = r.standard_normal((rows, F)) * 3, r.standard_normal((rows, F)) * 3
    g.flat[:5], u.flat[:5] = [limit, 100, -100, -limit, 0][:g.size], [100, -100, limit, -1, -limit][:u.size]
    got, want = bamd.op_clamped_glu(g, u, limit, dtype), so.clamped_glu(g, u, limit)
    assert np.abs(got - want).max() < (1e-5 if dtype == "float32" else 0.005) * (1 + np.abs(want).max())


# ---- attention ---------------------------------------------------------------------------------------------------------------------------------------------
@functools.lru_cache(None)
def seen_keys(n, size, keep_first):
    return [[j for j in range(i + 1) if so.visible(i, j, {"size": size, "keep_first": keep_first})] for i in range(n)]


def plain(a, T):
    """queries at the last T positions of the keys and values"""
    q, k, v = (np.asarray(a[x], np.float64) for x in "qkv")
    H, G = q.shape[1], k.shape[1]
    if a["past_k"] is not None:
        k, v = np.concatenate([a["past_k"], np.stack([[so.rms(x, a["eps"]) for x in row] for row in k]) if a["unit"] else k]), np.concatenate([a["past_v"], v])
    elif a["unit"]:
        k = np.stack([[so.rms(x, a["eps"]) for x in row] for row in k])
    n = len(k)
    out = np.zeros((T, H, v.shape[2]))
    bucket = None if a["rel"] is None else np.array([so.distance_bucket(x, len(a["rel"]), a["bias_max"]) for x in range(n)])
    for t in range(T):
        i = n - T + t
        seen = np.array(seen_keys(n, a["window"], a["keep"])[i])
        for h in range(H):
            qh = so.rms(q[t, h], a["eps"]) if a["unit"] else q[t, h]
            s = k[seen, h // (H // G)] @ qh * a["scale"]
            if a["cap"]:
                s = so.softcap(s, a["cap"])
            bias = 0 * s if a["rel"] is None else a["rel"][bucket[i - seen], h]
            out[t, h] = so.biased_softmax(s, bias) @ v[seen, h // (H // G)] * (so.sigmoid(a["gate"][t, h]) if a["gate"] is not None else 1) * a.get("out_scale", 1.0)
    return out


def case(dtype, H, G, d, dv, T, pos0, window, keep, rows=8, top=60, cap=8.0, unit=True, seed=0):
    """the keys in front as a cache of that type holds them"""
    r, rd = np.random.default_rng(seed + H * d + T + pos0 + window), rounder(dtype)
    k, v = r.standard_normal((pos0 + T, G, d)), rd(r.standard_normal((pos0 + T, G, dv)))
    past = rd(np.stack([[so.rms(x, 1e-5) for x in row] for row in k[:pos0]])) if pos0 else None
    return dict(q=rd(r.standard_normal((T, H, d))), k=rd(k[pos0:]), v=v[pos0:], gate=r.standard_normal((T, H)).astype(np.float32), past_k=past, past_v=v[:pos0] if pos0 else None, scale=2.0 / np.sqrt(d), cap=cap, eps=1e-5,
                unit=unit, rel=r.standard_normal((rows, H)).astype(np.float32) if rows else None, bias_max=top, window=window, keep=keep)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("H,G,d,dv", [(1, 1, 8, 8), (6, 2, 24, 40), (3, 3, 33, 12), (34, 2, 16, 32), (4, 1, 72, 130), (2, 2, 128, 64), (2, 1, 200, 16), (8, 4, 1, 3)])
@pytest.mark.parametrize("T,pos0,window,keep", [(1, 0, 5, 2), (3, 0, 1, 0), (130, 0, 20, 3), (200, 0, 64, 65), (2, 63, 30, 1), (2, 64, 1000, 0), (70, 130, 65, 5), (1, 63, 10, 3), (1, 64, 64, 64), (1, 300, 63, 70), (1, 500, 1 << 20, 0)])
def test_window_attention(bamd, dtype, H, G, d, dv, T, pos0, window, keep):
    a = case(dtype, H, G, d, dv, T, pos0, window, keep)
    want = plain(a, T).reshape(T, -1)
    for splits in (0, 1, 2, 7) if T == 1 else (0,):
        near(bamd.op_kv_attention(dtype=dtype, splits=splits, **a).reshape(T, -1), want, dtype)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("H,G,d,dv", [(1, 1, 8, 8), (6, 2, 24, 40), (34, 2, 16, 32), (4, 4, 72, 128), (8, 2, 128, 64)])
@pytest.mark.parametrize("pos0,window,keep", [(0, 5, 2), (1, 1, 0), (31, 100, 0), (63, 10, 3), (64, 64, 64), (255, 1 << 20, 0), (300, 63, 70), (513, 1 << 20, 0), (900, 700, 4)])
def test_window_attention_step_in_one_launch(bamd, dtype, H, G, d, dv, pos0, window, keep):
    """no key but the row's own, fewer half pages than waves, as many, more, and a share of them empty; groups of one, three, four and seventeen heads"""
    a = case(dtype, H, G, d, dv, 1, pos0, window, keep)
    near(bamd.op_kv_attention(dtype=dtype, splits=-1, out_scale=-0.7, **a).reshape(1, -1), -0.7 * plain(a, 1).reshape(1, -1), dtype)
    a["gate"] = None
    near(bamd.op_kv_attention(dtype=dtype, splits=-1, **a).reshape(1, -1), plain(a, 1).reshape(1, -1), dtype)


@pytest.mark.parametrize("H,G,d,T,window", [(128, 8, 24, 257, 100), (128, 32, 24, 512, 1000), (128, 4, 24, 513, 70), (85, 5, 40, 700, 130)])
def test_window_attention_in_paired_blocks(bamd, H, G, d, T, window):
    """tiles of 128 queries: one block per CU and a part of a second, two, two and a part of a third, and heads that do not divide the CUs"""
    a = case("bfloat16", H, G, d, d, T, 0, window, 3)
    unit = lambda x: x / np.sqrt((x.astype(np.float64) ** 2).mean(-1, keepdims=True) + a["eps"])
    q, k, i, j = unit(a["q"]), unit(a["k"]), np.arange(T)[:, None], np.arange(T)[None]
    bucket = np.array([so.distance_bucket(x, len(a["rel"]), a["bias_max"]) for x in range(T)])[np.maximum(i - j, 0)]
    want = np.zeros((T, H, d))
    for h in range(H):
        s = so.softcap(q[:, h] @ k[:, h // (H // G)].T * a["scale"], a["cap"]) + a["rel"][bucket, h]
        s = np.where((j > i) | ((i - j >= window) & (j >= 3)), -np.inf, s)
        w = np.exp(s - s.max(-1, keepdims=True))
        want[:, h] = w / w.sum(-1, keepdims=True) @ a["v"][:, h // (H // G)] * so.sigmoid(a["gate"][:, h])[:, None]
    near(bamd.op_kv_attention(dtype="bfloat16", splits=0, **a).reshape(T, -1), want.reshape(T, -1), "bfloat16")


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("splits", [0, 3])
def test_every_part_may_be_absent(bamd, dtype, splits):
    """no unit norm, no cap, no bias, no gate; an output scale"""
    base = case(dtype, 4, 2, 24, 24, 1, 150, 40, 3)
    for change in (dict(unit=False), dict(cap=0.0), dict(rel=None), dict(gate=None), dict(unit=False, cap=0.0, rel=None, gate=None), dict(out_scale=-1.7), dict(gate=np.array([[-30, 0, 2, 30.]], np.float32))):
        a = dict(base, **change)
        want, got = plain(a, 1), bamd.op_kv_attention(dtype=dtype, splits=splits, **a)
        live = np.abs(want).max(-1) > 1e-6
        near(got[live], want[live], dtype)
        assert np.abs(got[~live]).max(initial=0) < 1e-6


def pointed(dtype, n, pos0, window, keep, key, cap=40.0, d=24):
    """every query asks for one key: its score is far above the others' """
    a = case(dtype, 2, 1, d, 40, n, 0, window, keep, rows=6, top=90, cap=cap, seed=3)
    k = np.stack([so.rms(x[0], 1e-5) for x in a["k"]])
    rd = rounder(dtype)
    a["q"] = rd(np.repeat(np.repeat(k[key][None, None], n, 0), 2, 1))[pos0:]
    a["past_k"], a["past_v"] = (rd(k[:pos0])[:, None], a["v"][:pos0]) if pos0 else (None, None)
    a.update(k=a["k"][pos0:], v=a["v"][pos0:], gate=a["gate"][pos0:], scale=22.0 / d)
    return a


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("window,keep", [(1, 1), (64, 0), (65, 5), (63, 64), (100, 65), (128, 66), (31, 0)])
def test_one_key_stands_out_in_prompts(bamd, dtype, window, keep):
    """first tokens, page borders, far away: just inside and just outside the window and the kept tokens for the queries behind it"""
    n = 300
    for pos0 in (0, 129, 250):
        for key in sorted({0, keep - 1, keep, 62, 63, 64, 65, 127, 128, 191, 192, 250, 256, 298} - {-1}):
            a = pointed(dtype, n, pos0, window, keep, key)
            near(bamd.op_kv_attention(dtype=dtype, **a).reshape(n - pos0, -1), plain(a, n - pos0).reshape(n - pos0, -1), dtype, 3)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("window,keep", [(1, 0), (1, 1), (64, 0), (65, 5), (63, 64), (100, 65), (300, 3)])
def test_one_key_stands_out_in_decoding(bamd, dtype, window, keep):
    for last in (64, 65, 127, 128, 200, 255, 256):
        keys = {0, keep - 1, keep, last, last - 1, last - window + 1, last - window, 63, 64}
        for key in sorted(k for k in keys if 0 <= k <= last):
            a = pointed(dtype, last + 1, last, window, keep, key)
            want = plain(a, 1).reshape(1, -1)
            for splits in (1, 4):
                near(bamd.op_kv_attention(dtype=dtype, splits=splits, **a).reshape(1, -1), want, dtype, 3)


@pytest.mark.parametrize("rows,top", [(2, 2), (2, 9), (6, 90), (8, 5), (32, 200), (5, 40)])
def test_bias_of_every_distance(bamd, rows, top):
    """equal scores: the weights are the biases alone; rows far apart, so that a neighbouring row would show"""
    n, H = 260, 3
    a = case("float32", H, 1, 8, 250, n, 0, 1 << 20, 0, rows=rows, top=top)
    a.update(q=np.zeros((n, H, 8), np.float32), gate=None, v=np.concatenate([np.eye(250), np.zeros((10, 250))])[:, None].astype(np.float32), rel=(a["rel"] * 2).astype(np.float32))
    got = bamd.op_kv_attention(dtype="float32", **a)
    want = plain(a, n)
    assert np.abs(got - want).max() < 2e-5
    last = dict(a, q=a["q"][-1:], k=a["k"][-1:], v=a["v"][-1:], past_k=np.stack([[so.rms(x, 1e-5) for x in row] for row in a["k"][:-1]]), past_v=a["v"][:-1])
    assert np.abs(bamd.op_kv_attention(dtype="float32", splits=2, **last) - want[-1:]).max() < 2e-5


@pytest.mark.parametrize("dtype", DTYPES)
def test_scores_at_the_cap(bamd, dtype):
    """raw scores from nothing to a hundred times the cap"""
    for cap in (0.5, 5.0, 50.0):
        a = case(dtype, 3, 1, 16, 24, 80, 0, 1 << 20, 0, cap=cap)
        for scale in (1e-4, 0.1, 2.0, 40.0):
            a["scale"] = scale
            if dtype == "bfloat16" and scale > 1 and cap > 5:
                continue                                 # rounded operands decide which key wins
            near(bamd.op_kv_attention(dtype=dtype, **a).reshape(80, -1), plain(a, 80).reshape(80, -1), dtype, 2)


# ---- gated linear attention --------------------------------------------------------------------------------------------------------------------------------
def gla_case(H, d, dv, R, T, seed):
    r, f = np.random.default_rng(seed), lambda a: np.asarray(a, np.float32)
    return dict(q=f(r.standard_normal((T, H, d))), k=f(r.standard_normal((T, H, d))), v=f(r.standard_normal((T, H, dv))), gate=f(r.standard_normal((T, H, dv))), low=f(r.standard_normal((T, R))),
                a2=so.f32_to_bf16(r.standard_normal((H * d, R)) / np.sqrt(R)), a2b=f(r.uniform(-6, 9, H * d)), norm=f(1 + 0.3 * r.standard_normal(dv)), tau=8.0, q_scale=d ** -0.5, eps=1e-5)


def plain_gla(a, S, t0, t1):
    H, d = a["q"].shape[1:]
    ys, outs = [], []
    for t in range(t0, t1):
        al = so.gla_decay(so.bf16_to_f32(a["a2"]).astype(np.float64) @ a["low"][t] + a["a2b"], a["tau"]).reshape(H, d)
        y = np.zeros(a["v"].shape[1:])
        for h in range(H):
            S[h], y[h] = so.gla_step(S[h], al[h], a["k"][t, h].astype(np.float64), a["v"][t, h].astype(np.float64), a["q"][t, h] * a["q_scale"])
        ys.append(y)
        outs.append(np.stack([so.rms(y[h], a["eps"]) * a["norm"] * so.silu(a["gate"][t, h].astype(np.float64)) for h in range(H)]))
    return np.array(ys), np.array(outs), S


def part(a, t0, t1):
    return dict(a, **{k: a[k][t0:t1] for k in ("q", "k", "v", "gate", "low")})


@pytest.mark.parametrize("H,d,dv,R", [(1, 1, 1, 1), (3, 10, 14, 5), (5, 17, 33, 16), (2, 64, 64, 3), (2, 130, 70, 8), (1, 256, 20, 40), (40, 24, 16, 2), (1, 4, 200, 1)])
def test_gated_linear(bamd, H, d, dv, R):
    """portions from one token up, the state handed from portion to portion, channels that forget at once and channels that keep"""
    a = gla_case(H, d, dv, R, 75, H * d + dv)
    S, pos = np.zeros((H, d, dv)), 0
    gs = np.full((H, d, dv), 7, np.float32)               # what a fresh sequence finds in its place must not matter
    for n in (1, 1, 2, 7, 8, 9, 15, 32):
        y, out, S = plain_gla(a, S, pos, pos + n)
        gy, go, gs = bamd.op_gated_linear(pos0=pos, state=gs, dtype="float32", **part(a, pos, pos + n))
        assert rel(gy, y) < 1e-5 and rel(gs, S) < 1e-5, pos
        assert np.abs(go - out).max() < (3e-4 if dv < 4 else 1e-4) * (1 + np.abs(out).max()), pos      # (a norm over few columns magnifies)
        pos += n


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("H,d,dv,R", [(1, 1, 1, 1), (3, 10, 14, 5), (2, 64, 64, 3), (5, 66, 60, 16), (2, 60, 65, 17), (3, 128, 128, 16), (40, 24, 16, 2)])
def test_gated_linear_step_in_one_launch(bamd, H, d, dv, R, dtype):
    """a fresh state, then one that tokens left: the state's bits are those of two launches"""
    a = gla_case(H, d, dv, R, 4, H * d + dv)
    S, gs = np.zeros((H, d, dv)), np.full((H, d, dv), 7, np.float32)
    for t in range(4):
        _, out, S = plain_gla(a, S, t, t + 1)
        _, _, two = bamd.op_gated_linear(pos0=t, state=gs, dtype=dtype, **part(a, t, t + 1))
        _, go, gs = bamd.op_gated_linear(pos0=t, state=gs, dtype=dtype, out_scale=-0.6, segment=-1, **part(a, t, t + 1))
        assert np.array_equal(gs.view(np.uint32), two.view(np.uint32)) and rel(gs, S) < 1e-5
        e = np.abs(go + 0.6 * out)
        assert (e <= (3e-4 if dv < 4 else 1e-4) * (1 + np.abs(out).max()) + (2.0 ** -8 if dtype == "bfloat16" else 0) * np.abs(out)).all(), t      # (as above, and the result's own rounding)


@pytest.mark.parametrize("H,d,dv", [(2, 20, 24), (1, 130, 70), (3, 64, 16)])
@pytest.mark.parametrize("segment", [8, 16, 40, 104])
def test_gated_linear_in_segments(bamd, H, d, dv, segment):
    """a prompt scanned in segments gives what one scan gives, from a fresh state and from one that earlier tokens left"""
    a = gla_case(H, d, dv, 4, 230, 9)
    S = np.zeros((H, d, dv))
    gs = np.full((H, d, dv), 5, np.float32)
    for t0, t1 in ((0, 107), (107, 230)):
        y, out, S = plain_gla(a, S, t0, t1)
        gy, go, gs = bamd.op_gated_linear(pos0=t0, state=gs, dtype="float32", segment=segment, **part(a, t0, t1))
        assert rel(gy, y) < 1e-5 and rel(gs, S) < 1e-5
        for rows, ref in zip(gy, y):
            assert rel(rows, ref) < 1e-4


def test_a_long_memory(bamd):
    """decays next to one and strongly different ones per channel: a key of the first token is still read hundreds of tokens later, and only through the channels that keep it"""
    H, d, dv, T = 1, 8, 12, 400
    a = gla_case(H, d, dv, 1, T, 4)
    a["low"][:], a["a2b"][:] = 0, [14, 14, 14, 14, -8, -8, -8, -8]
    a["k"][1:] = 0; a["k"][0] = 1
    a["q"][:] = 0; a["q"][::2, :, :4] = 1; a["q"][1::2, :, 4:] = 1
    y, _, S = plain_gla(a, np.zeros((H, d, dv)), 0, T)
    for segment in (0, 64):
        gy, _, gs = bamd.op_gated_linear(pos0=0, state=np.zeros((H, d, dv)), dtype="float32", segment=segment, **a)
        assert rel(gy[::2], y[::2]) < 1e-4 and np.abs(gy[101::2]).max() < 1e-6 and rel(gs, S) < 1e-4


@pytest.mark.parametrize("dtype", DTYPES)
def test_head_norm_and_gate(bamd, dtype):
    a = gla_case(3, 12, 37, 2, 20, 8)
    _, out, _ = plain_gla(a, np.zeros((3, 12, 37)), 0, 20)
    _, go, _ = bamd.op_gated_linear(pos0=0, state=np.zeros((3, 12, 37)), dtype=dtype, out_scale=-0.6, **a)
    near(go.reshape(20, -1), -0.6 * out.reshape(20, -1), dtype)
    gy, go, _ = bamd.op_gated_linear(pos0=0, state=np.zeros((3, 12, 37)), dtype=dtype, **dict(a, gate=None))
    near(go, np.stack([[so.rms(y, 1e-5) * a["norm"] for y in row] for row in gy.astype(np.float64)]), dtype)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("H,d,dv", [(6, 64, 65), (7, 20, 30), (2, 100, 128)])
@pytest.mark.parametrize("rows", [1, 3, 9])
def test_steps_that_outgrow_one_launch(bamd, dtype, H, d, dv, rows, tmp_path):
    """sequences of different lengths around 224 and 448 positions, the most that one launch takes: the same graph key before, another behind"""
    cfg = stack_cases.mafurax(64, 97, [stack_cases.parallel(stack_cases.attend(4, 2, 24, 20, 0.4, 6.0, 50, 1 << 20, 0), 0.7, (H, d, dv, 8.0), 1.3, ff=80, limit=0.8)])
    case = Case(str(tmp_path / "m"), cfg, 3, dict(rel=8, rank=5))
    m = bamd.Model(case.folder, dtype=dtype)
    c = bamd.Context(m, 64 * 8 * rows, rows)
    for most in (224, 448):
        t = [tokens(cfg, most + 6, 30 + i) for i in range(min(rows, 3))]
        want = [case.logits(x) for x in t]
        at = [most - 4 - 30 * (s % 3) for s in range(rows)]
        for s in range(rows): c.seq_free(s)
        c.decode_batch([(s, t[s % 3][:at[s]], [at[s] - 1]) for s in range(rows)])
        for _ in range(8):
            got = c.decode_batch([(s, [t[s % 3][at[s]]], [0]) for s in range(rows)])
            near(got, np.stack([want[s % 3][at[s]] for s in range(rows)]), dtype)
            at = [a + 1 for a in at]
    c.close(); m.close()


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("H,d,dv,steps", [(3, 130, 70, (2, 21, 22, 42, 43, 64, 65)), (6, 64, 65, (5, 11, 22)), (7, 20, 30, (19, 37)), (2, 100, 9, (6, 64))])
def test_decoding_rows_that_share_launches(bamd, dtype, H, d, dv, steps, tmp_path):
    """a step of that many short sequences: one launch up to 64 rows (48 in 32-bit) and 128 channels, two beyond the channels, the branches' own launches beyond the rows"""
    cfg = stack_cases.mafurax(64, 97, [stack_cases.parallel(stack_cases.attend(4, 2, 24, 20, 0.4, 6.0, 50, 19, 3), 0.7, (H, d, dv, 8.0), 1.3, ff=80, limit=0.8)])
    case = Case(str(tmp_path / "m"), cfg, 3, dict(rel=8, rank=5))
    m = bamd.Model(case.folder, dtype=dtype)
    c = bamd.Context(m, 64 * max(steps), max(steps))
    t = [tokens(cfg, 7 + len(steps), 30 + i) for i in range(3)]
    want = [case.logits(x) for x in t]
    c.decode_batch([(s, t[s % 3][:5 + s % 3], [4 + s % 3]) for s in range(max(steps))])
    at = [5 + s % 3 for s in range(max(steps))]
    for n in steps:
        got = c.decode_batch([(s, [t[s % 3][at[s]]], [0]) for s in range(n)])
        near(got, np.stack([want[s % 3][at[s]] for s in range(n)]), dtype)
        for s in range(n): at[s] += 1
    c.close(); m.close()


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("H,d,dv,steps", [(3, 130, 70, (2, 22, 43, 64, 65)), (6, 64, 65, (5, 11, 22)), (7, 20, 30, (19, 37)), (2, 100, 9, (6, 64)), (16, 128, 128, (3, 6, 8))])
def test_decoding_long_rows_that_share_launches(bamd, dtype, H, d, dv, steps, tmp_path):
    """the same behind 452 positions and more, which is two launches whatever the rows: the recurrence takes 16, 32 or 64 columns a block, up to 64, 128 and more channels.  (The oracle with every product's
    operands rounded to bfloat16 moves no row of these by more than 0.0053.)"""
    cfg = stack_cases.mafurax(64, 97, [stack_cases.parallel(stack_cases.attend(4, 2, 24, 20, 0.4, 6.0, 50, 1 << 20, 0), 0.7, (H, d, dv, 8.0), 1.3, ff=80, limit=0.8)])
    case = Case(str(tmp_path / "m"), cfg, 3, dict(rel=8, rank=5))
    m = bamd.Model(case.folder, dtype=dtype)
    c = bamd.Context(m, 512 * max(steps), max(steps))
    t = [tokens(cfg, 454 + len(steps), 30 + i) for i in range(3)]
    want = [case.logits(x) for x in t]
    c.decode_batch([(s, t[s % 3][:452 + s % 3], [451 + s % 3]) for s in range(max(steps))])
    at = [452 + s % 3 for s in range(max(steps))]
    for n in steps:
        got = c.decode_batch([(s, [t[s % 3][at[s]]], [0]) for s in range(n)])
        near(got, np.stack([want[s % 3][at[s]] for s in range(n)]), dtype)
        for s in range(n): at[s] += 1
    c.close(); m.close()
