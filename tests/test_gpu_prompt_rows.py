"""Prompt rows over the f16 arena (K10): cached self-attention with a causal
offset (decoder.rs:857-891) and cross-attention of more rows than a decode
group (attention.rs:107-243), at the edges of its row blocks, and key steps, against float64 over the f16 cache values."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from gpu_util import dev, host, note

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx(wrs):
    c = wrs.Context(0)
    c.use_torch_stream()
    return c


def _f16(a):
    return a.astype(np.float16).astype(np.float32)


def _attend(q, k, v, heads, pos0=None):
    """Rows and row statistics (max, sum of 2^(s - max)) in float64."""
    qd, kd, vd = (a.astype(np.float64).reshape(a.shape[0], heads, 64).transpose(1, 0, 2)
                  for a in (q, k, v))
    s = (qd @ kd.transpose(0, 2, 1)) * (0.125 * np.log2(np.e))
    if pos0 is not None:
        s = np.where(np.arange(k.shape[0])[None, :] > pos0 + np.arange(q.shape[0])[:, None],
                     -np.inf, s)
    m = s.max(-1, keepdims=True)
    p = np.exp2(s - m)
    out = (p @ vd) / p.sum(-1, keepdims=True)
    return out.transpose(1, 0, 2).reshape(q.shape), m[..., 0], p.sum(-1)


def _bound(q, k, v, heads):
    """Largest error of each output row: its scores err by at most
    (64 2^-24 + 2^-21) max_j |q||k_j| / 8 (a sum of 64 products in f32, operands
    and scaling to 2^-22), so every normalized weight by twice that relative to
    itself, and the weighted sum adds 2^-20 max |v| (exp2, split weights, f32 sums)."""
    qa, ka, va = (np.abs(a.astype(np.float64)).reshape(a.shape[0], heads, 64).transpose(1, 0, 2)
                  for a in (q, k, v))
    ds = (64 * 2.0 ** -24 + 2.0 ** -21) * (qa @ ka.transpose(0, 2, 1)).max(-1) / 8.0
    b = (2.0 * np.expm1(ds) + 2.0 ** -20) * va.max((1, 2))[:, None]  # [head][row]
    return np.repeat(b.T[:, :, None], 64, axis=2).reshape(q.shape)


@pytest.mark.parametrize("heads,rows,keys", [
    (1, 9, 1), (6, 9, 1500), (3, 17, 200), (6, 24, 700), (1, 25, 1), (2, 31, 31), (2, 32, 33), (3, 33, 64), (20, 37, 1500), (20, 128, 1500),
    (6, 65, 511), (6, 64, 513), (1, 25, 4097), (20, 448, 300), (2, 26, 767), (2, 26, 768)])
def test_cross_rows(wrs, ctx, heads, rows, keys):
    note(f"cross rows heads={heads} rows={rows} keys={keys}")
    rng = np.random.default_rng(heads * 1000 + rows + keys)
    d = heads * 64
    k, v = (_f16(rng.standard_normal((keys, d))) for _ in range(2))
    q = rng.standard_normal((rows, d)).astype(np.float32)
    q[0] *= 30.0   # a peaked row
    q[1] *= 1e-30  # a flat one
    q[2] = 0.0
    arena = wrs.KvArena(1, 1, heads, 16, keys + 5, ctx=ctx)
    arena.set_cross(0, k, v)
    out = torch.full((rows + 1, d), float("nan"), device="cuda")
    lse = torch.full((heads * rows * 2 + 2,), float("nan"), device="cuda")
    ref, m, l = _attend(q, k, v, heads)
    tol = _bound(q, k, v, heads)
    arena.prefill_cross(0, dev(q), out[:rows], lse=lse)
    got = host(out)
    assert (np.abs(got[:rows] - ref) <= tol).all()
    assert np.isnan(got[rows]).all()
    st = host(lse)
    assert np.isnan(st[-2:]).all()
    st = st[:-2].reshape(heads, rows, 2).astype(np.float64)
    lg, lr = st[..., 0] + np.log2(st[..., 1]), m + np.log2(l)
    assert np.abs(lg - lr).max() <= 1e-5 * max(1.0, np.abs(lr).max())
    plain = torch.empty((rows, d), device="cuda")
    arena.prefill_cross(0, dev(q), plain)
    assert torch.equal(plain, out[:rows])
    arena.close()


@pytest.mark.parametrize("heads,rows,past", [
    (1, 2, 0), (2, 31, 0), (2, 32, 1), (3, 33, 30), (20, 37, 0), (20, 224, 224), (6, 2, 445),
    (1, 100, 1900), (4, 448, 0)])
def test_cached_self_rows(wrs, ctx, heads, rows, past):
    note(f"self rows heads={heads} rows={rows} past={past}")
    rng = np.random.default_rng(heads * 1000 + rows + past)
    d = heads * 64
    n = past + rows
    k, v = (_f16(rng.standard_normal((n, d))) for _ in range(2))
    buf = torch.zeros(rows * d + 1, device="cuda")
    q = buf[1:].view(rows, d)  # rows that start on any dword
    qh = rng.standard_normal((rows, d)).astype(np.float32)
    qh[-1] *= 30.0
    q.copy_(dev(qh))
    arena = wrs.KvArena(1, 2, heads, n + 3, 0, ctx=ctx)
    if past:
        arena.append(0, 1, k[:past], v[:past])
        arena.advance(1, past)
    arena.append(0, 1, np.ascontiguousarray(k[past:]), np.ascontiguousarray(v[past:]))
    out = torch.full((rows + 1, d), float("nan"), device="cuda")
    ref, _, _ = _attend(qh, k, v, heads, past)
    tol = _bound(qh, k, v, heads)
    arena.prefill_self(0, 1, q, out[:rows])
    got = host(out)
    assert (np.abs(got[:rows] - ref) <= tol).all()
    assert np.isnan(got[rows]).all()
    arena.close()


# The same where rows times heads put cross rows on K10 (more than 104 pairs of eight
# rows and a head; 320 over planes of up to 256 keys; more than 64 groups), at the
# edges of its 32-row blocks and 32-key steps and of the choice of waves.
@pytest.mark.parametrize("heads,rows,keys", [
    (81, 25, 1), (81, 31, 31), (81, 32, 32), (65, 33, 33), (20, 136, 255), (41, 64, 256),
    (29, 25, 257), (29, 32, 511), (23, 33, 513), (29, 31, 767), (23, 40, 768), (20, 48, 1500),
    (8, 128, 1500), (1, 513, 100), (1, 513, 300), (29, 27, 4097)])
def test_cross_rows_of_many_heads(wrs, ctx, heads, rows, keys):
    test_cross_rows(wrs, ctx, heads, rows, keys)


def test_cross_rows_recorded_without_scratch(wrs):
    # Rows that an eager call runs in decode groups are recorded without scratch for
    # those, on K10.
    note("cross rows captured without scratch")
    c = wrs.Context(0)
    c.use_torch_stream()
    heads, rows, keys = 3, 37, 700
    rng = np.random.default_rng(5)
    k, v = (_f16(rng.standard_normal((keys, heads * 64))) for _ in range(2))
    q = rng.standard_normal((rows, heads * 64)).astype(np.float32)
    arena = wrs.KvArena(1, 1, heads, 16, keys, ctx=c)
    arena.set_cross(0, k, v)
    qd, out = dev(q), torch.zeros((rows, heads * 64), device="cuda")
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        c.use_torch_stream()
        arena.prefill_cross(0, qd, out)
    c.use_torch_stream()
    ref, _, _ = _attend(q, k, v, heads)
    tol = _bound(q, k, v, heads)
    for _ in range(3):
        out.fill_(float("nan"))
        g.replay()
        assert (np.abs(host(out) - ref) <= tol).all()
        out.fill_(float("nan"))
        arena.prefill_cross(0, qd, out)
        assert (np.abs(host(out) - ref) <= tol).all()
    arena.close()
    c.close()


@pytest.mark.parametrize("heads,rows,past", [(1, 2, 3582), (1, 2, 3583), (2, 33, 3800),
                                             (16, 32, 3600), (17, 32, 3600), (16, 32, 6218),
                                             (16, 32, 6219)])
def test_cached_self_rows_of_long_caches(wrs, ctx, heads, rows, past):
    # Few blocks over more than 3584 keys: the f32 kernel, its keys dealt over workgroups.
    test_cached_self_rows(wrs, ctx, heads, rows, past)


# Rows whose output lives on weights far below the row's largest: one key, whose V
# row is zero, scores `octaves` powers of two above the others. Only columns 0 (that
# key alone) and 1 (the others alone) of K meet q, so a score is one product.
def _sink(rows, keys, octaves, seed):
    rng = np.random.default_rng(seed)
    k = np.zeros((keys, 64), np.float32)
    k[:, 1] = _f16(rng.uniform(-1, 1, keys))
    k[0] = 0.0
    k[0, 0] = 1.0
    v = _f16(rng.uniform(0.5, 1.5, (keys, 64)))
    v[0] = 0.0
    q = np.zeros((rows, 64), np.float32)
    q[:, 0] = octaves * 8.0 / np.log2(np.e)
    q[:, 1] = rng.uniform(-8, 8, rows)
    return q, k, v


def _sink_tol(ref, octaves, end):
    """Relative error per output: each exponent argument is one product of at most
    octaves + 2 in magnitude (operand split to 2^-22, scaling and product to 2^-24
    each, differences of two of them), every weight the other way round to 2^-22 or
    to half of the parts' end (2^-end of the largest, the weights being down to
    octaves + 2 below it), and a mean of positive values, summed in f32 (2^-20)."""
    arg = 2.0 * (octaves + 2.0) * (2.0 ** -22 + 3.0 * 2.0 ** -24) * np.log(2.0)
    return np.abs(ref) * (arg + 2.0 ** -20 + 2.0 ** -22 + 2.0 ** (octaves + 1 - end))


@pytest.mark.parametrize("octaves", [2, 14, 17, 20, 23, 26, 32])
@pytest.mark.parametrize("keys", [33, 448, 1500])
def test_cross_rows_keep_small_weights(wrs, ctx, octaves, keys):
    note(f"cross rows, one key {octaves} octaves up of {keys}")
    heads = 81  # on K10
    q, k, v = (np.tile(a, (1, heads)) for a in _sink(27, keys, octaves, octaves + keys))
    arena = wrs.KvArena(1, 1, heads, 16, keys, ctx=ctx)
    arena.set_cross(0, k, v)
    out = torch.zeros((27, heads * 64), device="cuda")
    ref, _, _ = _attend(q, k, v, heads)
    arena.prefill_cross(0, dev(q), out)
    assert (np.abs(host(out) - ref) <= _sink_tol(ref, octaves, 39)).all()
    arena.close()


@pytest.mark.parametrize("octaves", [2, 14, 17, 20, 23, 26, 32])
@pytest.mark.parametrize("rows,past", [(2, 31), (33, 415), (40, 1900)])
def test_cached_self_rows_keep_small_weights(wrs, ctx, octaves, rows, past):
    note(f"self rows, one key {octaves} octaves up of {past + rows}")
    n = past + rows
    q, k, v = _sink(rows, n, octaves, octaves + n)
    arena = wrs.KvArena(1, 1, 1, n, 0, ctx=ctx)
    arena.append(0, 0, k[:past], v[:past])
    arena.advance(0, past)
    arena.append(0, 0, np.ascontiguousarray(k[past:]), np.ascontiguousarray(v[past:]))
    out = torch.zeros((rows, 64), device="cuda")
    ref, _, _ = _attend(q, k, v, 1, past)
    arena.prefill_self(0, 0, dev(q), out)
    assert (np.abs(host(out) - ref) <= _sink_tol(ref, octaves, 61)).all()
    arena.close()


@pytest.mark.parametrize("rows,past", [(2, 31), (33, 415)])
def test_cached_self_rows_keep_small_queries(wrs, ctx, rows, past):
    # A query column far above the others that no key answers: the others decide.
    note(f"self rows, one dead query column, {past + rows} keys")
    rng = np.random.default_rng(past)
    n = past + rows
    k, v = (_f16(rng.standard_normal((n, 64))) for _ in range(2))
    k[:, 5] = 0.0
    q = rng.standard_normal((rows, 64)).astype(np.float32)
    arena = wrs.KvArena(1, 1, 1, n, 0, ctx=ctx)
    arena.append(0, 0, k, v)
    arena.advance(0, past)
    out = torch.zeros((rows, 64), device="cuda")
    ref, _, _ = _attend(q, k, v, 1, past)
    tol = _bound(q, k, v, 1)
    q[:, 5] = 2.0 ** 30
    arena.prefill_self(0, 0, dev(q), out)
    assert (np.abs(host(out) - ref) <= tol).all()
    arena.close()


@pytest.mark.parametrize("rows,past", [(2, 0), (33, 3), (40, 1000)])
def test_cached_self_rows_over_infinite_keys(wrs, ctx, rows, past):
    # A key value past f16's range is infinite in the cache. Rows whose score for
    # it is -inf give it no weight, as the f32 arithmetic does; the others are NaN.
    note(f"self rows, an infinite key value, past={past}")
    rng = np.random.default_rng(rows)
    n = past + rows
    k, v = (_f16(rng.standard_normal((n, 64))) for _ in range(2))
    q = rng.standard_normal((rows, 64)).astype(np.float32)
    q[:, 7] = -1.0 - np.abs(q[:, 7])
    q[-1, 7] = 1.5
    k[past, 7] = 1e6
    arena = wrs.KvArena(1, 1, 1, n, 0, ctx=ctx)
    if past:
        arena.append(0, 0, k[:past], v[:past])
        arena.advance(0, past)
    arena.append(0, 0, np.ascontiguousarray(k[past:]), np.ascontiguousarray(v[past:]))
    out = torch.zeros((rows, 64), device="cuda")
    arena.prefill_self(0, 0, dev(q), out)
    got = host(out)
    kz = k.copy()
    kz[past, 7] = 0.0
    qd, kd, vd = (a.astype(np.float64) for a in (q, kz, v))
    s = qd @ kd.T / 8.0
    j, i = np.arange(n)[None, :], np.arange(rows)[:, None]
    s = np.where((j > past + i) | (j == past), -np.inf, s)
    m = s.max(-1, keepdims=True)
    with np.errstate(invalid="ignore"):
        p = np.where(np.isfinite(m), np.exp(s - m), 0.0)
        ref = (p @ vd) / p.sum(-1, keepdims=True)
    seen = np.isfinite(m[:, 0])  # rows with a key besides it
    seen[-1] = False
    assert np.isnan(got[-1]).all()
    tol = _bound(q, kz, v, 1)
    assert (np.abs(got - ref) <= tol)[seen].all()
    arena.close()


@pytest.mark.parametrize("keys", [300, 1500])
@pytest.mark.parametrize("where,value", [("k", 1e6), ("k", -1e6), ("k", float("nan")),
                                         ("q", float("inf")), ("q", float("nan"))])
def test_cross_rows_with_infinite_scores(wrs, ctx, keys, where, value):
    # A key or query that gives a row a NaN score: on K10 the row comes out as the
    # single-row decode has it (zeros; a row whose score is -inf gives that key no
    # weight), and the other rows are untouched.
    note(f"cross rows, {value} in {where}, {keys} keys")
    heads, rows = 29, 27
    rng = np.random.default_rng(keys)
    k, v = (_f16(rng.standard_normal((keys, heads * 64))) for _ in range(2))
    q = rng.standard_normal((rows, heads * 64)).astype(np.float32)
    plain, _, _ = _attend(q, k, v, heads)
    tol = _bound(q, k, v, heads)
    if where == "k":
        k[keys // 2, 7] = value
    else:
        q[5, 7] = value
    arena = wrs.KvArena(1, 1, heads, 16, keys, ctx=ctx)
    arena.set_cross(0, k, v)
    qd, out = dev(q), torch.full((rows, heads * 64), float("nan"), device="cuda")
    arena.prefill_cross(0, qd, out)
    one = torch.zeros((rows, heads * 64), device="cuda")
    for r in range(rows):
        arena.decode_cross(0, qd[r:r + 1].contiguous(), one[r:r + 1])
    got, ref = host(out), host(one)
    hit = np.zeros(got.shape, bool)  # head 0, whose key or query it is
    hit[(slice(None) if where == "k" else 5), :64] = True
    # the same rows are zero; the others lie within tol of the same exact result each
    assert np.array_equal(got[hit] == 0.0, ref[hit] == 0.0)
    assert (np.abs(got - ref) <= 2 * tol)[hit].all()
    assert value == value and where == "k" or (got[hit] == 0.0).all()
    assert (np.abs(got - plain) <= tol)[~hit].all()
    arena.close()
