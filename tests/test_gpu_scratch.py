"""GPU regression tests of the runtime's edge paths: decode over a layer
without cross K/V, device zero fills for empty key sets, per-layer cross
lengths, and context scratch that is sized before graph capture (and refused
during it)."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from gpu_util import dev, host, maxerr, note

pytestmark = pytest.mark.gpu


@pytest.fixture()
def fresh_ctx(wrs):
    c = wrs.Context(0)
    c.use_torch_stream()
    yield c
    c.close()


def test_decode_cross_without_cross_plane_is_zero(wrs, fresh_ctx):
    # An arena created with n_audio_max = 0 has no cross planes at all; the
    # reference returns zeros for t_kv == 0 (attention.rs:93-96).
    note("decode_cross on an arena with n_audio_max = 0")
    H, beams = 4, 5
    arena = wrs.KvArena(2, 1, H, 16, 0, ctx=fresh_ctx)
    q = torch.randn((beams, H * 64), device="cuda")
    out = torch.full((beams, H * 64), float("nan"), device="cuda")
    arena.decode_cross(1, q, out)
    assert np.array_equal(host(out), np.zeros((beams, H * 64), np.float32))
    arena.close()


def test_decode_and_prefill_cross_after_invalidate_are_zero(wrs, fresh_ctx):
    note("decode_cross / prefill_cross after invalidate_cross")
    from wrs_amd import workloads as W
    H, n_audio = 2, 300
    arena = wrs.KvArena(1, 1, H, 16, n_audio, ctx=fresh_ctx)
    k = W.normal((n_audio, H * 64), 1, storage="f16")
    arena.set_cross(0, dev(k), dev(k))
    arena.invalidate_cross()
    assert arena.cross_len(0) == 0
    q = torch.randn((3, H * 64), device="cuda")
    for n in (1, 3):
        out = torch.full((n, H * 64), float("nan"), device="cuda")
        if n == 1:
            arena.decode_cross(0, q[:1], out)
        else:
            arena.prefill_cross(0, q[:n], out)
        assert np.array_equal(host(out), np.zeros((n, H * 64), np.float32)), n
    arena.close()


def test_cross_len_is_per_layer(wrs, fresh_ctx):
    # DecoderKvCache keeps cross K/V per layer (decoder.rs:136-139).
    note("cross_len per layer")
    arena = wrs.KvArena(3, 1, 1, 8, 64, ctx=fresh_ctx)
    rows = np.ones((40, 64), np.float32)
    arena.set_cross(1, rows, rows)
    assert [arena.cross_len(l) for l in range(3)] == [0, 40, 0]
    with pytest.raises(RuntimeError):
        arena.cross_len(3)
    arena.close()


def test_prefill_with_no_keys_zero_fills_strided_rows(wrs, fresh_ctx):
    # t_kv == 0 zero-fills the output (attention.rs:93-96) through a fill
    # kernel; columns outside the heads' [t_q][d_head] blocks stay untouched.
    note("prefill t_kv = 0 zero fill, strided output")
    B, H, T, dh = 2, 3, 5, 64
    row = H * dh + 16
    out = torch.full((B, T, row), 7.0, device="cuda")
    q = torch.randn((B, T, H * dh), device="cuda")
    lq = wrs.token_major(T, H * dh, dh)
    lo = wrs.Layout(T * row, dh, row)
    wrs.prefill(q, q, q, out, batch=B, n_heads=H, t_q=T, t_kv=0, d_head=dh, q_layout=lq,
                kv_layout=lq, out_layout=lo, ctx=fresh_ctx)
    got = host(out)
    assert np.array_equal(got[:, :, :H * dh], np.zeros((B, T, H * dh), np.float32))
    assert np.array_equal(got[:, :, H * dh:], np.full((B, T, 16), 7.0, np.float32))


def _decode_setup(wrs, ctx, W):
    H, n_audio, beams = 4, 1500, 5
    cross = wrs.KvArena(1, 1, H, 448, n_audio, ctx=ctx)
    k = W.normal((n_audio, H * 64), 11, storage="f16")
    v = W.normal((n_audio, H * 64), 12, storage="f16")
    cross.set_cross(0, dev(k), dev(v))
    slots = 5
    selfa = wrs.KvArena(1, slots, H, 448, 0, ctx=ctx)
    ks = W.normal((400, H * 64), 13, storage="f16")
    for s_ in range(slots):
        selfa.append(0, s_, dev(ks[:300 + 20 * s_]), dev(ks[:300 + 20 * s_]))
        selfa.advance(s_, 300 + 20 * s_ - 1)
    q = torch.from_numpy(W.normal((beams, H * 64), 14)).cuda()
    return H, beams, slots, cross, selfa, q


def test_reserved_scratch_allows_graph_capture(wrs, fresh_ctx):
    # Sized before capture, the split-K decode allocates nothing while a graph
    # records it; replays (with eager work between them) match eager calls.
    from wrs_amd import workloads as W
    note("reserve + graph capture of decode_cross / decode_self")
    ctx = fresh_ctx
    H, beams, slots, cross, selfa, q = _decode_setup(wrs, ctx, W)
    ctx.reserve(n_heads=H, decode_rows=slots, decode_keys=1500)
    out_c = torch.zeros((beams, H * 64), device="cuda")
    out_s = torch.zeros((slots, H * 64), device="cuda")
    cross.decode_cross(0, q, out_c)
    selfa.decode_self(0, list(range(slots)), q, out_s)
    ref_c, ref_s = out_c.clone(), out_s.clone()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        ctx.use_torch_stream()
        cross.decode_cross(0, q, out_c)
        selfa.decode_self(0, list(range(slots)), q, out_s)
    ctx.use_torch_stream()
    for rep in range(3):
        out_c.fill_(float("nan"))
        out_s.fill_(float("nan"))
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out_c, ref_c), f"replay {rep}: cross decode differs from eager"
        assert torch.equal(out_s, ref_s), f"replay {rep}: self decode differs from eager"
        # eager work between replays
        cross.decode_cross(0, q * 0.5, out_c)
        torch.cuda.synchronize()
    cross.close()
    selfa.close()


def test_scratch_growth_during_capture_is_refused(wrs, fresh_ctx):
    from wrs_amd import workloads as W
    note("decode_cross during capture without reserved scratch -> WRS_ECAPTURE")
    ctx = fresh_ctx
    H, beams, slots, cross, selfa, q = _decode_setup(wrs, ctx, W)
    out_c = torch.zeros((beams, H * 64), device="cuda")
    g = torch.cuda.CUDAGraph()
    with pytest.raises(RuntimeError, match="reserve"):
        with torch.cuda.graph(g):
            out_c.add_(0.0)  # the graph is not empty when the capture ends
            ctx.use_torch_stream()
            cross.decode_cross(0, q, out_c)
    ctx.use_torch_stream()
    torch.cuda.synchronize()
    # outside capture the same call sizes its scratch and runs
    cross.decode_cross(0, q, out_c)
    ref = np.zeros((beams, H * 64), np.float32)
    torch.cuda.synchronize()
    assert np.isfinite(host(out_c)).all() and maxerr(host(out_c), ref) < 10
    cross.close()
    selfa.close()


def test_split_prefill_under_graph_capture(wrs, fresh_ctx):
    # One whisper-base window (96 blocks of 128 queries, fewer than half the
    # CUs) splits each block over two workgroups through context scratch that
    # the first call outside capture allocates. Captured before that call,
    # the prefill takes the key split instead (no allocation, no error);
    # captured after it, the split blocks replay bit-identically to eager
    # calls, with eager work between the replays.
    from wrs_amd import workloads as W
    note("16-bit prefill of one whisper-base window under graph capture")
    ctx = fresh_ctx
    H, T = 8, 1500
    x = [dev(W.normal((T, H * 64), 40 + i, storage="f16"), torch.float16) for i in range(3)]
    lay = wrs.token_major(T, H * 64, 64)
    out = torch.zeros((T, H * 64), device="cuda")

    def run():
        wrs.prefill(x[0], x[1], x[2], out, batch=1, n_heads=H, t_q=T, t_kv=T, d_head=64,
                    q_layout=lay, kv_layout=lay, out_layout=lay, ctx=ctx)

    g0 = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g0):
        ctx.use_torch_stream()
        run()
    ctx.use_torch_stream()
    out.fill_(float("nan"))
    g0.replay()
    torch.cuda.synchronize()
    before = out.clone()
    run()  # outside capture: allocates the scratch, runs the split blocks
    torch.cuda.synchronize()
    ref = out.clone()
    assert torch.isfinite(ref).all()
    assert maxerr(host(before), host(ref)) < 1e-4, "key split and split blocks disagree"
    g1 = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g1):
        ctx.use_torch_stream()
        run()
    ctx.use_torch_stream()
    for rep in range(3):
        out.fill_(float("nan"))
        g1.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, ref), f"replay {rep}: split prefill differs from eager"
        run()  # eager work between replays
        torch.cuda.synchronize()
        assert torch.equal(out, ref), f"eager call after replay {rep} differs"


def test_f32_workgroup_split_under_graph_capture(wrs, fresh_ctx):
    # flash_attention_2's (64, 1500) x 6 heads shape in f32: each 32-query
    # block's key tiles go to 12 workgroups folded through the same context
    # scratch. Captured before any eager call the launch keeps one workgroup
    # per block (no allocation); captured after, it replays the workgroup
    # split bit-identically to eager calls, with eager work between replays.
    note("f32 prefill (64, 1500) x 6 heads under graph capture")
    ctx = fresh_ctx
    H, TQ, TK = 6, 64, 1500
    g = torch.Generator(device="cuda")
    g.manual_seed(7)
    q = torch.randn((TQ, H * 64), generator=g, device="cuda")
    k = torch.randn((TK, H * 64), generator=g, device="cuda")
    v = torch.randn((TK, H * 64), generator=g, device="cuda")
    lq, lk = wrs.token_major(TQ, H * 64, 64), wrs.token_major(TK, H * 64, 64)
    out = torch.zeros((TQ, H * 64), device="cuda")

    def run():
        wrs.prefill(q, k, v, out, batch=1, n_heads=H, t_q=TQ, t_kv=TK, d_head=64,
                    q_layout=lq, kv_layout=lk, out_layout=lq, ctx=ctx)

    g0 = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g0):
        ctx.use_torch_stream()
        run()
    ctx.use_torch_stream()
    out.fill_(float("nan"))
    g0.replay()
    torch.cuda.synchronize()
    before = out.clone()
    run()  # outside capture: allocates the scratch, runs the workgroup split
    torch.cuda.synchronize()
    ref = out.clone()
    assert torch.isfinite(ref).all()
    assert maxerr(host(before), host(ref)) < 1e-5, "one and twelve workgroups per block disagree"
    g1 = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g1):
        ctx.use_torch_stream()
        run()
    ctx.use_torch_stream()
    for rep in range(3):
        out.fill_(float("nan"))
        g1.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, ref), f"replay {rep}: f32 workgroup split differs from eager"
        run()
        torch.cuda.synchronize()
        assert torch.equal(out, ref), f"eager call after replay {rep} differs"


def _capture(ctx, fn):
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        ctx.use_torch_stream()
        fn()
    ctx.use_torch_stream()
    return g


@pytest.mark.parametrize("call,rows,n_in", [
    (call, rows, n_in) for call in ("linear", "group", "fused", "cross_proj")
    for rows, n_in in ((9, 64), (37, 1280), (37, 5120), (448, 1280))
    if call != "cross_proj" or n_in <= 1280])
def test_reserved_projection_allows_graph_capture(wrs, fresh_ctx, call, rows, n_in):
    # A context that has reserved the rows records their projection as its first
    # call: the split rows (and the k split's partials) fit what was reserved.
    note(f"reserve + graph capture of {call} rows={rows} n_in={n_in}")
    gen = torch.Generator(device="cuda")
    gen.manual_seed(rows + n_in)
    n_out = n_in if call == "cross_proj" else 128
    x = torch.randn((rows, n_in), generator=gen, device="cuda")
    ws = [(torch.randn((n_out, n_in), generator=gen, device="cuda") / n_in ** 0.5).half()
          for _ in range(2)]
    bs = [torch.randn(n_out, generator=gen, device="cuda") for _ in range(2)]
    ln = (torch.rand(n_in, generator=gen, device="cuda"),
          torch.randn(n_in, generator=gen, device="cuda"), 1e-5)
    out = torch.zeros((2, rows, n_out), device="cuda")
    q = torch.randn((1, n_out), generator=gen, device="cuda")

    def setup(ctx):
        arena = None
        if call == "cross_proj":
            arena = wrs.KvArena(1, 1, n_in // 64, 4, rows, ctx=ctx)

        def run():
            if call == "linear":
                wrs.linear(x, ws[0], bs[0], out[0], ctx=ctx)
            elif call == "group":
                wrs.linear_group(x, ws, bs, [out[0], out[1]], ctx=ctx)
            elif call == "fused":
                wrs.linear_fused(x, ws, bs, [out[0], out[1]], ln=ln, act="gelu", ctx=ctx)
            else:
                arena.set_cross_proj(x, [ws[0]], [ws[1]], [bs[1]])
                arena.decode_cross(0, q, out[0, :1])
        return run, arena

    other = wrs.Context(0)
    other.use_torch_stream()
    run, arena = setup(other)
    run()
    torch.cuda.synchronize()
    ref = out.clone()
    assert torch.isfinite(ref).all()
    if arena is not None:
        arena.close()
    other.close()
    ctx = fresh_ctx
    ctx.reserve(linear_tokens=rows, linear_n_in=n_in, n_heads=n_in // 64, decode_rows=1,
                decode_keys=rows)
    run, arena = setup(ctx)
    out.zero_()
    g = _capture(ctx, run)
    for rep in range(3):
        out.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, ref), f"replay {rep}"
        out.zero_()
        run()  # eager work between replays
        torch.cuda.synchronize()
        assert torch.equal(out, ref), f"eager call after replay {rep}"
    if arena is not None:
        arena.close()


def _replays_equal(g, out, ref, eager, n=3):
    """n replays into a cleared `out`, with eager work between them, keep ref's bits."""
    for rep in range(n):
        out.fill_(float("nan"))
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, ref), f"replay {rep}"
        eager()
        torch.cuda.synchronize()


@pytest.mark.parametrize("f32", [False, True])
def test_captured_decode_outlives_exact_calls(wrs, fresh_ctx, f32):
    # A recorded decode keeps its scratch whatever exact (f32) attention its context
    # runs eagerly afterwards: host slices of any size, and f32 arenas of no more
    # scores than before in more rows or slots.
    from wrs_amd import workloads as W
    note(f"captured decode, exact calls, replays; f32={f32}")
    ctx = fresh_ctx
    H, n_audio, beams = 6, 1500, 8
    dt = wrs.WRS_F32 if f32 else wrs.WRS_F16
    arena = wrs.KvArena(1, 1, H, 16, n_audio, ctx=ctx, dtype=dt)
    k, v = (dev(W.normal((n_audio, H * 64), 31 + i, storage="f16")) for i in range(2))
    arena.set_cross(0, k, v)
    q = dev(W.normal((beams, H * 64), 33))
    out = torch.zeros((beams, H * 64), device="cuda")
    if not f32:
        ctx.reserve(n_heads=H, decode_rows=beams, decode_keys=n_audio)
    arena.decode_cross(0, q, out)
    torch.cuda.synchronize()
    ref = out.clone()
    g = _capture(ctx, lambda: arena.decode_cross(0, q, out))

    long = wrs.KvArena(1, 8, H, 704, 0, ctx=ctx, dtype=wrs.WRS_F32)
    rows = torch.randn((700, H * 64), device="cuda")
    for slot in range(8):
        long.append(0, slot, rows, rows)
        long.advance(slot, 600)
    o8 = torch.zeros_like(q)
    prompt = torch.randn((17, H * 64), device="cuda")
    o17 = torch.zeros_like(prompt)
    rng = np.random.default_rng(34)

    def exact():
        long.decode_self(0, list(range(8)), q, o8)  # 8 blocks of rows, 4808 scores a head
        long.prefill_self(0, 3, prompt, o17)        # 3 blocks, 10489 scores a head
        for heads, tokens, keys in ((8, 1, 1500), (6, 100, 600), (20, 40, 1500)):
            d = heads * 64
            hq, ho = (rng.standard_normal(tokens * d).astype(np.float32) for _ in range(2))
            hk, hv = (rng.standard_normal(keys * d).astype(np.float32) for _ in range(2))
            wrs.mha_with_cache(hq, hk, hv, tokens, keys, keys - tokens, heads, d, ho, ctx=ctx)
        junk = [torch.full((n,), -1, dtype=torch.int32, device="cuda")
                for n in (1 << 8, 1 << 12, 1 << 16, 1 << 20)]
        del junk

    exact()
    _replays_equal(g, out, ref, exact)
    long.close()
    arena.close()


@pytest.mark.parametrize("rows", [9, 15, 17, 23])
def test_reserved_cross_rows_allow_graph_capture(wrs, fresh_ctx, rows):
    # Cross-attention rows that are no multiple of a decode group's eight fit the
    # partials reserved for exactly that many rows.
    from wrs_amd import workloads as W
    note(f"reserve + graph capture of {rows} cross rows")
    ctx = fresh_ctx
    H, n_audio = 3, 700
    arena = wrs.KvArena(1, 1, H, 16, n_audio, ctx=ctx)
    k, v = (W.normal((n_audio, H * 64), 21 + i, storage="f16") for i in range(2))
    arena.set_cross(0, dev(k), dev(v))
    q = dev(W.normal((rows, H * 64), 23))
    out = torch.zeros((rows, H * 64), device="cuda")
    ctx.reserve(n_heads=H, decode_rows=rows, decode_keys=n_audio)
    g = _capture(ctx, lambda: arena.prefill_cross(0, q, out))
    arena.prefill_cross(0, q, out)
    torch.cuda.synchronize()
    ref = out.clone()
    qd, kd, vd = (a.astype(np.float64).reshape(-1, H, 64).transpose(1, 0, 2)
                  for a in (host(q), k, v))
    s = qd @ kd.transpose(0, 2, 1) / 8.0
    p = np.exp(s - s.max(-1, keepdims=True))
    want = ((p / p.sum(-1, keepdims=True)) @ vd).transpose(1, 0, 2).reshape(rows, -1)
    assert maxerr(host(ref), want) < 1e-5
    _replays_equal(g, out, ref, lambda: arena.prefill_cross(0, q * 0.5, out))
    arena.close()


@pytest.mark.parametrize("held,rows", [(8, 9), (16, 23), (8, 23)])
def test_captured_decode_outlives_cross_rows(wrs, fresh_ctx, held, rows):
    # Scratch that holds a prompt's whole groups of eight rows serves its last rows
    # too: the call replaces nothing that a recorded decode holds (the first two).
    # One that needs more than is there (the third) is made before the recording.
    from wrs_amd import workloads as W
    note(f"captured decode of {held} rows, {rows} cross rows, replays")
    ctx = fresh_ctx
    H, n_audio = 3, 700
    arena = wrs.KvArena(1, 1, H, 16, n_audio, ctx=ctx)
    k, v = (W.normal((n_audio, H * 64), 41 + i, storage="f16") for i in range(2))
    arena.set_cross(0, dev(k), dev(v))
    q = dev(W.normal((rows, H * 64), 43))
    out = torch.zeros((held, H * 64), device="cuda")
    all_rows = torch.zeros((rows, H * 64), device="cuda")
    ctx.reserve(n_heads=H, decode_rows=held, decode_keys=n_audio)
    if rows - held >= 8:
        arena.prefill_cross(0, q, all_rows)
    arena.prefill_cross(0, q[:held], out)
    torch.cuda.synchronize()
    ref = out.clone()
    g = _capture(ctx, lambda: arena.prefill_cross(0, q[:held], out))
    _replays_equal(g, out, ref, lambda: arena.prefill_cross(0, q, all_rows))
    other = wrs.Context(0)  # no scratch yet: all rows in one launch
    other.use_torch_stream()
    arena2 = wrs.KvArena(1, 1, H, 16, n_audio, ctx=other)
    arena2.set_cross(0, dev(k), dev(v))
    whole = torch.zeros_like(all_rows)
    arena2.prefill_cross(0, q, whole)
    assert maxerr(host(whole), host(all_rows)) < 1e-6
    arena2.close()
    other.close()
    arena.close()


def test_captured_projection_outlives_forced_prefill(wrs, fresh_ctx):
    # A recorded projection that splits k keeps its partials when a forced prefill
    # schedule on a larger grid outgrows the prefill's own.
    from wrs_amd import workloads as W
    note("captured k split, forced prefill schedules, replays")
    ctx = fresh_ctx
    rows, n_in, n_out = 37, 5120, 256
    x = dev(W.normal((rows, n_in), 51))
    w = dev(W.normal((n_out, n_in), 52, sigma=0.02), torch.float16)
    out = torch.zeros((rows, n_out), device="cuda")
    wrs.linear(x, w, None, out, ctx=ctx)
    torch.cuda.synchronize()
    ref = out.clone()
    want = x.double() @ w.double().t()
    assert float((ref.double() - want).abs().max()) < 1e-5 * float(want.abs().max())
    g = _capture(ctx, lambda: wrs.linear(x, w, None, out, ctx=ctx))
    H, T = 20, 1500
    qkv = [dev(W.normal((T, H * 64), 53 + i, storage="f16")) for i in range(3)]
    h16 = [t.half() for t in qkv]
    lay = wrs.token_major(T, H * 64, 64)
    o = torch.zeros((T, H * 64), device="cuda")

    def forced():
        for t, queries, f32_split in ((qkv, 0, 5), (h16, -3, -1), (h16, -2, -1)):
            ctx.set_schedule(queries, f32_split)
            wrs.prefill(t[0], t[1], t[2], o, batch=1, n_heads=H, t_q=T, t_kv=T, d_head=64,
                        q_layout=lay, kv_layout=lay, out_layout=lay, ctx=ctx)
        ctx.set_schedule()

    forced()
    _replays_equal(g, out, ref, forced)


@pytest.mark.parametrize("f32,rows", [(False, 1), (False, 129), (True, 1000), (False, 4_200_001)])
def test_copy_slot_of_any_length(wrs, fresh_ctx, f32, rows):
    # Also planes of more 16 KB pieces than the grid has workgroups for.
    from gpu_util import read_f16, read_f32
    note(f"copy_slot of {rows} rows, f32={f32}")
    arena = wrs.KvArena(1, 2, 1, rows, 0, ctx=fresh_ctx,
                        dtype=wrs.WRS_F32 if f32 else wrs.WRS_F16)
    k = (torch.arange(rows * 64, device="cuda", dtype=torch.float32) % 2039).view(rows, 64)
    v = -k
    arena.append(0, 0, k, v)
    arena.advance(0, rows)
    arena.copy_slot(1, 0)
    assert arena.slot_len(1) == rows
    torch.cuda.synchronize()
    kp, vp, _, _ = arena.plane_pointers()
    read = read_f32 if f32 else read_f16
    n = min(rows * 64, 100_000)
    for at in (0, rows * 64 - n):
        want = host(k.view(-1)[at:at + n])
        assert np.array_equal(read(kp, rows * 64 + at, n), want)
        assert np.array_equal(read(vp, rows * 64 + at, n), -want)
    arena.close()
