"""Calls under graph capture on a context that has not run them before: what
needs no workspace, or no more than an earlier call of the context left, can be
captured without a run of its own, and each replay gives the eager result."""
import contextlib

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@contextlib.contextmanager
def fresh_context():
    import ferrum_hip

    ctx = ferrum_hip.Context(0)
    try:
        yield ctx
    finally:
        ctx.sync()
        ctx.close()


def replays_equal_eager(ctx, call, out):
    """Capture `call` (which fills `out`) before it has run on `ctx`; three
    replays with eager runs between them, every result the same bits."""
    import torch

    g, s = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    torch.cuda.synchronize()
    try:
        with torch.cuda.graph(g, stream=s):
            ctx.set_stream(torch.cuda.current_stream().cuda_stream)
            call()
    finally:
        ctx.set_stream(None)
    seen = []
    for _ in range(3):
        out.fill_(float("nan"))
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        seen.append(out.cpu().numpy().view(np.uint32).copy())
        out.fill_(float("nan"))
        torch.cuda.synchronize()
        call()
        ctx.sync()
        seen.append(out.cpu().numpy().view(np.uint32).copy())
    assert np.isfinite(seen[0].view(np.float32)).all()
    assert all(np.array_equal(v, seen[0]) for v in seen)


def on_device(*arrays):
    import torch

    return [torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in arrays]


# SwiGLU of a narrow model: up to 24 blocks of K it splits no K, and needs no
# workspace.
@pytest.mark.parametrize("m,ffn,k", [(3, 2048, 768), (32, 2048, 768), (17, 512, 288), (32, 3072, 768)])
def test_swiglu_up_to_24_blocks_needs_no_workspace(orc, m, ffn, k):
    import torch

    import ferrum_hip

    rng = np.random.default_rng(m + ffn)
    with fresh_context() as ctx:
        w = ferrum_hip.Q8_0Weight.upload(ctx, orc.quantize_weight(2 * ffn, k, ffn, 0.05), 2 * ffn, k)
        x = rng.standard_normal((m, k)).astype(np.float32)
        grp = x.reshape(m, k // 32, 32)
        stats = np.stack([grp.mean(2), ((grp - grp.mean(2, keepdims=True)) ** 2).sum(2)], axis=2).astype(np.float32)
        dx, st, gam = on_device(x, stats, rng.standard_normal(k).astype(np.float32))
        y = torch.empty((m, ffn), device="cuda")
        replays_equal_eager(ctx, lambda: ferrum_hip.linear_normed_async(
            ctx, w, dx, m, k, st, gam, None, 1e-6, True, None, 0, y, ferrum_hip.ACT_SWIGLU32), y)
        w.free()


# After one call at the longest prompt, any shorter one over as many inputs can be
# captured, whichever kernel each takes: K splits (768 x 3072 at 97 rows) after
# a call that asks for no workspace (511 rows) or for fewer partials (127), the
# 128 x 128 tiles' panel (4096 x 1024 at 1050 rows, 50257 x 64 at 65) after
# smaller needs.
@pytest.mark.parametrize("n,k,longest,m", [(768, 3072, 511, 97), (1344, 3072, 127, 96), (4096, 1024, 2100, 1050),
                                           (50257, 64, 300, 65), (768, 3072, 511, 511), (130, 96, 200, 70)])
def test_shorter_prompts_after_the_longest(orc, n, k, longest, m):
    import torch

    import ferrum_hip

    rng = np.random.default_rng(n + m)
    with fresh_context() as ctx:
        w = ferrum_hip.Q8_0Weight.upload(ctx, orc.quantize_weight(n, k, m, 0.05), n, k)
        x, b = on_device(rng.standard_normal((longest, k)).astype(np.float32),
                         rng.standard_normal(n).astype(np.float32))
        y = torch.empty((longest, n), device="cuda")
        torch.cuda.synchronize()
        ferrum_hip.linear_forward_async(ctx, w, x, longest, k, b, n, y)
        ctx.sync()
        out = torch.empty((m, n), device="cuda")
        replays_equal_eager(ctx, lambda: ferrum_hip.linear_forward_async(ctx, w, x, m, k, b, n, out), out)
        w.free()


# W8A8: after a call of a few outputs at m rows (the block-parallel kernel), one of
# many outputs (the matrix cores, whose panel has whole 64-row tiles) needs no more
# workspace, nor does any of fewer rows.
@pytest.mark.parametrize("numerics", ["W8A8", "W8A8_FAST"])
@pytest.mark.parametrize("m1,m2", [(20, 20), (31, 9), (511, 300)])
def test_w8a8_of_wider_outputs_after_narrow_ones(orc, numerics, m1, m2):
    import torch

    import ferrum_hip

    k, mode, rng = 2048, getattr(ferrum_hip, numerics), np.random.default_rng(m1)
    with fresh_context() as ctx:
        wide = ferrum_hip.Q8_0Weight.upload(ctx, orc.quantize_weight(30000, k, 1, 0.05), 30000, k)
        narrow = ferrum_hip.Q8_0Weight.upload(ctx, orc.quantize_weight(64, k, 2, 0.05), 64, k)
        x, = on_device(rng.standard_normal((m1, k)).astype(np.float32))
        y = torch.empty((m1, 64), device="cuda")
        torch.cuda.synchronize()
        ferrum_hip.linear_forward_async(ctx, narrow, x, m1, k, None, 0, y, mode)
        ctx.sync()
        out = torch.empty((m2, 30000), device="cuda")
        replays_equal_eager(ctx, lambda: ferrum_hip.linear_forward_async(ctx, wide, x, m2, k, None, 0, out, mode), out)
        wide.free()
        narrow.free()


def test_prompt_attention_of_one_row_at_width_32(orc):
    """Head width 32, one row after 700 positions: the vector units, whose partial
    sums need the context's areas. Captured on a context that has none, it runs
    on the matrix cores; either way within 1e-5 of the oracle."""
    import torch

    import ferrum_hip

    d, heads, pos0 = 128, 4, 700
    rng = np.random.default_rng(700)
    qkv = rng.standard_normal((1, 3 * d)).astype(np.float32)
    kc, vc = (rng.standard_normal((pos0 + 1, d)).astype(np.float32) for _ in range(2))
    want = orc.attention_decode(qkv[0], kc.copy(), vc.copy(), heads, pos0)
    with fresh_context() as ctx:
        tq, tk, tv = on_device(qkv, kc, vc)
        out = torch.empty((1, d), device="cuda")

        def call():
            ferrum_hip.attention_prefill_seqs_async(ctx, tq, tk, tv, 0, pos0 + 1, d, heads, pos0, 1, 1, out)

        g, s = torch.cuda.CUDAGraph(), torch.cuda.Stream()
        torch.cuda.synchronize()
        try:
            with torch.cuda.graph(g, stream=s):
                ctx.set_stream(torch.cuda.current_stream().cuda_stream)
                call()
        finally:
            ctx.set_stream(None)
        for run in (g.replay, call, g.replay, call, g.replay):
            out.fill_(float("nan"))
            torch.cuda.synchronize()
            run()
            ctx.sync()
            torch.cuda.synchronize()
            got = out.cpu().numpy()[0]
            assert np.all(np.abs(got - want) <= 1e-5 * np.maximum(1.0, np.abs(want)))
