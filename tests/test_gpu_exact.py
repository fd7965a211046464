"""FH_W8A32_EXACT: the Q8_0 linear bit for bit as ferrum_core computes it.

The reference expands Q8_0 weights to f32 at load and runs ops::linear_forward
(ops.rs:233-256): every output is the products x[p] * w[p][j] added to 0.0 in
ascending p, each product and add rounded, then + bias.  The oracle restates
that (fo_linear_forward over fo_q8_0_to_ferrum_weight; the oracle's own tests
pin it against a numpy sequential sum), and the exact mode must match it in
every bit, including -0.0, infinities and NaN propagation.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def bits_equal(got, want):
    got = np.ascontiguousarray(got, np.float32)
    want = np.ascontiguousarray(want, np.float32)
    assert got.shape == want.shape
    same = got.view(np.uint32) == want.view(np.uint32)
    both_nan = np.isnan(got) & np.isnan(want)
    bad = ~(same | both_nan)
    assert not bad.any(), (f"{bad.sum()} of {bad.size} outputs differ in their bits; first at "
                           f"{np.argwhere(bad)[0].tolist()}: {got[bad][0]!r} vs {want[bad][0]!r}")


def reference(orc, x, raw, n, k, bias):
    return orc.linear_forward(x, orc.q8_0_to_ferrum_weight(raw, n, k), bias)


@pytest.mark.parametrize("m,n,k,with_bias", [
    (1, 768, 768, True), (1, 2304, 768, True), (1, 3072, 768, True), (1, 768, 3072, True),
    (1, 50257, 768, False), (1, 130, 4864, True), (1, 1, 32, True), (1, 65, 224, False),
    (2, 768, 768, True), (3, 100, 416, True), (8, 3072, 768, True), (32, 768, 3072, False),
    (64, 896, 896, True), (2, 20000, 224, True), (1, 16384, 4864, False)])
def test_exact_matches_the_reference_bit_for_bit(fh, orc, m, n, k, with_bias):
    import ferrum_hip

    seed = m * 1009 + n * 31 + k
    raw = orc.quantize_weight(n, k, seed, 0.02)
    x = np.random.default_rng(seed).standard_normal((m, k), dtype=np.float32)
    b = (np.random.default_rng(seed + 1).standard_normal(n, dtype=np.float32) * np.float32(0.1)
         if with_bias else None)
    w = ferrum_hip.Q8_0Weight.upload(fh, raw, n, k)
    got = ferrum_hip.linear_forward(fh, x, w, b, numerics=ferrum_hip.W8A32_EXACT)
    w.free()
    want = reference(orc, x, raw, n, k, b)
    bits_equal(got, want)
    # the restatement straight from GGUF rows agrees too (the same sums)
    bits_equal(got, orc.q8_0_linear(x, raw, n, b))


def test_exact_keeps_signed_zeros_and_specials(fh, orc):
    """0 + (-0) is +0 in the reference's sum; inf and NaN propagate as f32
    arithmetic says (inf - inf is NaN)."""
    import ferrum_hip

    n, k = 70, 96
    raw = orc.quantize_weight(n, k, 5, 0.05)
    x = np.zeros((4, k), np.float32)
    x[0] = -0.0                      # products of -0 and +-w: signed zeros
    x[1, 5] = np.inf                 # one infinite activation
    x[2, 3] = np.nan
    x[3, ::2] = np.float32(3.0e38)   # sums that overflow to +-inf
    x[3, 1::2] = np.float32(-3.0e38)
    w = ferrum_hip.Q8_0Weight.upload(fh, raw, n, k)
    got = ferrum_hip.linear_forward(fh, x, w, None, numerics=ferrum_hip.W8A32_EXACT)
    w.free()
    want = reference(orc, x, raw, n, k, None)
    assert np.signbit(want[0]).sum() == 0, "the reference's sums start at +0"
    bits_equal(got, want)


def test_exact_device_form_and_blocking_form_agree(fh, orc):
    import torch

    import ferrum_hip

    m, n, k = 5, 2304, 768
    raw = orc.quantize_weight(n, k, 77, 0.02)
    x = np.random.default_rng(3).standard_normal((m, k), dtype=np.float32)
    b = np.random.default_rng(4).standard_normal(n, dtype=np.float32)
    w = ferrum_hip.Q8_0Weight.upload(fh, raw, n, k)
    host = ferrum_hip.linear_forward(fh, x, w, b, numerics=ferrum_hip.W8A32_EXACT)
    dx, db = torch.from_numpy(x).cuda(), torch.from_numpy(b).cuda()
    dy = torch.full((m, n), float("nan"), device="cuda")
    torch.cuda.synchronize()
    ferrum_hip.linear_forward_async(fh, w, dx, m, k, db, n, dy, numerics=ferrum_hip.W8A32_EXACT)
    fh.sync()
    w.free()
    bits_equal(dy.cpu().numpy(), host)
    bits_equal(host, reference(orc, x, raw, n, k, b))


def test_exact_and_fast_modes_agree_to_the_rounding_rule(fh, orc):
    """The fast W8A32 mode stays within 1e-5 of the term mass of the exact one."""
    import ferrum_hip

    n, k = 3072, 3072
    raw = orc.quantize_weight(n, k, 9, 0.02)
    x = np.random.default_rng(9).standard_normal((1, k), dtype=np.float32)
    w = ferrum_hip.Q8_0Weight.upload(fh, raw, n, k)
    exact = ferrum_hip.linear_forward(fh, x, w, None, numerics=ferrum_hip.W8A32_EXACT)
    fast = ferrum_hip.linear_forward(fh, x, w, None, numerics=ferrum_hip.W8A32)
    w.free()
    mass = np.abs(x.astype(np.float64)) @ np.abs(orc.q8_0_to_ferrum_weight(raw, n, k).astype(np.float64))
    assert (np.abs(fast.astype(np.float64) - exact) <= 1e-5 * np.maximum(np.abs(exact), mass)).all()


# One row per lane (tm = 1), and two and four, which the launch rule takes as the
# tiles of 16 columns and 16 rows outnumber the CUs, each with a K that ends
# inside a 128-position chunk or a 16-position piece of it, ragged rows and
# columns.
@pytest.mark.parametrize("m,n,k,tm", [(16, 17, 128, 1), (17, 16, 160, 1), (33, 130, 352, 1), (65, 4081, 96, 1),
                                      (130, 4090, 160, 1), (63, 4090, 160, 2), (96, 4081, 352, 2), (125, 4090, 96, 4),
                                      (128, 4081, 288, 4)])
@pytest.mark.parametrize("f32", [False, True])
def test_exact_rows_per_lane_and_ragged_edges(fh, orc, m, n, k, tm, f32):
    import ferrum_hip
    import seq_tiles

    assert seq_tiles.rows_per_lane(16, -(-n // 16), m) == tm

    rng = np.random.default_rng(m + n + k)
    k -= 7 if f32 else 0
    x = rng.standard_normal((m, k), dtype=np.float32)
    x[m // 2, k - 1], x[m - 1, 0], x[0] = np.inf, np.nan, -0.0
    b = rng.standard_normal(n, dtype=np.float32)
    if f32:
        rows = (rng.standard_normal((n, k)) * 0.05).astype(np.float32)
        rows[n - 1, k - 1] = -np.inf
        w, want = ferrum_hip.Q8_0Weight.upload_f32(fh, rows), orc.linear_forward(x, np.ascontiguousarray(rows.T), b)
    else:
        raw = orc.quantize_weight(n, k, m, 0.02)
        w, want = ferrum_hip.Q8_0Weight.upload(fh, raw, n, k), reference(orc, x, raw, n, k, b)
    got = ferrum_hip.linear_forward(fh, x, w, b, numerics=ferrum_hip.W8A32_EXACT)
    w.free()
    bits_equal(got, want)


# The decode form (one row, or a few workgroups per CU): K below, at and past its
# chunks (192 positions for a wide output, 384) and 16-position jobs, an odd and an
# even number of chunks, ragged columns, several rows, and both sides of the limit
# of two workgroups per CU and, from K = 2048, three.
@pytest.mark.parametrize("m,n,k", [(1, 15, 160), (1, 33, 384), (2, 16, 416), (5, 130, 768), (3, 47, 1184),
                                   (64, 126, 160), (65, 126, 160), (96, 125, 2048), (97, 125, 2048),
                                   (1, 8193, 192), (1, 8209, 416), (1, 8209, 608)])
@pytest.mark.parametrize("f32", [0, 5, 15])
def test_exact_few_outputs(fh, orc, m, n, k, f32):
    import ferrum_hip

    rng = np.random.default_rng(m + n + k + f32)
    k -= f32
    x = rng.standard_normal((m, k), dtype=np.float32)
    x[m - 1, k - 1], x[m // 2, 0] = np.inf, -0.0
    b = rng.standard_normal(n, dtype=np.float32) if m != 2 else None
    if f32:
        rows = (rng.standard_normal((n, k)) * 0.05).astype(np.float32)
        rows[n - 1, k - 1] = np.nan
        w, want = ferrum_hip.Q8_0Weight.upload_f32(fh, rows), orc.linear_forward(x, np.ascontiguousarray(rows.T), b)
    else:
        raw = orc.quantize_weight(n, k, m, 0.02)
        w, want = ferrum_hip.Q8_0Weight.upload(fh, raw, n, k), reference(orc, x, raw, n, k, b)
    got = ferrum_hip.linear_forward(fh, x, w, b, numerics=ferrum_hip.W8A32_EXACT)
    w.free()
    bits_equal(got, want)


def test_exact_more_columns_than_one_grid_dimension_holds(fh, orc):
    """2^28 and more outputs: their tiles of 16 columns, 256 threads each, pass
    what one grid dimension can count.  The weight repeats 4093 rows, so the
    outputs repeat the oracle's."""
    import torch

    import ferrum_hip

    n, k, period = (1 << 28) + 23, 32, 4093
    raw = orc.quantize_weight(period, k, 5, 0.05)
    x = np.random.default_rng(28).standard_normal((1, k), dtype=np.float32)
    want = torch.from_numpy(reference(orc, x, raw, period, k, None)).cuda().ravel()
    rows = torch.from_numpy(np.ascontiguousarray(raw).view(np.uint8).reshape(period, 34)).cuda()
    wide = rows.repeat(n // period + 1, 1)[:n].contiguous()
    torch.cuda.synchronize()
    w = ferrum_hip.Q8_0Weight.upload_device(fh, wide, n, k)
    fh.sync()
    del wide
    y = torch.full((n,), float("nan"), device="cuda")
    dx = torch.from_numpy(x).cuda()
    torch.cuda.synchronize()
    ferrum_hip.linear_forward_async(fh, w, dx, 1, k, None, 0, y, ferrum_hip.W8A32_EXACT)
    fh.sync()
    w.free()
    whole = n // period * period
    assert torch.equal(y[:whole].view(-1, period), want.expand(whole // period, period))
    assert torch.equal(y[whole:], want[:n - whole])
    del y
    torch.cuda.empty_cache()
