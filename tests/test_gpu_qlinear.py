"""ops::qlinear on the GPU (packed per-row int8 / int4 QWeight): every output
bit-equal to the oracle's restatement of qaccum_cols (bias first, p
ascending, no FMA), across int8 / int4, odd widths (the split-half nibble
layout's last column), several rows of x, K beyond one LDS chunk, the
one-row kernel's chunk and 4-row-group tails (K = 1, 2, 7, 389) and its
16-, 32- and 64-byte column tiles (chosen by the output width; int4 takes
the 64-byte tile, where a lane owns two nibble columns, only above 16,384
outputs, so two such cases end on partial chunks and row groups), and the
reference's dimension errors (ops.rs:316-330)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def dev(a):
    import torch

    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def host(fh, t):
    import torch

    fh.sync()
    torch.cuda.synchronize()
    return t.cpu().numpy()


@pytest.mark.parametrize("kind", [0, 1])
@pytest.mark.parametrize("m,k,n,bias", [(1, 768, 768, True), (1, 768, 50257, False), (3, 1100, 333, True),
                                        (5, 64, 7, True), (8, 3072, 768, True), (1, 513, 1, True),
                                        (1, 3072, 2304, True), (1, 389, 129, True), (1, 7, 130, False),
                                        (1, 1, 5, True), (1, 2, 64, True), (1, 777, 5000, True),
                                        (1, 1000, 10000, False), (1, 1001, 9000, True),
                                        (1, 1001, 20001, True), (1, 389, 50257, False)])
def test_qlinear_is_bit_exact(fh, orc, kind, m, k, n, bias):
    import torch

    import ferrum_hip

    rng = np.random.default_rng(k * 7 + n + kind)
    wf = (rng.standard_normal((k, n)) * 0.05).astype(np.float32)
    ow = orc.QWeight(wf, k, n, kind)
    x = rng.standard_normal((m, k)).astype(np.float32)
    b = (rng.standard_normal(n) * 0.1).astype(np.float32) if bias else np.zeros(n, np.float32)
    want = orc.qlinear(x, ow, b, threads=1)
    w = ferrum_hip.QWeight(fh, ow.scales, ow.q, k, n, kind)
    y = torch.full((m, n), float("nan"), device="cuda")
    torch.cuda.synchronize()
    ferrum_hip.qlinear_async(fh, w, dev(x), m, k, dev(b) if bias else None, n if bias else 0, y)
    got = host(fh, y)
    w.free()
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))


def test_qlinear_errors(fh, orc):
    import torch

    import ferrum_hip

    ow = orc.QWeight(np.ones((64, 10), np.float32), 64, 10, 0)
    w = ferrum_hip.QWeight(fh, ow.scales, ow.q, 64, 10, 0)
    x, y = dev(np.ones((1, 64), np.float32)), torch.empty(10, device="cuda")
    with pytest.raises(ferrum_hip.DimMismatch, match="input width 63"):
        ferrum_hip.qlinear_async(fh, w, x, 1, 63, None, 0, y)
    with pytest.raises(ferrum_hip.DimMismatch, match="bias length 9"):
        ferrum_hip.qlinear_async(fh, w, x, 1, 64, dev(np.zeros(9, np.float32)), 9, y)
    with pytest.raises(ferrum_hip.FerrumHipError, match="unknown kind"):
        ferrum_hip.QWeight(fh, ow.scales, ow.q, 64, 10, 2)
    w.free()


# Both tile widths of the kernel for several rows (or k_qlinear, where the launch rule
# takes it), one row per lane, K ending inside a chunk and inside a 16-position piece,
# odd widths (the int4 halves' last columns), a bias of -0 under products of -0 (no
# padding may turn the sum to +0) and non-finite activations.
@pytest.mark.parametrize("kind", [0, 1])
@pytest.mark.parametrize("m,k,n", [(2, 15, 1), (16, 128, 33), (17, 129, 31), (40, 300, 2303), (66, 130, 4095),
                                   (129, 97, 4097), (5, 70, 32769), (2, 33, 40001)])
def test_qlinear_rows_per_lane_and_ragged_edges(fh, orc, kind, m, k, n):
    import torch

    import ferrum_hip

    rng = np.random.default_rng(m * 7 + n + kind)
    wf = (rng.standard_normal((k, n)) * 0.05).astype(np.float32)
    wf[:, 0] = np.abs(wf[:, 0])
    ow = orc.QWeight(wf, k, n, kind)
    x = rng.standard_normal((m, k)).astype(np.float32)
    x[0], x[m - 1, k - 1] = -0.0, np.inf
    b = (rng.standard_normal(n) * 0.1).astype(np.float32)
    b[0] = -0.0
    want = orc.qlinear(x, ow, b, threads=1)
    assert np.signbit(want[0, 0]) and want[0, 0] == 0
    w = ferrum_hip.QWeight(fh, ow.scales, ow.q, k, n, kind)
    y = torch.full((m, n), float("nan"), device="cuda")
    torch.cuda.synchronize()
    ferrum_hip.qlinear_async(fh, w, dev(x), m, k, dev(b), n, y)
    got = host(fh, y)
    w.free()
    nan = np.isnan(got) & np.isnan(want)
    assert np.array_equal(np.where(nan, 0, got.view(np.uint32)), np.where(nan, 0, want.view(np.uint32)))


# A few rows of a wide output (k_qlinear: 64-byte column tiles, four rows of x per
# workgroup, K in chunks of 512 positions), where the launch rule takes it over the
# kernel above by half of its time or more: the last tile's columns ragged (odd int4
# widths), one, three and four rows of the last group, K of one chunk, of whole chunks
# and ending inside one, non-finite values and a sum of -0.
@pytest.mark.parametrize("kind,m,k,n", [(0, 2, 255, 28673), (0, 3, 512, 28671), (0, 4, 130, 31999), (0, 5, 256, 16385),
                                        (0, 8, 513, 14337), (1, 2, 129, 32001), (1, 3, 100, 28673), (1, 4, 250, 28671),
                                        (1, 7, 129, 32001), (1, 8, 1025, 32767), (0, 4, 1537, 16384)])
def test_qlinear_few_rows_of_a_wide_output(fh, orc, kind, m, k, n):
    test_qlinear_rows_per_lane_and_ragged_edges(fh, orc, kind, m, k, n)


# Two and four rows per lane, in tiles of 16 columns and of 32 (more than 64 rows never
# take k_qlinear).
@pytest.mark.parametrize("kind", [0, 1])
@pytest.mark.parametrize("m,k,n,tm", [(95, 300, 4090, 2), (90, 129, 4089, 2), (125, 130, 4090, 4), (128, 97, 4095, 4),
                                      (80, 70, 32769, 2), (78, 145, 32768, 2), (128, 33, 32769, 4), (123, 130, 32771, 4)])
def test_qlinear_two_and_four_rows_per_lane(fh, orc, kind, m, k, n, tm):
    import seq_tiles

    cols, row_bytes = 32 if n >= 32768 else 16, n if kind == 0 else (n + 1) // 2
    tiles = -(-row_bytes // (cols if kind == 0 else cols // 2))
    assert seq_tiles.rows_per_lane(cols, tiles, m) == tm
    test_qlinear_rows_per_lane_and_ragged_edges(fh, orc, kind, m, k, n)
