"""The matrix-core product (ut_gemm.hip: five or more activation rows) against
the closed form of the integer arithmetic, bit for bit, and against the
one-row GEMV's rows.  The sums are exact integers, so the tolerance is zero.
"""
import numpy as np
import pytest
import torch

from conftest import dev, host
from qgen import INT4, INT8, gemv_closed_form, rand_qtensor

pytestmark = pytest.mark.gpu

# weight tiles of 256 rows and their remainders, K steps of 128 columns and
# their tails, rows that are not 16-byte aligned, a payload's last bytes
SHAPES = [(1, 1), (5, 17), (15, 16), (256, 128), (257, 160), (300, 1000), (1003, 1537), (64, 31),
          (576, 7168), (255, 4096)]
SEQS = [5, 15, 16, 17, 32, 33, 70]


def run(ctx, q, x):
    out = torch.full((x.shape[0], q.out_dim), float("nan"), device="cuda:0")
    q.matmul(out, dev(x), x.shape[0])
    return host(out)


@pytest.mark.parametrize("fmt", [INT8, INT4])
@pytest.mark.parametrize("o,i", SHAPES)
def test_gemm_is_the_closed_form(ctx, fmt, o, i):
    import undertow_amd as U
    rng = np.random.default_rng(o * 7 + i + fmt)
    payload, scales = rand_qtensor(rng, fmt, o, i)
    q = U.QTensor(ctx, fmt, payload, scales, o, i)
    x = rng.standard_normal((max(SEQS), i)).astype(np.float32)
    x[1] = 0.0
    x[2] *= 1e-30
    x[3, 0] = 1e30
    want = gemv_closed_form(fmt, payload, scales, o, i, x)
    one = run(ctx, q, x[4:5])
    for seq in SEQS:
        got = run(ctx, q, x[:seq])
        assert np.array_equal(got, want[:seq]), seq
        assert np.array_equal(got[4:5], one)


@pytest.mark.parametrize("fmt", [INT8, INT4])
def test_gemm_largest_codes_do_not_overflow(ctx, fmt):
    """65,536 columns (the widest the int32 plane sums take) of extreme codes
    and digits: every x~ is 2^22, whose planes are 0, 0 and 64."""
    import undertow_amd as U
    o, i, seq = 17, 65536, 6
    payload = (np.full((o, i), -127, np.int8) if fmt == INT8 else np.full((o, i // 2), 0x88, np.uint8))
    scales = np.ones(o, np.float32)
    x = np.full((seq, i), np.float32(1.0))
    x[1] = -1.0
    x[2] = np.float32(0.99999988)  # x~ = 2^22 - 1 rounds up to 2^22 at E = 0
    x[3, ::2] = np.float32(0.50196) # digits near the balanced limit
    q = U.QTensor(ctx, fmt, payload, scales, o, i)
    assert np.array_equal(run(ctx, q, x), gemv_closed_form(fmt, payload, scales, o, i, x))


# one-launch GEMV of few outputs: pieces that fill no wave, the widest rows,
# outputs past a workgroup's four, the largest output counts and the first
# beyond them
@pytest.mark.parametrize("fmt", [INT8, INT4])
@pytest.mark.parametrize("o,i", [(1, 32), (5, 96), (7, 2080), (1024, 1024), (1025, 4096), (2048, 992),
                                 (2049, 128), (6, 8192), (6, 8224)])
def test_few_outputs_are_the_closed_form(ctx, fmt, o, i):
    import undertow_amd as U
    rng = np.random.default_rng(o + i + fmt)
    payload, scales = rand_qtensor(rng, fmt, o, i)
    q = U.QTensor(ctx, fmt, payload, scales, o, i)
    x = rng.standard_normal((4, i)).astype(np.float32)
    x[2] *= np.float32(1e-38)  # digits by the general scaling
    want = gemv_closed_form(fmt, payload, scales, o, i, x)
    for seq in (1, 2, 3, 4):
        assert np.array_equal(run(ctx, q, x[:seq]), want[:seq]), seq
    bad = x[:2].copy()
    bad[1, i - 1] = np.nan
    got = run(ctx, q, bad)
    assert np.isnan(got[1]).all() and np.array_equal(got[0], want[0])


# either side of the lines of gemv_direct_ok, where both ways were timed
@pytest.mark.parametrize("fmt,o,i,seq,direct", [
    (INT8, 64, 64, 4, True), (INT8, 1, 1024, 4, True), (INT8, 1, 1040, 4, False), (INT8, 16, 4096, 2, True),
    (INT8, 16, 8192, 1, True), (INT8, 16, 8208, 1, False), (INT4, 256, 256, 4, False), (INT4, 64, 64, 4, False),
    (INT4, 64, 256, 3, True), (INT4, 64, 4096, 2, True), (INT4, 64, 4128, 2, False), (INT4, 16, 8192, 1, True)])
def test_few_rows_take_the_faster_way(ctx, fmt, o, i, seq, direct):
    import undertow_amd as U
    rng = np.random.default_rng(o + i + seq)
    payload, scales = rand_qtensor(rng, fmt, o, i)
    q = U.QTensor(ctx, fmt, payload, scales, o, i)
    x = rng.standard_normal((seq, i)).astype(np.float32)
    ctx.enable_timing(True)
    before = ctx.kernel_time("gemv_direct")[0]
    got = run(ctx, q, x)
    launches = ctx.kernel_time("gemv_direct")[0] - before
    ctx.enable_timing(False)
    assert launches == int(direct)
    assert np.array_equal(got, gemv_closed_form(fmt, payload, scales, o, i, x))


@pytest.mark.parametrize("seq", [1, 4, 9])
@pytest.mark.parametrize("fmt", [INT8, INT4])
def test_product_over_its_own_input(ctx, fmt, seq):
    # x is digitised before anything is written: the output may replace it
    import undertow_amd as U
    rng = np.random.default_rng(seq)
    payload, scales = rand_qtensor(rng, fmt, 256, 256)
    q = U.QTensor(ctx, fmt, payload, scales, 256, 256)
    x = rng.standard_normal((seq, 256)).astype(np.float32)
    buf = dev(x)
    q.matmul(buf, buf, seq)
    np.testing.assert_array_equal(host(buf), gemv_closed_form(fmt, payload, scales, 256, 256, x))


def test_gemm_nonfinite_rows_are_nan(ctx):
    import undertow_amd as U
    rng = np.random.default_rng(5)
    payload, scales = rand_qtensor(rng, INT8, 40, 256)
    x = rng.standard_normal((9, 256)).astype(np.float32)
    want = gemv_closed_form(INT8, payload, scales, 40, 256, x)
    x[2, 7] = np.inf
    x[5, 255] = np.nan
    got = run(ctx, U.QTensor(ctx, INT8, payload, scales, 40, 256), x)
    assert np.isnan(got[[2, 5]]).all()
    ok = [r for r in range(9) if r not in (2, 5)]
    assert np.array_equal(got[ok], want[ok])


# f32 slices of one to four 64-column steps and none, tails of a step, outputs
# past a 64-row tile, K % 4 != 0 (the generic kernel), more columns than a
# slice of the product takes (the GEMV passes)
@pytest.mark.parametrize("o,i", [(256, 7168), (3, 4), (65, 60), (70, 132), (130, 200), (1000, 1028),
                                 (2048, 1024), (4096, 1024), (17, 131), (20000, 256)])
def test_f32_rows_equal_one_row_calls(ctx, o, i):
    """Each output's products are added in the one-row GEMV's order: bitwise."""
    import undertow_amd as U
    rng = np.random.default_rng(o + i)
    w = rng.standard_normal((o, i)).astype(np.float32)
    q = U.QTensor(ctx, U.F32, w, None, o, i)
    x = rng.standard_normal((131, i)).astype(np.float32)
    rows = [0, 3, 4, 63, 64, 127, 128, 130]
    one = np.concatenate([run(ctx, q, x[r:r + 1]) for r in rows])
    for seq in (5, 9, 64, 131):
        got = run(ctx, q, x[:seq])
        n = [k for k, r in enumerate(rows) if r < seq]
        assert np.array_equal(got[[rows[k] for k in n]], one[n]), seq
    ref = x.astype(np.float64) @ w.astype(np.float64).T
    err = np.linalg.norm(run(ctx, q, x) - ref) / np.linalg.norm(ref)
    assert err <= 2.0 ** -23 * max(1.0, np.log2(i))  # tree-wise f32 sums


# the lines of gemm_f32_min_rows: split and unsplit slices of one to four
# steps, more tiles than one wave; (rows in passes, rows in the product)
@pytest.mark.parametrize("o,i,few,more", [(64, 64, 4, 5), (65, 128, 8, 9), (65, 132, 12, 13), (65, 252, 13, 14),
                                          (16500, 252, 24, 25), (130, 1028, 4, 5), (256, 1024, 4, 5),
                                          (1024, 7168, 8, 9), (3000, 1500, 12, 13),
                                          (2048, 7168, 16, 17)])
def test_f32_rows_take_the_faster_way(ctx, o, i, few, more):
    import undertow_amd as U
    rng = np.random.default_rng(o + i)
    q = U.QTensor(ctx, U.F32, rng.standard_normal((o, i)).astype(np.float32), None, o, i)
    x = rng.standard_normal((more, i)).astype(np.float32)
    got, launches = {}, {}
    ctx.enable_timing(True)
    for n in (few, more):
        before = ctx.kernel_time("gemm_f32")[0]
        got[n] = run(ctx, q, x[:n])
        launches[n] = ctx.kernel_time("gemm_f32")[0] - before
    ctx.enable_timing(False)
    assert launches == {few: 0, more: 1}
    assert np.array_equal(got[more][:few], got[few])


# unsplit slices either side of the line between the two LDS tiles (16 stages
# of 128 columns; one odd, one even count past it), rows past both tile edges
@pytest.mark.parametrize("i", [2048, 2176, 2304])
@pytest.mark.parametrize("fmt", [INT8, INT4])
def test_long_slices_equal_few_rows(ctx, fmt, i):
    import torch
    import undertow_amd as U
    rng = np.random.default_rng(i)
    o, seq = 128 * 130 + 16, 65  # 262 tiles: no K split
    payload, scales = rand_qtensor(rng, fmt, o, i)
    q = U.QTensor(ctx, fmt, payload, scales, o, i)
    x = dev(rng.standard_normal((seq, i)).astype(np.float32))
    got, few = (torch.empty((seq, o), device="cuda") for _ in range(2))
    q.matmul(got, x, seq)
    for r in range(0, seq, 4):
        n = min(4, seq - r)
        q.matmul(few[r:r + n], x[r:r + n], n)
    assert torch.equal(got, few)
