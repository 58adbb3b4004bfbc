"""The grouped expert products (ut_moe_rows.hip: six or more rows, int8 eight) against
one-to-four-row calls of the same rows, bit for bit: every total is an exact
integer and SiLU and the choices' sum run in the same order, so the tolerance
is zero.  (Four-row calls are checked against the oracle in test_gpu_moe.py.)
"""
import numpy as np
import pytest
import torch

from conftest import dev, host
from qgen import INT4, INT8, rand_qtensor

pytestmark = pytest.mark.gpu


def table(ctx, rng, fmt, E, H, I, skip=()):
    import undertow_amd as U
    tbl = U.ExpertTable(ctx, E, H, I)
    for e in range(E):
        if e in skip:
            continue
        tbl.set(e, *[U.QTensor(ctx, fmt, *rand_qtensor(rng, fmt, o, i), o, i)
                     for o, i in ((I, H), (I, H), (H, I))])
    return tbl


def graph_nodes(g):
    import ctypes as C
    import undertow_amd as U
    n = C.c_size_t(0)  # (through the library: the HIP runtime that it is linked to)
    assert U.lib().hipGraphGetNodes(C.c_void_p(g.raw_cuda_graph()), None, C.byref(n)) == 0
    return n.value


def by_fours(tbl, ids, w, x):
    return torch.cat([tbl.moe_experts(ids[r:r + 4].contiguous(), w[r:r + 4].contiguous(),
                                      x[r:r + 4].contiguous()) for r in range(0, len(x), 4)])


# h rows of a 64-row tile and remainders, down rows of a 128-row tile and
# remainders, widths with and without padded planes
@pytest.mark.parametrize("fmt,H,I", [(INT4, 512, 256), (INT4, 288, 160), (INT8, 272, 144),
                                     (INT8, 256, 128), (INT4, 7168, 2048)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_rows_equal_four_row_calls(ctx, fmt, H, I, dtype):
    rng = np.random.default_rng(H + I + fmt)
    E, k, rows = 6, 3, 41
    tbl = table(ctx, rng, fmt, E, H, I)
    ids = dev(np.stack([rng.permutation(E)[:k] for _ in range(rows)]).astype(np.int32))
    w = dev(rng.random((rows, k)).astype(np.float32))
    x = dev(rng.standard_normal((rows, H)).astype(np.float32)).to(dtype)
    want = by_fours(tbl, ids, w, x)
    for n in (5, 6, 8, 41):
        got = tbl.moe_experts(ids[:n].contiguous(), w[:n].contiguous(), x[:n].contiguous())
        assert torch.equal(got, want[:n]), n


# an expert with every row (tiles of 32 and their remainders), experts with
# none, more rows than one group of pairs takes
@pytest.mark.parametrize("rows,k,E", [(16, 1, 4), (17, 1, 4), (33, 2, 4), (64, 1, 300),
                                      (133, 64, 64)])
def test_tiles_of_one_expert(ctx, rows, k, E):
    rng = np.random.default_rng(rows * k)
    H, I = 64, 32
    tbl = table(ctx, rng, INT4, E, H, I)
    ids = np.stack([rng.permutation(E)[:k] for _ in range(rows)]).astype(np.int32)
    ids[:, 0] = E - 1 if k == 1 else ids[:, 0]
    x = dev(rng.standard_normal((rows, H)).astype(np.float32))
    w = dev(rng.random((rows, k)).astype(np.float32))
    assert torch.equal(tbl.moe_experts(dev(ids), w, x), by_fours(tbl, dev(ids), w, x))


def test_invalid_choices_are_skipped_and_reported(ctx):
    import undertow_amd as U
    rng = np.random.default_rng(3)
    E, H, I, k, rows = 5, 64, 32, 3, 9
    tbl = table(ctx, rng, INT8, E, H, I, skip=(4,))
    ids = np.stack([rng.permutation(4)[:k] for _ in range(rows)]).astype(np.int32)
    ids[1, 0] = -1  # no choice (top_k above the expert count): not an error
    x = dev(rng.standard_normal((rows, H)).astype(np.float32))
    w = dev(rng.random((rows, k)).astype(np.float32))
    assert torch.equal(tbl.moe_experts(dev(ids), w, x), by_fours(tbl, dev(ids), w, x))
    ctx.synchronize()
    for bad in (E, -7, 4):  # out of range, negative, not loaded
        ids[2, 1] = bad
        got = tbl.moe_experts(dev(ids), w, x)
        with pytest.raises(U.UtError) as e:
            ctx.synchronize()
        assert e.value.code == U.runtime.UT_ERR_BAD_EXPERT
        want = by_fours(tbl, dev(ids), w, x)
        with pytest.raises(U.UtError):
            ctx.synchronize()
        assert torch.equal(got, want)


@pytest.mark.parametrize("E,k,ng,tg", [(8, 2, 4, 2), (16, 4, 1, 1), (4, 6, 1, 1)])
def test_routed_rows_equal_route_then_experts(ctx, E, k, ng, tg):
    import undertow_amd as U
    rng = np.random.default_rng(E)
    H, I, rows = 64, 32, 22
    tbl = table(ctx, rng, INT4, E, H, I)
    logits = dev(rng.standard_normal((rows, E)).astype(np.float32))
    x = dev(rng.standard_normal((rows, H)).astype(np.float32))
    out, ids, w = tbl.moe_route_experts(logits, None, x, k, ng, tg, True, 2.5)
    ids1, w1 = U.route(ctx, logits, None, k, ng, tg, True, 2.5)
    assert torch.equal(ids, ids1) and torch.equal(w, w1)
    assert torch.equal(out, by_fours(tbl, ids1, w1, x))


def test_rows_under_capture_without_scratch_fall_back(ctx):
    """A captured call whose grouped scratch is not there takes the four-row
    passes (which one earlier call of four rows sized): its graph holds their
    launches, three and more per pass, and not the grouped path's six."""
    import undertow_amd as U
    rng = np.random.default_rng(8)
    E, H, I, k, rows = 6, 256, 128, 2, 600
    # the arena after four rows: 1 MiB and 1.25 times six slots of four rows
    # (h, its digits, d) with the row digits; 600 rows' h and d alone are more
    four = 6 * 4 * (I * 4 + 6 * I // 2 + H * 4) + 4 * 6 * H // 2 + 16384
    assert rows * k * (H + I) * 4 > four * 1.25 + (1 << 20)
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        c = U.Context(0)
        tbl = table(c, rng, INT4, E, H, I)
        ids = dev(np.stack([rng.permutation(E)[:k] for _ in range(rows)]).astype(np.int32))
        w = dev(rng.random((rows, k)).astype(np.float32))
        x = dev(rng.standard_normal((rows, H)).astype(np.float32))
        want = by_fours(tbl, ids, w, x)
        s.synchronize()
        g = torch.cuda.CUDAGraph(keep_graph=True)
        with torch.cuda.graph(g, stream=s):
            got = tbl.moe_experts(ids, w, x)
        assert graph_nodes(g) >= 3 * rows // 4
        for _ in range(3):
            got.zero_()
            g.replay()
            s.synchronize()
            assert torch.equal(got, want)
            # eager, the grouped products: the arena grows past the graph's block
            assert torch.equal(tbl.moe_experts(ids, w, x), want)
