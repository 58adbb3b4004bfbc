"""Calls captured into graphs beside eager calls of other sizes on the same
context: what a capture needs is there after an eager call of its size or a
larger one, and what it recorded stays valid when later calls need more."""
import numpy as np
import pytest
import torch

from conftest import dev
from qgen import INT4, INT8, rand_qtensor

pytestmark = pytest.mark.gpu


@pytest.fixture
def side():
    """A stream of its own with a fresh context bound to it."""
    import undertow_amd as U
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        c = U.Context(0)
        yield s, c
        s.synchronize()


def expert_table(c, rng, fmt, E, H, I):
    import undertow_amd as U
    tbl = U.ExpertTable(c, E, H, I)
    for e in range(E):
        tbl.set(e, *[U.QTensor(c, fmt, *rand_qtensor(rng, fmt, o, i), o, i)
                     for o, i in ((I, H), (I, H), (H, I))])
    return tbl


def expert_rows(rng, E, H, k, rows):
    ids = dev(np.stack([rng.permutation(E)[:k] for _ in range(rows)]).astype(np.int32))
    return ids, dev(rng.random((rows, k)).astype(np.float32)), dev(rng.standard_normal((rows, H)).astype(np.float32))


def capture(s, f):
    s.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        out = f()
    return g, out


def test_captured_experts_outlive_a_longer_prompt(side):
    """A decode call's graph keeps its arena block when a prompt grows the
    arena past it (600 rows: 2.6 MB and more of scratch, the four rows'
    block is under 1.7 MB)."""
    s, c = side
    rng = np.random.default_rng(8)
    E, H, I, k = 6, 256, 128, 2
    assert 600 * k * (H + I) * 4 > 1.7e6
    tbl = expert_table(c, rng, INT4, E, H, I)
    ids, w, x = expert_rows(rng, E, H, k, 600)
    few = [t[:4].contiguous() for t in (ids, w, x)]
    want = tbl.moe_experts(*few)
    g, got = capture(s, lambda: tbl.moe_experts(*few))
    every = tbl.moe_experts(ids, w, x)
    spill = torch.zeros(64 << 20, dtype=torch.uint8, device="cuda")  # what a freed block would hold
    for _ in range(3):
        got.zero_()
        spill.fill_(255)
        g.replay()
        s.synchronize()
        assert torch.equal(got, want)
        assert torch.equal(tbl.moe_experts(ids, w, x), every)
    assert torch.equal(every[:4], want)


def test_few_experts_rows_captured_after_a_prompt(side):
    """The scratch of a four-row pass is there after a call of six rows, whose
    own grouped scratch is smaller (64 slots of four rows against 96 pairs:
    4.2 MB, more than an arena of 1.17 MB * 1.25 + 1 MiB)."""
    s, c = side
    rng = np.random.default_rng(9)
    E, H, I, k = 64, 2048, 512, 16
    tbl = expert_table(c, rng, INT4, E, H, I)
    ids, w, x = expert_rows(rng, E, H, k, 6)
    want = tbl.moe_experts(ids, w, x)
    few = [t[:4].contiguous() for t in (ids, w, x)]
    g, got = capture(s, lambda: tbl.moe_experts(*few))
    for _ in range(3):
        got.zero_()
        g.replay()
        s.synchronize()
        assert torch.equal(got, want[:4])
        assert torch.equal(tbl.moe_experts(ids, w, x), want)


@pytest.mark.parametrize("fmt", [INT8, INT4])
def test_few_matmul_rows_captured_after_a_prompt(side, fmt):
    """A 512-row product of 7168 x 2048 is 448 workgroups and splits no
    columns; four rows split them: the partials' buffer is there all the same."""
    import undertow_amd as U
    s, c = side
    rng = np.random.default_rng(fmt)
    q = U.QTensor(c, fmt, *rand_qtensor(rng, fmt, 7168, 2048), 7168, 2048)
    x = dev(rng.standard_normal((512, 2048)).astype(np.float32))
    every, few = (torch.empty((n, 7168), device="cuda") for n in (512, 4))
    q.matmul(every, x, 512)
    g, _ = capture(s, lambda: q.matmul(few, x[:4], 4))
    for _ in range(3):
        few.zero_()
        g.replay()
        s.synchronize()
        assert torch.equal(few, every[:4])


def test_product_captured_without_partials(side):
    """A first product under capture has no buffer for the partials of a K
    split and runs unsplit; the arena is there from a call of another kind."""
    import undertow_amd as U
    s, c = side
    rng = np.random.default_rng(4)
    q = U.QTensor(c, INT4, *rand_qtensor(rng, INT4, 1024, 7168), 1024, 7168)
    x = dev(rng.standard_normal((37, 7168)).astype(np.float32))
    y = torch.empty((37, 1024), device="cuda")
    qa = torch.randn((16, 128, 576), device="cuda")  # 67 MB of slice partials, no split-K buffer
    kc = U.mla_cache_split(c, torch.randn((512, 512), device="cuda"), torch.randn((512, 64), device="cuda"))
    U.mla_attend_split(c, qa[..., :512].contiguous(), qa[..., 512:].contiguous(), kc, 496, 0.07)
    g, _ = capture(s, lambda: q.matmul(y, x, 37))
    for _ in range(3):
        y.zero_()
        g.replay()
        s.synchronize()
        got = y.clone()
        q.matmul(y, x, 37)  # split, from the first eager call on
        assert torch.equal(got, y)


# a prompt unsplit (1,600 column groups), then fewer rows that split; the same
# rows over at most 128 positions, whose slices are the context length's; few
# rows whose slices are
@pytest.mark.parametrize("first,then", [((400, 400), (24, 400)), ((300, 300), (128, 128)),
                                        ((128, 129), (128, 128)), ((200, 9000), (20, 9000)),
                                        ((200, 9000), (16, 9000))])
def test_shorter_attention_captured_after_a_prompt(side, first, then):
    import undertow_amd as U
    s, c = side
    g = torch.Generator(device="cuda").manual_seed(3)
    rnd = lambda *d: torch.randn(d, device="cuda", generator=g)
    T = first[1]
    kc = U.mla_cache_split(c, rnd(T, 512), rnd(T, 64))
    q, p = rnd(first[0], 128, 512), rnd(first[0], 128, 64)
    out = torch.empty_like(q)
    call = lambda R, T: U.mla_attend_split(c, q[:R], p[:R], kc, T - R, 0.07, out=out[:R])
    call(*first)
    gr, _ = capture(s, lambda: call(*then))
    out.zero_()
    gr.replay()
    s.synchronize()
    got = out[:then[0]].clone()
    call(*then)
    assert torch.equal(got, out[:then[0]])
