"""A prompt of up to 128 positions equals its decode steps bit for bit: the
products, the grouped experts, the router gate (k_rowdot_f32_rows against
k_rowdot_f32), the norms and, at DeepSeek-V3 attention shapes, the attention
of one call are compared with one-row calls, so no kernel is on both sides.
Beyond 16 rows and 128 positions the attention splits positions by the rows
of the call: there the oracle tests' 1e-3 / 1e-4 hold.
"""
import numpy as np
import pytest

from models import C1, C1_E256, C1_MLA, checkpoint, gpu_model, prompt_ids

pytestmark = pytest.mark.gpu


def by_ones(m, ids):
    s = m.session()
    return np.stack([s.decode(t) for t in ids])


# (C1_E256 at 128 rows: the gate's 16 rows per workgroup)
@pytest.mark.parametrize("cfg", [C1, C1_E256, C1_MLA], ids=["c1", "e256", "mla"])
def test_prompt_equals_decode_steps(ctx, cfg):
    m = gpu_model(ctx, checkpoint(cfg, fmt="int4"))
    ids = prompt_ids(128, cfg["vocab_size"], seed=5)
    want = by_ones(m, ids)
    for n in (5, 16, 17, 40, 128):
        assert np.array_equal(m.session().prefill(ids[:n]), want[:n]), n


# the gate's columns in one to eight steps of 1,024 (each instantiation, with
# full and part-filled last steps); ten experts: its last workgroup of four
@pytest.mark.parametrize("hidden,experts", [(1024, 8), (1056, 8), (3072, 8), (5120, 10), (7168, 8),
                                            (8192, 10)])
def test_gate_of_many_rows_equals_one_row(ctx, hidden, experts):
    cfg = dict(C1, vocab_size=64, hidden_size=hidden, intermediate_size=64, moe_intermediate_size=64,
               num_hidden_layers=1, first_k_dense_replace=0, n_routed_experts=experts, n_group=2,
               topk_group=1, mtp=0)
    m = gpu_model(ctx, checkpoint(cfg, fmt="int4"))
    ids = prompt_ids(21, 64, seed=hidden)
    ctx.enable_timing(True)
    before = ctx.kernel_time("rowdot_f32_rows")[0]
    got = m.session().prefill(ids)
    launches = ctx.kernel_time("rowdot_f32_rows")[0] - before
    ctx.enable_timing(False)
    assert launches == 1
    assert np.array_equal(got, by_ones(m, ids))


def test_rows_past_128_positions(ctx):
    """The first calls that leave the decode kernels' sums: 17 rows that reach
    position 129, beside 16 rows (as one) and 17 that end at 128 (as one)."""
    m = gpu_model(ctx, checkpoint(C1_MLA, fmt="int4"))
    ids = prompt_ids(129, C1_MLA["vocab_size"], seed=6)
    want = by_ones(m, ids)

    def tail(n, end):
        s = m.session()
        for i in range(0, end - n, 16):
            s.prefill(ids[i:min(i + 16, end - n)])
        return s.prefill(ids[end - n:end])

    assert np.array_equal(tail(16, 129), want[113:129])
    assert np.array_equal(tail(17, 128), want[111:128])
    e = np.abs(tail(17, 129) - want[112:129])
    assert e.max() <= 1e-3 and e.mean() <= 1e-4
