"""The absorbed kv_b halves over a prompt's rows (ut_absorb.hip: more than 16
rows) in the model: DeepSeek-V3 attention shapes on the config-1 model.

Up to 128 positions every kernel of a prompt keeps the short calls' sums, so
one call equals calls of at most 16 rows bit for bit (absorb_v's matrix-core
sums among them, at rows and value heads that fill no tile).  Beyond, the
prompt attention and absorb_q round differently; the bars are the oracle
tests' 1e-3 / 1e-4 on the logits.
"""
import numpy as np
import pytest

from models import C1_MLA, C1_MLA_V40, C1_MLA_V42, checkpoint, gpu_model, prompt_ids
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def by_sixteen(m, ids):
    s = m.session()
    return np.concatenate([s.prefill(ids[i:i + 16]) for i in range(0, len(ids), 16)])


@pytest.mark.parametrize("cfg", [C1_MLA, C1_MLA_V40])
def test_short_prompt_equals_short_calls(ctx, cfg):
    m = gpu_model(ctx, checkpoint(cfg, fmt="int4"))
    ids = prompt_ids(128, cfg["vocab_size"], seed=3)
    want = by_sixteen(m, ids)
    for n in (17, 64, 65, 128):
        assert np.array_equal(m.session().prefill(ids[:n]), want[:n]), n


def test_long_prompt_matches_oracle(ctx):
    ck = checkpoint(C1_MLA, fmt="int4")
    m = gpu_model(ctx, ck)
    ids = prompt_ids(150, C1_MLA["vocab_size"], seed=4)
    want = O.Model(ck).forward(ids)
    got = m.forward(ids)
    few = by_sixteen(m, ids)
    for a in (got, few):
        e = np.abs(a - want)
        assert e.max() <= 1e-3 and e.mean() <= 1e-4, (e.max(), e.mean())
    # a prompt continued: 60 rows at positions 90 ..
    s = m.session()
    s.prefill(ids[:90])
    e = np.abs(s.prefill(ids[90:]) - want[90:])
    assert e.max() <= 1e-3 and e.mean() <= 1e-4


@pytest.mark.parametrize("cfg,taken", [(C1_MLA_V40, True), (C1_MLA_V42, False)])
def test_value_heads_of_whole_float4s(ctx, cfg, taken):
    """absorb_q's matrix-core kernel loads each head's scales 16 bytes at a
    time, so it leaves a value head that is no multiple of four floats."""
    ck = checkpoint(cfg, fmt="int4")
    m = gpu_model(ctx, ck)
    ids = prompt_ids(150, cfg["vocab_size"], seed=4)
    ctx.enable_timing(True)
    before = ctx.kernel_time("absorb_q_rows")[0]
    got = m.forward(ids)
    launches = ctx.kernel_time("absorb_q_rows")[0] - before
    ctx.enable_timing(False)
    assert (launches > 0) == taken
    e = np.abs(got - O.Model(ck).forward(ids))
    assert e.max() <= 1e-3 and e.mean() <= 1e-4, (e.max(), e.mean())
