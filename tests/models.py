"""Test models: the reference's oracle-tiny fixture and BASELINE config 1,
generated by the oracle's restated generator (undertow-bench/src/oracle.rs)
and loaded into the GPU backend tensor by tensor."""
import numpy as np

from oracle import oracle as O

CFG_KEYS = ["vocab_size", "hidden_size", "intermediate_size", "moe_intermediate_size",
            "num_hidden_layers", "first_k_dense_replace", "num_attention_heads", "n_routed_experts",
            "num_experts_per_tok", "n_shared_experts", "n_group", "topk_group", "norm_topk_prob",
            "routed_scaling_factor", "q_lora_rank", "kv_lora_rank", "qk_nope_head_dim",
            "qk_rope_head_dim", "v_head_dim", "rms_norm_eps", "rope_theta", "mtp",
            "max_position_embeddings"]

# Config 1, the tiny benchmark model: OracleSpec at its dimensions (undertow-bench/src/oracle.rs:150-310).
C1 = dict(seed=20260712, vocab_size=1024, hidden_size=256, intermediate_size=512,
          moe_intermediate_size=128, num_hidden_layers=2, first_k_dense_replace=1,
          num_attention_heads=4, n_routed_experts=8, num_experts_per_tok=2, n_shared_experts=1,
          n_group=4, topk_group=2, norm_topk_prob=1, routed_scaling_factor=2.5, q_lora_rank=96,
          kv_lora_rank=64, qk_nope_head_dim=32, qk_rope_head_dim=16, v_head_dim=32,
          init_std=0.02, mtp=1)

# Config 1 with DeepSeek-V3's attention dims (128 heads, latent 512 + rope
# 64, nope 128, v_head 128) and hidden 1024: the shapes the matrix-core
# attention, the int8 absorb kernels and the split-K kv_a / q_a pair (with
# its fused finish) take.
C1_MLA = dict(C1, hidden_size=1024, num_attention_heads=128, kv_lora_rank=512, qk_nope_head_dim=128,
              qk_rope_head_dim=64, v_head_dim=128)

# The same with a value head of 40 dims: the absorbed V's last workgroup of
# each head holds rows past the head (tails of its two 8-row passes).
C1_MLA_V40 = dict(C1_MLA, v_head_dim=40)

# A value head of 42: the heads' scales start at any even float.
C1_MLA_V42 = dict(C1_MLA, v_head_dim=42)

# Config 1 with DeepSeek-V3's router shape: 256 routed experts in 8 groups,
# top-4 groups, top-8 experts (the wave router with four keys per lane,
# which the gate/up launch runs itself on the decode path).
C1_E256 = dict(C1, n_routed_experts=256, num_experts_per_tok=8, n_group=8, topk_group=4)

FMT = {"f32": (O.F32, O.F32), "int8": (O.INT8, O.INT8), "int4": (O.INT4, O.INT8)}


def spec(overrides=None):
    return O.default_spec(**(overrides or {}))


def checkpoint(overrides=None, fmt="f32"):
    ck = O.Checkpoint(spec(overrides))
    ef, df = FMT[fmt]
    if fmt != "f32":
        ck.convert(ef, df)
    return ck


def prompt_ids(n, vocab, seed=7, stream=1):
    """Uniform ids in [0, vocab) from the restated PCG32 (uniform floats)."""
    u = O.pcg32_fill(seed, stream, n, kind="uniform")
    return [min(int(v * vocab), vocab - 1) for v in u]


def gpu_model(ctx, ck):
    import undertow_amd as U
    s = ck.spec
    cfg = {k: getattr(s, k) for k in CFG_KEYS}
    m = U.Model(ctx, cfg)
    for name, fmt, shape, payload, scales in ck.tensors():
        if len(shape) == 1:
            m.set_tensor(name, U.F32, payload, None, shape)
        else:
            m.set_tensor(name, fmt, payload, scales, shape)
    m.finalize()
    return m


# A one-layer MoE model whose MTP module restates the main model (the
# construction that pins draft_logits, mtp.rs:74-133): eh_proj = [I | 0]
# and enorm = 1 make the MTP input rmsnorm(embed(t_next)), which equals the
# embedding row to rounding because every row has unit RMS; the MTP layer
# copies layer 0 with its experts in reversed group order (router rows and
# bias permuted alike, so the routed function is unchanged but a lookup in
# the wrong layer's experts is not); the head's norm is the final norm
# times 0.5 and the head the lm_head times 4 (powers of two: exact).  Draft
# logits at pending position i are then exactly twice the main model's
# logits at position i of the sequence shifted by one token (to rounding).
IDENTITY = dict(num_hidden_layers=1, first_k_dense_replace=0, mtp=1)


def _group_reversal(E, n_group):
    g = E // n_group
    return np.concatenate([np.arange(b * g, (b + 1) * g) for b in reversed(range(n_group))])


def identity_mtp_checkpoint(overrides=None, fmt="f32"):
    """fmt "int4": experts int4 and dense matrices int8 (converted before the
    copies are made, so copies share codes and the head's scales are exactly
    4x); the embedding and eh_proj stay f32 in every format."""
    sp = spec(dict(IDENTITY, **(overrides or {})))
    base = O.Checkpoint(sp)
    emb = next(np.frombuffer(p.tobytes(), np.float32).reshape(sh)
               for n, f, sh, p, sc in base.tensors() if n == "model.embed_tokens.weight")
    if fmt != "f32":
        base.convert(*FMT[fmt])
    t = {name: (f, shape, payload, scales) for name, f, shape, payload, scales in base.tensors()}
    H, E = sp.hidden_size, sp.n_routed_experts
    perm = _group_reversal(E, sp.n_group)

    def f32(name):
        return np.frombuffer(t[name][2].tobytes(), np.float32).reshape(t[name][1])

    emb = emb.astype(np.float64)
    emb = (emb / np.sqrt((emb * emb).mean(axis=1, keepdims=True))).astype(np.float32)
    t["model.embed_tokens.weight"] = (O.F32, t["model.embed_tokens.weight"][1], emb, None)
    L = sp.num_hidden_layers  # the MTP module's layer index
    pre0, preL = "model.layers.0.", f"model.layers.{L}."
    for name in [n for n in t if n.startswith(preL)]:
        del t[name]
    for name in [n for n in t if n.startswith(pre0)]:
        rest = name[len(pre0):]
        fmt, shape, payload, scales = t[name]
        if rest.startswith("mlp.experts."):
            e, tail = rest[len("mlp.experts."):].split(".", 1)
            src = f"{pre0}mlp.experts.{perm[int(e)]}.{tail}"
            fmt, shape, payload, scales = t[src]
        elif rest == "mlp.gate.weight":
            payload = f32(name)[perm].copy()
        elif rest == "mlp.gate.e_score_correction_bias":
            payload = f32(name)[perm].copy()
        t[preL + rest] = (fmt, shape, payload, scales)
    eh = np.zeros((H, 2 * H), np.float32)
    eh[:, :H] = np.eye(H, dtype=np.float32)
    t[preL + "eh_proj.weight"] = (O.F32, (H, 2 * H), eh, None)
    t[preL + "enorm.weight"] = (O.F32, (H,), np.ones(H, np.float32), None)
    t[preL + "hnorm.weight"] = (O.F32, (H,), f32("model.norm.weight").copy(), None)
    t[preL + "shared_head.norm.weight"] = (O.F32, (H,), f32("model.norm.weight") * np.float32(0.5),
                                           None)
    hf, hshape, hp, hs = t["lm_head.weight"]
    if hf == O.F32:
        t[preL + "shared_head.head.weight"] = (O.F32, hshape, f32("lm_head.weight") * np.float32(4.0),
                                               None)
    else:
        t[preL + "shared_head.head.weight"] = (hf, hshape, hp.copy(), hs * np.float32(4.0))
    tensors = [(n, fmt, shape, np.ascontiguousarray(p), s) for n, (fmt, shape, p, s) in t.items()]
    return O.Checkpoint.from_tensors(sp, tensors)


def greedy_sim(stream, depth, corrupt_at, max_new):
    """What the speculative loop emits and accepts when each round's drafts
    are the greedy continuation `stream` with the draft at corrupt_at(round)
    (None: no draft) made wrong: (emitted, drafted, accepted).  The
    reference's accept rule applied to a known sequence."""
    k, emitted, drafted, accepted, rnd = 0, [stream[0]], 0, 0, 0
    while len(emitted) < max_new:
        p = corrupt_at(rnd)
        a = depth if p is None else min(p, depth)
        drafted += depth
        for j in range(a):
            emitted.append(stream[k + 1 + j])
            accepted += 1
            if len(emitted) >= max_new:
                return emitted, drafted, accepted
        k += a + 1
        emitted.append(stream[k])
        rnd += 1
    return emitted, drafted, accepted


# DeepSeek-V3 width, 4 layers (1 dense), 256 routed
# experts top-8 in 8 groups (top-4 groups), 1 shared expert, MTP module.
C4 = dict(vocab_size=129280, hidden_size=7168, intermediate_size=18432, moe_intermediate_size=2048,
          num_hidden_layers=4, first_k_dense_replace=1, num_attention_heads=128,
          n_routed_experts=256, num_experts_per_tok=8, n_shared_experts=1, n_group=8,
          topk_group=4, norm_topk_prob=1, routed_scaling_factor=2.5, q_lora_rank=1536,
          kv_lora_rank=512, qk_nope_head_dim=128, qk_rope_head_dim=64, v_head_dim=128,
          init_std=0.02, mtp=1, max_position_embeddings=4096)


def gpu_model_raw(ctx, ck):
    """gpu_model without host copies: each tensor goes from the oracle's
    buffers straight to ut_model_set_tensor (tens of GB at config 4)."""
    import undertow_amd as U
    s = ck.spec
    cfg = {k: getattr(s, k) for k in CFG_KEYS}
    m = U.Model(ctx, cfg)
    L = U.lib()
    for name, fmt, shape, addr, nbytes, saddr in ck.raw_tensors():
        d0 = shape[0]
        d1 = shape[1] if len(shape) == 2 else 1
        f = U.F32 if len(shape) == 1 else fmt
        ctx.check(L.ut_model_set_tensor(m._h, name.encode(), f, addr, nbytes, saddr, d0, d1))
    m.finalize()
    return m


def write_converted(ck, d, expert_layers):
    """The converter's layout (undertow-convert/src/lib.rs:273-345): routed
    experts of layer L in experts-{L:05}.safetensors, the rest in
    dense.safetensors, plus model.safetensors.index.json; shard bytes from
    the oracle's restated writer (undertow-io/src/writer.rs:73-110)."""
    import json
    groups = {}
    for t in ck.tensors():
        name = t[0]
        shard = "dense.safetensors"
        for L in expert_layers:
            if name.startswith(f"model.layers.{L}.mlp.experts."):
                shard = f"experts-{L:05d}.safetensors"
        groups.setdefault(shard, []).append(t)
    wm = {}
    for shard, ts in groups.items():
        sub = O.Checkpoint.from_tensors(ck.spec, ts)
        (d / shard).write_bytes(sub.safetensors_bytes())
        for name, fmt, shape, payload, scales in ts:
            wm[name] = shard
            if fmt != O.F32:
                wm[name + ".scales"] = shard
    (d / "model.safetensors.index.json").write_text(json.dumps({"metadata": {}, "weight_map": wm}))
    return groups
