"""RMSNorm ahead of the skinny GEMMs (batched streams, the full-sequence depth
pass): the norm weights multiply the rounded activations, as RMSNorm rounds them
(modules.cpp:72-84), and no weight of the matrix is rounded a second time.

Weights are chosen so that a matrix multiplied by the norm weights ahead of time
and rounded to the storage type would show:
  * every |W| 1.5 x a power of two and every norm weight 1 + one step of the
    type: each product lies halfway between two values and rounds up, so the
    logits grow by the same factor (bf16 1.00258, fp16 1.00033) -- the scale of
    the logits against the oracle's has to be nearer 1 than half of that;
  * fp16 with small norm weights: products below the smallest normal number lose
    bits (1.3e-2 of the logits here), the operands apart do not (the logits' own
    rounding, 1.2e-3).
"""

from __future__ import annotations

import dataclasses

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

STEP = {"bf16": 2.0 ** -7, "fp16": 2.0 ** -10}


def scale(got, exp):
    got, exp = np.asarray(got, np.float64), np.asarray(exp, np.float64)
    return float((got * exp).sum() / (exp * exp).sum())


def halfway(w, dtype):
    """The tiny model's weights with the head and its norm at halfway products,
    and how much such a head would grow."""
    w = dict(w)
    w["lm_head.weight"] = (np.sign(w["lm_head.weight"]) * 1.5 / 16).astype(np.float32)
    w["decoder_norm.weight"] = np.full_like(w["decoder_norm.weight"], 1 + STEP[dtype])
    exact = 1.5 * (1 + STEP[dtype])
    return w, np.ceil(exact / STEP[dtype]) * STEP[dtype] / exact - 1


@pytest.fixture(scope="module")
def env(gpu_available):
    import mrt_df
    import synth_bundle
    from oracle import depthformer_oracle as O
    cfg = mrt_df.Config.tiny(8)
    return dict(mrt_df=mrt_df, O=O, cfg=cfg, w=synth_bundle.make_weights(cfg, seed=31, norm_jitter=0.1),
                ocfg=O.DepthformerConfig(**dataclasses.asdict(cfg)))


def _embs(om, k, D):
    return om.P.r(np.random.default_rng(k).standard_normal((2, k, D)).astype(np.float32))


@pytest.mark.parametrize("dtype", ["bf16", "fp16"])
def test_depth_forward_full_scale(env, dtype):
    import torch
    w, grown = halfway(env["w"], dtype)
    om = env["O"].OracleDepthformer(w, env["ocfg"], mode=dtype)
    e = _embs(om, 16, env["cfg"].d_model)
    m = env["mrt_df"].Depthformer(w, env["cfg"], dtype=dtype)
    got = m.new_state(max_frames=1).depth_forward_full(torch.tensor(e, device="cuda").to(m.torch_dtype)).cpu().numpy()
    m.close()
    assert abs(scale(got, om.depth_forward_full(e)) - 1) < grown / 2


@pytest.mark.parametrize("B", [1, 3, 20])
def test_batched_slices_scale(env, B):
    import torch
    O, cfg, F, L, C = env["O"], env["cfg"], 3, 16, 8
    w, grown = halfway(env["w"], "bf16")
    rng = np.random.default_rng(B)
    tok = rng.integers(2, 130, size=(2 * B, cfg.max_encoder_length)).astype(np.int32)
    teacher = (2 + C * np.arange(L) + rng.integers(0, C, size=(B, F, L))).astype(np.int32)
    m = env["mrt_df"].Depthformer(w, cfg, dtype="bf16")
    b = env["mrt_df"].Batch(m, B, max_frames=F)
    sl = torch.zeros((F, L, 2 * B, C), dtype=torch.float32, device="cuda")
    kw = dict(num_frames=F, rvq_depth=L, temperature=1.1, top_k=4, guidance_weight=5.0, codebook_size=C,
              codec_offset=2)
    b.generate_tokens(tok, env["mrt_df"].GenOptions(seed=0, **kw), seeds=list(range(B)), teacher=teacher,
                      record=dict(slices=sl))
    sl = sl.cpu().numpy()
    b.close()
    m.close()
    om = O.OracleDepthformer(w, env["ocfg"], mode="bf16")
    for s in {0, B - 1}:
        rec = {}
        O.generate_tokens(om, tok[2 * s:2 * s + 2], O.GenerateOptions(seed=s, **kw), teacher=teacher[s], record=rec)
        assert abs(scale(sl[:, :, 2 * s:2 * s + 2], rec["slices"]) - 1) < grown / 2


def test_small_fp16_norm_weights(env):
    import torch
    w = dict(env["w"])
    w["lm_head.weight"] = w["lm_head.weight"] / 16
    w["decoder_norm.weight"] = w["decoder_norm.weight"] * np.float32(2.0 ** -12)
    om = env["O"].OracleDepthformer(w, env["ocfg"], mode="fp16")
    e = _embs(om, 16, env["cfg"].d_model)
    m = env["mrt_df"].Depthformer(w, env["cfg"], dtype="fp16")
    got = m.new_state(max_frames=1).depth_forward_full(torch.tensor(e, device="cuda").half()).cpu().numpy()
    m.close()
    exp = om.depth_forward_full(e).astype(np.float64)
    assert np.linalg.norm(got - exp) <= 4e-3 * np.linalg.norm(exp)
