"""Widths that the matrix-core GEMMs do not take: the vector-ALU GEMM, the scalar
encoder attention and the fp32 matrix instruction's convolution carry those, and rows
wider than the wave norm's registers go through the block norm."""

from __future__ import annotations

import dataclasses

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL = {"fp32": 1e-5, "bf16": 1.2e-2, "fp16": 1.5e-3}  # as the encoder tests of the matrix-core paths


def rel(a, b):
    return float(np.linalg.norm(np.asarray(a, np.float64) - b) / np.linalg.norm(np.asarray(b, np.float64)))


@pytest.mark.parametrize("dtype", ["fp32", "bf16", "fp16"])
@pytest.mark.parametrize("S", [1, 33, 65])
def test_encoder_of_odd_widths(gpu_available, dtype, S):
    """d_model 192 and 3 heads: no output width is a multiple of 128."""
    import mrt_df
    import synth_bundle
    from oracle import depthformer_oracle as O
    cfg = dataclasses.replace(mrt_df.Config.tiny(8), d_model=192, num_heads=3, d_ff=192, max_encoder_length=65)
    w = synth_bundle.make_weights(cfg, seed=5, norm_jitter=0.1)
    tok = np.random.default_rng(S).integers(0, cfg.vocab_size, (2, S)).astype(np.int32)
    om = O.OracleDepthformer(w, O.DepthformerConfig(**dataclasses.asdict(cfg)), mode=dtype)
    m = mrt_df.Depthformer(w, cfg, dtype=dtype)
    st = m.new_state(max_frames=1, enc_len=S)
    st.encode(tok)
    enc = om.encode(tok)
    assert rel(st.read(mrt_df.BUF_ENC_OUT).float().cpu().numpy(), enc) <= TOL[dtype]
    k, v = om.precompute_cross_kv(enc)[-1]
    last = cfg.num_temporal_layers - 1
    assert rel(st.read(mrt_df.BUF_CROSS_K, last).float().cpu().numpy(), k) <= TOL[dtype]
    assert rel(st.read(mrt_df.BUF_CROSS_V, last).float().cpu().numpy(), v) <= TOL[dtype]
    st.close()
    m.close()


def test_scalar_attention_after_nan(gpu_available):
    """The rows of a key tile that hold no keys do not take part, whatever the kernels
    before left in LDS: here an encode whose keys and values are all NaN."""
    import mrt_df
    import synth_bundle
    from oracle import depthformer_oracle as O
    cfg = dataclasses.replace(mrt_df.Config.tiny(8), d_model=192, num_heads=3, d_ff=192, max_encoder_length=64)
    w = synth_bundle.make_weights(cfg, seed=5, norm_jitter=0.1)
    bad = dict(w)
    for i in range(cfg.num_encoder_layers):
        k = f"encoder_layers.{i}.pre_attn_norm.weight"
        bad[k] = np.full_like(w[k], np.nan)
    om = O.OracleDepthformer(w, O.DepthformerConfig(**dataclasses.asdict(cfg)), mode="fp32")
    models = [mrt_df.Depthformer(x, cfg, dtype="fp32") for x in (bad, w)]
    states = [m.new_state(max_frames=1, enc_len=S) for m, S in zip(models, (64, 5))]
    tok = np.random.default_rng(1).integers(0, cfg.vocab_size, (2, 64)).astype(np.int32)
    exp = om.encode(tok[:, :5])
    for _ in range(4):
        states[0].encode(tok)
        states[1].encode(np.ascontiguousarray(tok[:, :5]))
        assert rel(states[1].read(mrt_df.BUF_ENC_OUT).cpu().numpy(), exp) <= TOL["fp32"]
    for x in states + models:
        x.close()


@pytest.mark.parametrize("ids", [1, 7, 31])
def test_style_model_of_odd_widths(gpu_available, ids):
    """Widths that are multiples of 16 and not of 32."""
    import mrt_df
    import synth_bundle
    from oracle import musiccoca_oracle as M
    cfg = dataclasses.replace(mrt_df.CocaConfig.tiny(), d_model=144, num_heads=3, d_head=16, d_ff=208,
                              pooler_d_head=48)
    w = synth_bundle.make_coca_weights(cfg)
    tok, pad = M.text_ids(np.random.default_rng(ids).integers(3, cfg.vocab_size, ids).tolist(), cfg.max_text_len)
    ref = M.OracleCoca(w, M.CocaConfig(**{f: getattr(cfg, f) for f in vars(M.CocaConfig())}), "fp32").embed_text(
        tok, pad, {})
    sm = mrt_df.StyleModel(w, cfg)
    for _ in range(2):
        assert rel(sm.embed_text(tok, pad), ref) <= 1e-5
    sm.close()


@pytest.mark.parametrize("D,B", [(576, 3), (768, 9), (2048, 1)])
def test_batched_streams_of_other_widths(gpu_available, D, B):
    """Batched streams whose rows the wave norm takes (2,048 columns) and does not (no
    multiples of 512), up to the widest that the sampler takes: teacher-forced logits
    within the bf16 parity bound of the oracle."""
    import torch
    import mrt_df
    import synth_bundle
    from oracle import depthformer_oracle as O
    F, L, C = 2, 16, 8
    cfg = dataclasses.replace(mrt_df.Config.tiny(C), d_model=D, num_encoder_layers=1, max_encoder_length=14)
    w = synth_bundle.make_weights(cfg, seed=6, norm_jitter=0.1)
    rng = np.random.default_rng(D + B)
    tok = rng.integers(2, 130, size=(2 * B, cfg.max_encoder_length)).astype(np.int32)
    teacher = (2 + C * np.arange(L) + rng.integers(0, C, size=(B, F, L))).astype(np.int32)
    kw = dict(num_frames=F, rvq_depth=L, temperature=1.1, top_k=4, guidance_weight=5.0, codebook_size=C,
              codec_offset=2)
    m = mrt_df.Depthformer(w, cfg, dtype="bf16")
    b = mrt_df.Batch(m, B, max_frames=F)
    sl = torch.zeros((F, L, 2 * B, C), dtype=torch.float32, device="cuda")
    b.generate_tokens(tok, mrt_df.GenOptions(seed=0, **kw), seeds=list(range(B)), teacher=teacher,
                      record=dict(slices=sl))
    sl = sl.cpu().numpy()
    b.close()
    om = O.OracleDepthformer(w, O.DepthformerConfig(**dataclasses.asdict(cfg)), mode="bf16")
    for s in {0, B - 1}:
        rec = {}
        O.generate_tokens(om, tok[2 * s:2 * s + 2], O.GenerateOptions(seed=s, **kw), teacher=teacher[s], record=rec)
        assert rel(sl[:, :, 2 * s:2 * s + 2], rec["slices"]) <= 2e-2
    m.close()


def test_wide_rows(gpu_available):
    """More than 4,096 columns: the prefill of a batch and the full-sequence depth pass."""
    import torch
    import mrt_df
    import synth_bundle
    from oracle import depthformer_oracle as O
    D = 4160
    cfg = dataclasses.replace(mrt_df.Config.tiny(8), d_model=D, num_encoder_layers=1, num_temporal_layers=1,
                              max_encoder_length=14)
    w = synth_bundle.make_weights(cfg, seed=6, norm_jitter=0.1)
    om = O.OracleDepthformer(w, O.DepthformerConfig(**dataclasses.asdict(cfg)), mode="bf16")
    rng = np.random.default_rng(D)
    m = mrt_df.Depthformer(w, cfg, dtype="bf16")
    tok = rng.integers(2, 130, size=(2, cfg.max_encoder_length)).astype(np.int32)
    b = mrt_df.Batch(m, 1, max_frames=1)
    b.encode(tok)
    assert rel(b.read_enc_out().float().cpu().numpy().reshape(2, -1, D), om.encode(tok)) <= TOL["bf16"]
    b.close()
    st = m.new_state(max_frames=1)
    embs = om.P.r(rng.standard_normal((2, 5, D)).astype(np.float32))
    full = st.depth_forward_full(torch.tensor(embs, device="cuda").bfloat16()).cpu().numpy()
    assert rel(full, om.depth_forward_full(embs)) <= 2e-2
    st.close()
    m.close()
