"""Widths off the main path: rows that the wave norm does not take go through the block
norm."""

from __future__ import annotations

import dataclasses

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL = {"fp32": 1e-5, "bf16": 1.2e-2, "fp16": 1.5e-3}  # as the encoder tests of the matrix-core paths


def rel(a, b):
    return float(np.linalg.norm(np.asarray(a, np.float64) - b) / np.linalg.norm(np.asarray(b, np.float64)))


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
