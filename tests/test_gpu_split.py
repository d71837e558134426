"""The fp32 encoder on operands split into three bf16 parts (GEMMs) and on the
fp32 matrix instruction (attention), against the fp32 oracle."""

from __future__ import annotations

import dataclasses

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# 2 layers of 6 products of at most 192 terms: two orders of an fp32 sum of n
# terms differ by about sqrt(n) 2^-24 of its size, 12 x sqrt(192) x 6e-8 = 1e-5
# if every product's differences added up.
TOL = 1e-5


def rel(a, b):
    return float(np.linalg.norm(np.asarray(a, np.float64) - b) / np.linalg.norm(np.asarray(b, np.float64)))


def test_encoder_output_of_any_alignment(gpu_available):
    """An fp32 encoder output that the caller passes may start at any float."""
    import mrt_df
    import synth_bundle
    import torch
    cfg = mrt_df.Config.tiny(8)
    m = mrt_df.Depthformer(synth_bundle.make_weights(cfg, seed=3, norm_jitter=0.1), cfg, dtype="fp32")
    st = m.new_state(max_frames=1, enc_len=33)
    n = 2 * 33 * cfg.d_model
    flat = torch.randn(n + 4, device="cuda")
    x = torch.randn((2, cfg.d_model), device="cuda")
    outs = []
    for off in range(4):
        enc = flat[off:off + n]
        enc.copy_(torch.arange(n, device="cuda") % 97 / 97.0 - 0.5)
        st.reset_cache("temporal")
        outs.append(st.temporal_step(x, 0, enc_out=enc.view(2, 33, cfg.d_model)).cpu())
        assert torch.equal(outs[-1], outs[0]), off
    st.close()
    m.close()


@pytest.mark.parametrize("ffn_scale", [1.0, 2.0 ** 40])
@pytest.mark.parametrize("S", [1, 33, 63, 64, 65, 127, 129, 200])
def test_encode_edges(gpu_available, S, ffn_scale):
    """Context lengths at the edges of the 64-row tile (the one that these widths take)
    and of the key tile pairs, and hidden FFN values far outside the range of 16-bit
    floats."""
    import mrt_df
    import synth_bundle
    from oracle import depthformer_oracle as O
    cfg = dataclasses.replace(mrt_df.Config.tiny(8), max_encoder_length=200)
    w = synth_bundle.make_weights(cfg, seed=3, norm_jitter=0.1)
    for i in range(cfg.num_encoder_layers):
        w[f"encoder_layers.{i}.ffn.wi_1.weight"] = w[f"encoder_layers.{i}.ffn.wi_1.weight"] * np.float32(ffn_scale)
        w[f"encoder_layers.{i}.ffn.wo.weight"] = w[f"encoder_layers.{i}.ffn.wo.weight"] / np.float32(ffn_scale)
    tok = np.random.default_rng(S).integers(0, cfg.vocab_size, (2, S)).astype(np.int32)
    m = mrt_df.Depthformer(w, cfg, dtype="fp32")
    st = m.new_state(max_frames=1, enc_len=S)
    st.encode(tok)
    om = O.OracleDepthformer(w, O.DepthformerConfig(**dataclasses.asdict(cfg)), mode="fp32")
    enc = om.encode(tok)
    assert rel(st.read(mrt_df.BUF_ENC_OUT).cpu().numpy(), enc) <= TOL
    k, v = om.precompute_cross_kv(enc)[-1]
    assert rel(st.read(mrt_df.BUF_CROSS_K, cfg.num_temporal_layers - 1).cpu().numpy(), k) <= TOL
    assert rel(st.read(mrt_df.BUF_CROSS_V, cfg.num_temporal_layers - 1).cpu().numpy(), v) <= TOL
    st.close()
    m.close()
