"""The encoder prefill through the persistent GEMM, whole: small widths, which take its
64 x 128 tile (test_gpu_gemm_tiles.py has every tile by itself)."""

from __future__ import annotations

import dataclasses

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# One bf16 rounding is 2^-9 of a value; a layer rounds its output about 4 times and
# the two layers' errors add in squares: sqrt(8) x 2^-9 = 5.5e-3, doubled for the
# rounded normalisations (fp16: 2^-12 a rounding).
TOL = {"bf16": 1.2e-2, "fp16": 1.5e-3}


@pytest.mark.parametrize("dtype", ["bf16", "fp16"])
@pytest.mark.parametrize("S", [1, 31, 33, 64, 65, 96, 97, 129, 200])
def test_encode_edges(gpu_available, S, dtype):
    """Row counts 2 S at the edges of the 64-row tile and of the 32-row matrix
    instruction, against the oracle; a second encode finds the buffers of the first."""
    import mrt_df
    import synth_bundle
    from oracle import depthformer_oracle as O
    cfg = dataclasses.replace(mrt_df.Config.tiny(8), max_encoder_length=200)
    w = synth_bundle.make_weights(cfg, seed=3, norm_jitter=0.1)
    tok = np.random.default_rng(S).integers(0, cfg.vocab_size, (2, S)).astype(np.int32)
    m = mrt_df.Depthformer(w, cfg, dtype=dtype)
    st = m.new_state(max_frames=1, enc_len=S)
    om = O.OracleDepthformer(w, O.DepthformerConfig(**dataclasses.asdict(cfg)), mode=dtype)
    enc = om.encode(tok)
    for _ in range(2):
        st.encode(tok)
        got = st.read(mrt_df.BUF_ENC_OUT).float().cpu().numpy()
        assert np.linalg.norm(got - enc) <= TOL[dtype] * np.linalg.norm(enc)
    st.close()
    m.close()


def test_many_rows_equal_few(gpu_available):
    """Rows do not depend on the rows beside them: 32 streams (several tiles a block)
    against one stream, bit for bit."""
    import mrt_df
    import synth_bundle
    cfg = dataclasses.replace(mrt_df.Config.tiny(8), max_encoder_length=300)
    w = synth_bundle.make_weights(cfg, seed=4, norm_jitter=0.1)
    S = cfg.max_encoder_length
    tok = np.random.default_rng(5).integers(0, cfg.vocab_size, (64, S)).astype(np.int32)
    m = mrt_df.Depthformer(w, cfg, dtype="bf16")
    b = mrt_df.Batch(m, 32, max_frames=1, enc_len=S)
    b.encode(tok)
    got = b.read_enc_out().reshape(64, S, -1)
    st = m.new_state(max_frames=1, enc_len=S)
    for i in (0, 13, 31):
        st.encode(tok[2 * i:2 * i + 2])
        assert (st.read(mrt_df.BUF_ENC_OUT).reshape(2, S, -1) == got[2 * i:2 * i + 2]).all()
    b.close()
    st.close()
    m.close()
