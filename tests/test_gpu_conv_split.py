"""The codec's convolutions on split operands at the edges of their tiles and
K splits, against the fp32 oracle."""

from __future__ import annotations

import numpy as np
import pytest

import synth_bundle
from oracle import codec_oracle as C

pytestmark = pytest.mark.gpu

# Every value is a chain of 18 convolutions whose fp32 sums of up to 9,216 terms
# differ between orders by about sqrt(9216) 2^-24 = 6e-6 of their size in the
# largest, 1.5e-6 in the others: 6e-6 + sqrt(17) x 1.5e-6 = 1.2e-5.
TOL = 1.2e-5


def rel(a, b):
    return float(np.linalg.norm(np.asarray(a, np.float64) - b) / np.linalg.norm(np.asarray(b, np.float64)))


@pytest.fixture(scope="module")
def full():
    import mrt_df
    w = synth_bundle.make_codec_weights(synth_bundle.CodecShape.reference())
    codec = mrt_df.Codec(w, max_frames=17)
    yield w, codec
    codec.close()


@pytest.mark.parametrize("frames", [1, 2, 3, 11, 17])
def test_frame_counts(gpu_available, full, frames):
    """Pixel counts that fill no tile, with 1 to 16 slices of the sums; a second
    decode finds the slice counters as the first did."""
    import mrt_df
    w, codec = full
    tok = np.random.default_rng(frames).integers(0, 1024, (frames, 16)).astype(np.int32)
    rec = {}
    ref = C.OracleCodec(w, C.CodecConfig.reference(), "fp32").decode(tok, rec)
    first = codec.decode(tok)
    assert rel(first, ref) <= TOL
    for i in range(7):
        assert rel(codec.read(mrt_df.CODEC_BUF_BLOCK0 + i, rec[f"block{i}"].shape), rec[f"block{i}"]) <= TOL
    np.testing.assert_array_equal(codec.decode(tok), first)


def test_infinite_activations(gpu_available):
    """One frame whose first projection overflows: every residual of it is -inf from
    there on and every ELU of one is -1, so the audio is finite, as the oracle has it.
    (An infinite activation meets weights of three parts with both signs.)"""
    import mrt_df
    w = synth_bundle.make_codec_weights(synth_bundle.CodecShape.reference())
    w = {k: np.array(v) for k, v in w.items()}
    w["codebooks"][:, :, 0] = 0
    w["codebooks"][0, 5, 0] = 4.0
    w["input_proj.conv1.weight"][0] = 0
    w["input_proj.conv1.weight"][0, 0] = 3e38
    w["input_proj.conv2.weight"][:, 0] = -np.abs(w["input_proj.conv2.weight"][:, 0]) - 1e-3
    for k in w:
        if k.startswith("decoder_blocks") and k.endswith("shortcut.weight"):
            w[k] = np.abs(w[k]) + 1e-4
    tok = np.random.default_rng(3).integers(6, 1024, (4, 16)).astype(np.int32)
    tok[2, 0] = 5
    rec = {}
    with np.errstate(all="ignore"):
        ref = C.OracleCodec(w, C.CodecConfig.reference(), "fp32").decode(tok, rec)
    assert np.isfinite(ref).all() and np.isneginf(rec["block6"]).any()
    codec = mrt_df.Codec(w, max_frames=4)
    got = codec.decode(tok)
    last = codec.read(mrt_df.CODEC_BUF_BLOCK0 + 6, rec["block6"].shape)
    codec.close()
    assert np.isfinite(got).all() and rel(got, ref) <= TOL
    np.testing.assert_array_equal(np.isneginf(last), np.isneginf(rec["block6"]))
