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
