"""fp32 models against the same evaluated in 64 bits, at the benchmark dims: the
split GEMMs of the encoder and of the cross K/V may not cost precision that the
fp32 arithmetic had.  A temporal step shows it: the cross attention averages
the keys' independent roundings away and keeps what they have in common.

Bounds: 1.25 times the errors of fp32 products with an fp32 accumulator (a chain
of fused multiply-adds over K: temporal step 6.3e-7 at every context; encoder
1.33e-6 at 64 ids and 2.8e-6 at 517).  With all six products of the split operands
in one sum the temporal step shows 1.16e-6 and 1.33e-6.
"""

from __future__ import annotations

import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("path,enc_len,bound", [("temporal_step", 64, 7.9e-7), ("temporal_step", 517, 7.9e-7),
                                                ("encode", 64, 1.7e-6), ("encode", 517, 3.5e-6)])
def test_fp32_against_64_bits(gpu_available, path, enc_len, bound):
    from perf import cases
    c = dict(path=path, model="bench", dtype="fp32", enc_len=enc_len, pos=5)
    got, exact = cases.run(cases.prepare(c, 3)), cases.exact(c, 3)
    if path == "encode":
        got, exact = got["out"], exact["out"]
    err = float((got.double() - exact).norm() / exact.norm())
    print(f"{path} {enc_len}: {err:.3g}")
    assert err <= bound
