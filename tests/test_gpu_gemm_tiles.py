"""The encoder's matrix-core GEMM, tile by tile, against exact sums.

Operands are small integers (times a power of two), so every sum is exact in fp32 in
any order and the results have to be equal bit for bit.  For the split fp32 GEMM one
operand has 18 bits, which fills all three of its parts.  Row counts: 1, one less and
one more than the tile, and enough for one to three tiles a block with a last row
tile of one row; the rows past the last are not written.
"""

from __future__ import annotations

import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TILES = {"bf16": [(256, 256), (192, 256), (128, 256), (128, 192), (64, 128)],
         "fp32": [(128, 192), (128, 128), (64, 128)]}
TILES["fp16"] = TILES["bf16"]
STORE, RESID, GEGLU, CROSS, STORE_F32, GEGLU_SPLIT = range(6)
CODE = {"fp32": 0, "bf16": 1, "fp16": 2}
N, CUS = 768, 256
CASES = [(d, t) for d in ("bf16", "fp16", "fp32") for t in range(len(TILES[d]))]


@pytest.fixture(scope="module")
def gemm(gpu_available):
    import mrt_df
    import torch
    lib = mrt_df.load_library()
    vp, i32 = ctypes.c_void_p, ctypes.c_int
    lib.mrt_test_gemm.argtypes = [i32, i32, vp, vp] + [i32] * 9 + [vp, ctypes.POINTER(i32)]
    lib.mrt_test_gemm.restype = i32

    def run(dtype, path, A, B, kind, C, tile=-1, nb=1, H=1, S=1):
        taken = i32(-9)
        torch.cuda.synchronize()
        rc = lib.mrt_test_gemm(CODE[dtype], path, A.data_ptr(), B.data_ptr(), A.shape[0], B.shape[0], A.shape[1], kind,
                               tile, nb, H, S, 64 * H, C.data_ptr(), ctypes.byref(taken))
        if rc:
            raise mrt_df.MrtError(rc, lib.mrt_last_error().decode())
        return taken.value

    run.dt = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
    return run


def operands(dtype, M, K, scale=1.0, n=N):
    import torch
    g = torch.Generator(device="cuda").manual_seed(1000 * M + K)

    def ints(shape, top):
        return torch.randint(-top, top + 1, shape, generator=g, device="cuda").float()

    if dtype == "fp32":  # the wide operand is A for odd M, B for even M
        wide, small = (1 << 17) - 1, 1
        return (ints((M, K), wide if M % 2 else small) * scale, ints((n, K), small if M % 2 else wide))
    return ints((M, K), 3) * scale, ints((n, K), 3)


def rows(dtype, tile):
    bm, bn = TILES[dtype][tile]
    return [1, bm - 1, bm + 1] + [bm * -(-int(x * CUS) // (N // bn)) + 1 for x in (1.6, 2.5)]


def path_of(dtype):
    return 2 if dtype == "fp32" else 0


@pytest.mark.parametrize("kind", [STORE, RESID, STORE_F32, CROSS])
@pytest.mark.parametrize("dtype,tile", CASES)
def test_tiles(gemm, dtype, tile, kind):
    import torch
    dt = gemm.dt[dtype]
    for M in rows(dtype, tile):
        for K in ((32, 160) if dtype == "fp32" else (64, 320)):
            A, B = operands(dtype, M, K)
            acc = (A.double() @ B.double().T).float()
            out = torch.float32 if kind == STORE_F32 else dt
            C = torch.randint(-4, 5, (M + 2, N), device="cuda").to(out)
            want = C.clone()
            nb = 2 if M % 2 == 0 else 1
            kw = {}
            if kind == RESID:
                want[:M] = (want[:M].float() + acc.to(dt).float()).to(dt)
            elif kind == CROSS:  # one layer: k and v of 6 heads
                kw = dict(nb=nb, H=6, S=M // nb)
                want.view(-1)[:M * N] = acc.view(nb, M // nb, 2, 6, 64).permute(2, 0, 3, 1, 4).reshape(-1).to(dt)
            else:
                want[:M] = acc.to(dt).to(out)
            gemm(dtype, path_of(dtype), A.to(dt), B.to(dt), kind, C, tile, **kw)
            assert torch.equal(C, want), (M, K)


@pytest.mark.parametrize("dtype,tile", [c for c in CASES if TILES[c[0]][c[1]][1] != 192])
def test_gated_gelu_tiles(gemm, dtype, tile):
    """Gate and up columns in groups of 32, on exact sums: the 16-bit epilogue equals the
    vector-ALU GEMM's; the fp32 one is within 8 x 2^-24 |gate up| of 64 bits (tanhf 2 steps
    of 1, its argument 1.5, 1 + tanh 1, halved, and the products' roundings 3)."""
    import torch
    dt = gemm.dt[dtype]
    for M in rows(dtype, tile):
        for K in ((32, 160) if dtype == "fp32" else (64, 320)):
            A, B = operands(dtype, M, K, 2.0 ** -18 if dtype == "fp32" else 2.0 ** -5)
            A, B = A.to(dt), B.to(dt)
            if dtype == "fp32":
                C = torch.full((M + 2, N // 64, 3, 32), 7, dtype=torch.bfloat16, device="cuda")
                gemm(dtype, 2, A, B, GEGLU_SPLIT, C, tile)
                got = C[:M].double().sum(2).view(M, N // 2)
                acc = (A.double() @ B.double().T).view(M, N // 64, 2, 32)
                g, u = (acc[:, :, i].reshape(M, N // 2) for i in (0, 1))
                want = 0.5 * g * (1 + torch.tanh(0.7978845608028654 * (g + 0.044715 * g ** 3))) * u
                assert bool(((got - want).abs() <= 8 * 2.0 ** -24 * (g * u).abs() + 1e-37).all()), (M, K)
            else:
                C = torch.full((M + 2, N // 2), 7, dtype=dt, device="cuda")
                gemm(dtype, 0, A, B, GEGLU, C, tile)
                want = torch.zeros((M, N // 2), dtype=dt, device="cuda")
                gemm(dtype, 1, A, B, GEGLU, want)
                assert torch.equal(C[:M], want), (M, K)
            assert bool((C[M:] == 7).all())


@pytest.mark.parametrize("dtype", ["bf16", "fp16"])
def test_gated_gelu_of_every_value(gemm, dtype):
    """Every finite 16-bit gate value, up = 1: the matrix-core epilogue's tanh against
    tanhf."""
    import torch
    dt = gemm.dt[dtype]
    bits = torch.arange(-32768, 32768, device="cuda").to(torch.int16)
    x = bits.view(dt)
    x = x[torch.isfinite(x)]
    A = torch.zeros((len(x), 64), dtype=dt, device="cuda")
    A[:, 0], A[:, 1] = x, 1
    B = torch.zeros((128, 64), dtype=dt, device="cuda")
    gate = torch.arange(128, device="cuda") % 64 < 32
    B[gate, 0], B[~gate, 1] = 1, 1
    got, want = torch.zeros((len(x), 64), dtype=dt, device="cuda"), torch.zeros((len(x), 64), dtype=dt, device="cuda")
    gemm(dtype, 0, A, B, GEGLU, got)
    gemm(dtype, 1, A, B, GEGLU, want)
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))


@pytest.mark.parametrize("tile", range(3))
@pytest.mark.parametrize("M,K", [(5, 32), (200, 160)])
def test_split_gemm_not_finite(gemm, M, K, tile):
    """Infinities, NaN and overflow of fp32 operands give what fp32 products give: an
    infinite element meets weights with one, two and three parts of both signs."""
    import torch
    g = torch.Generator(device="cuda").manual_seed(M)
    A = torch.randn((M, K), generator=g, device="cuda")
    B = torch.randn((N, K), generator=g, device="cuda")
    B[1::3] = B[1::3].bfloat16().float()  # their second and third parts are zero
    B[2::3, 3] = 0
    inf, big = float("inf"), 3.0e38
    A[0, 3], A[1, 7], A[2, 0], A[3, K - 1] = inf, -inf, float("nan"), big
    A[4, 3], A[4, 9] = inf, -inf
    B[5, 7], B[6, 1] = inf, float("nan")
    C = torch.zeros((M, N), device="cuda")
    gemm("fp32", 2, A, B, STORE, C, tile)
    want = (A.double().cpu() @ B.double().cpu().T)
    want = torch.where(want.abs() > 3.4028235e38, torch.sign(want) * inf, want)
    got = C.double().cpu()
    assert torch.equal(torch.isnan(got), torch.isnan(want))
    assert torch.equal(torch.isinf(got), torch.isinf(want))
    assert torch.equal(got[torch.isinf(want)], want[torch.isinf(want)])
    ok = torch.isfinite(want)
    scale = A.double().abs().nan_to_num(0, 0, 0).cpu() @ B.double().abs().nan_to_num(0, 0, 0).cpu().T
    assert bool(((got - want)[ok].abs() <= 2.0 ** -22 * scale[ok]).all())


@pytest.mark.parametrize("kind", [STORE, RESID, STORE_F32, GEGLU])
@pytest.mark.parametrize("dtype", ["bf16", "fp16"])
def test_sequential_skinny_gemm(gemm, dtype, kind):
    """The skinny GEMM of the full-sequence depth pass sums every output as the encoder's
    GEMM does: bit for bit, on random operands, at the edges of its 16-row tiles and of
    its runs of 16 k-steps, and with two column tiles a wave (16,384 columns)."""
    import torch
    dt = gemm.dt[dtype]
    g = torch.Generator(device="cuda").manual_seed(7)
    for M, K, n in [(1, 64, 128), (15, 512, 384), (16, 576, 128), (17, 1024, 384), (32, 1088, 128), (33, 2816, 128),
                    (64, 2112, 256), (17, 1088, 16384), (1, 64, 16384)]:
        A = torch.randn((M, K), generator=g, device="cuda").to(dt)
        B = (torch.randn((n, K), generator=g, device="cuda") / K ** 0.5).to(dt)
        out = torch.float32 if kind == STORE_F32 else dt
        cols = n // 2 if kind == GEGLU else n
        want = torch.randn((M, cols), generator=g, device="cuda").to(out)
        mp = -(-M // 16) * 16
        C = torch.full((mp + 1, cols), 7, device="cuda", dtype=out)
        if kind == RESID:
            C[:M] = want
        gemm(dtype, 0, A, B, kind, want)
        gemm(dtype, 3, A, B, kind, C)
        if kind == GEGLU:  # 16-row x 32-column tiles: (column group of 8, row, 8)
            assert bool((C[mp:] == 7).all())
            C = C[:mp].reshape(mp // 16, cols // 32, 4, 16, 8).permute(0, 3, 1, 2, 4).reshape(mp, cols)
        assert torch.equal(C[:M], want), (M, K, n)
        assert bool((C[M:] == 7).all())


def test_sequential_skinny_gemm_odd_columns(gemm):
    """A last column tile by itself, and one partly filled; exact sums."""
    import torch
    for n in (16400, 16390, 24):
        A, B = operands("bf16", 33, 1088, n=n)
        C = torch.full((35, n), 7, device="cuda", dtype=torch.float32)
        gemm("bf16", 3, A.bfloat16(), B.bfloat16(), STORE_F32, C)
        want = (A.double() @ B.double().T).float().bfloat16().float()
        assert torch.equal(C[:33], want) and bool((C[33:] == 7).all()), n


@pytest.mark.parametrize("dtype,M,n,kind,tile", [
    ("bf16", 64384, 5632, GEGLU, 0), ("bf16", 2012, 5632, GEGLU, 1), ("bf16", 8048, 1024, RESID, 2),
    ("bf16", 2012, 3072, STORE, 3), ("bf16", 2012, 1024, RESID, 4), ("fp32", 2012, 3072, STORE, 0),
    ("fp32", 2012, 5632, GEGLU_SPLIT, 1), ("fp32", 2012, 1024, RESID, 2), ("bf16", 256, 40960, STORE, 0),
    ("bf16", 28168, 5632, GEGLU, 0), ("bf16", 50300, 3072, STORE, 0), ("bf16", 41600, 5632, GEGLU, 1)])
def test_rule(gemm, dtype, M, n, kind, tile):
    """The tile that the rule takes for shapes of the encoder at the benchmark dims (256
    CUs): one of each, and shapes at which the next smaller tile measured 9 to 32 %
    slower."""
    import torch
    K = 64
    A, B = (torch.zeros((r, K), dtype=gemm.dt[dtype], device="cuda") for r in (M, n))
    C = torch.zeros((M, n * (3 if kind == GEGLU_SPLIT else 1)), dtype=gemm.dt[dtype], device="cuda")
    assert gemm(dtype, path_of(dtype), A, B, kind, C) == tile


def test_refused_kinds(gemm):
    """fp32 pairs are written split, and only by the split GEMM: the store count that its
    waits rely on is that of the split epilogue."""
    import mrt_df
    import torch
    A = torch.zeros((64, 64), device="cuda")
    B = torch.zeros((128, 64), device="cuda")
    C = torch.zeros((64, 128 * 3), device="cuda")
    with pytest.raises(mrt_df.MrtError, match="split"):
        gemm("fp32", 2, A, B, GEGLU, C)
    for dtype, path in (("fp32", 0), ("fp32", 1), ("bf16", 0)):
        with pytest.raises(mrt_df.MrtError, match="split"):
            gemm(dtype, path, A.to(gemm.dt[dtype]), B.to(gemm.dt[dtype]), GEGLU_SPLIT, C)
    for tile in (5, 99):
        with pytest.raises(mrt_df.MrtError, match="tile"):
            gemm("bf16", 0, A.bfloat16(), B.bfloat16(), STORE, C, tile)
