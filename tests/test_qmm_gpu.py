"""int4 g64 few-row qmm on the GPU against the CPU oracle (fp32 dequant + matmul).

Reference cases: the verify qmv (Sources/Ingot/Shaders/verify_nax.metal:102-176) is checked in the reference against a
CPU matmul of the dequantised weights (Tests/IngotTests/KernelHarness.swift:95-115,189-195) and for row invariance
(KernelCaseTests.swift:66-86, qmv4-rows at :614-621).
"""
import numpy as np
import pytest

import oracle
from ingot_amd._lib import QMat, lib, check
from synth import rng, int4_matrix, bf16_normal, cosine

pytestmark = pytest.mark.gpu

# fp32 accumulation on both sides: the GPU sums per group of 64 on MFMA, the oracle in 16 interleaved lanes.
REL_TOL = 2e-5


def run_qmm(ctx, W, xb, M, out_mode=0, y0=None):
    K = W.K
    dx = ctx.to_device(xb)
    if out_mode == 2:
        dy = ctx.buffer(M * W.N * 2)
    else:
        dy = ctx.to_device(y0.astype(np.float32)) if y0 is not None else ctx.buffer(M * W.N * 4).fill(0)
    check(lib().ih_qmm_int4(ctx.handle, W.handle, dx.ptr, K, M, dy.ptr, W.N, out_mode))
    ctx.sync()
    out = dy.download(np.uint16 if out_mode == 2 else np.float32, (M, W.N))
    dx.free()
    dy.free()
    return out


@pytest.mark.parametrize(
    "M,N,K,seed",
    [
        (8, 4096, 4096, 0),      # benchmark configuration 0
        (1, 256, 2048, 1),
        (5, 512, 4096, 2),
        (16, 1024, 1024, 3),
        (17, 6144, 4096, 4),     # config 1 qkv at k = 16
        (32, 256, 768, 5),
        (18, 512, 1024, 8),      # token 16 on VALU, tokens 17+ on the second MFMA tile
        (17, 1000, 2880, 6),     # K % 128 == 64 (config 4 hidden), N not a multiple of 16
        (17, 5120, 2880, 9),     # 23 K-blocks in one split of 8 waves × 3: the last wave's third block is past K
        (5, 32768, 2880, 10),    # the same with 4 row tiles per wave (vocabulary-sized N)
        (32, 512, 2880, 12),     # the same with two 16-token tiles (M = 32)
        (3, 4096, 14336, 7),     # down projection K
    ],
)
def test_qmm_matches_oracle(ctx, M, N, K, seed):
    g = rng(seed)
    w, s, b = int4_matrix(g, N, K)
    xb, xf = bf16_normal(g, (M, K))
    W = QMat.int4(ctx, w, s, b)
    try:
        got = run_qmm(ctx, W, xb, M)
    finally:
        W.free()
    ref = oracle.qmm_int4(xf, w, s, b)
    err = np.abs(got - ref).max()
    assert np.isfinite(got).all()
    assert err <= REL_TOL * np.abs(ref).max() + 1e-6, f"max-abs {err} vs scale {np.abs(ref).max()}"
    assert cosine(got, ref) >= 0.999999


def test_qmm_bf16_out_and_accumulate(ctx):
    g = rng(11)
    M, N, K = 8, 512, 2048
    w, s, b = int4_matrix(g, N, K)
    xb, xf = bf16_normal(g, (M, K))
    y0 = g.normal(0, 3, size=(M, N)).astype(np.float32)
    W = QMat.int4(ctx, w, s, b)
    try:
        got16 = run_qmm(ctx, W, xb, M, out_mode=2)
        gotacc = run_qmm(ctx, W, xb, M, out_mode=1, y0=y0)
    finally:
        W.free()
    ref = oracle.qmm_int4(xf, w, s, b)
    # bf16 output: within one bf16 ulp of the fp32 reference (plus the fp32 accumulation difference).
    g16 = oracle.bf16_to_f32(got16)
    assert np.all(np.abs(g16 - ref) <= np.abs(ref) * 2.0 ** -8 + 1e-4)
    assert np.abs(gotacc - (y0 + ref)).max() <= REL_TOL * np.abs(ref).max() + 1e-5


def test_qmm_row_invariance(ctx):
    """Row r gives the same bits whatever M and whatever its neighbours (KernelCaseTests.swift:66-86)."""
    g = rng(21)
    N, K = 2048, 4096
    w, s, b = int4_matrix(g, N, K)
    xb, _ = bf16_normal(g, (17, K))
    other, _ = bf16_normal(g, (17, K))
    W = QMat.int4(ctx, w, s, b)
    try:
        full = run_qmm(ctx, W, xb, 17)
        for m in (1, 2, 8, 16):
            part = run_qmm(ctx, W, np.ascontiguousarray(xb[:m]), m)
            assert np.array_equal(part.view(np.uint32), full[:m].view(np.uint32)), f"M={m}"
        mixed = xb.copy()
        mixed[5:] = other[5:]
        got = run_qmm(ctx, W, mixed, 17)
        assert np.array_equal(got[:5].view(np.uint32), full[:5].view(np.uint32))
        # Repeated launches give the same bits (fixed split-K order).
        again = run_qmm(ctx, W, xb, 17)
        assert np.array_equal(again.view(np.uint32), full.view(np.uint32))
    finally:
        W.free()


def test_qmm_rejects_bad_shapes(ctx):
    g = rng(3)
    w, s, b = int4_matrix(g, 64, 128)
    W = QMat.int4(ctx, w, s, b)
    try:
        dx = ctx.buffer(33 * 128 * 2)
        dy = ctx.buffer(33 * 64 * 4)
        assert lib().ih_qmm_int4(ctx.handle, W.handle, dx.ptr, 128, 33, dy.ptr, 64, 0) == 1
        assert lib().ih_qmm_int4(ctx.handle, W.handle, dx.ptr, 64, 4, dy.ptr, 64, 0) == 1
        assert lib().ih_qmm_int4(ctx.handle, W.handle, dx.ptr, 128, 4, dy.ptr, 64, 7) == 1
        dx.free()
        dy.free()
    finally:
        W.free()


# Every launch shape the verify step of config 1 uses (qkv, o, gate|up, down, head) at B = 1, 8 and 17.
CFG1_SHAPES = [(6144, 4096), (4096, 4096), (28672, 4096), (4096, 14336), (151936, 4096)]


@pytest.mark.parametrize("N,K", CFG1_SHAPES)
def test_qmm_config1_shapes(ctx, N, K):
    g = rng(N + K)
    w, s, b = int4_matrix(g, N, K)
    xb, xf = bf16_normal(g, (17, K))
    W = QMat.int4(ctx, w, s, b)
    try:
        ref = oracle.qmm_int4(xf, w, s, b)
        full = run_qmm(ctx, W, xb, 17)
        assert np.isfinite(full).all()
        err = np.abs(full - ref).max()
        assert err <= REL_TOL * np.abs(ref).max() + 1e-6, err
        for m in (1, 8, 16):
            part = run_qmm(ctx, W, np.ascontiguousarray(xb[:m]), m)
            assert np.array_equal(part.view(np.uint32), full[:m].view(np.uint32)), m
    finally:
        W.free()


# Just above 512 row tiles (a count that four, two and one divides; whole K, a short K and a K-block count no shape tiles)
# and K split over workgroups of four and of two row tiles.
# 31 and 29 K-blocks: no exact shape, and two and four row tiles would split K over different waves.
TILED = [(8256, 4096), (8224, 4096), (8208, 2048), (8320, 2048), (16448, 1472), (16384, 3968), (16384, 3648), (4096, 12288), (4096, 10240), (1024, 8192),
         (3072, 6144)]


@pytest.mark.parametrize("N,K", TILED)
def test_qmm_row_tiles_and_k_splits(ctx, N, K):
    test_qmm_config1_shapes(ctx, N, K)


# K-block counts that no exact launch shape tiles: below, at and above the spans of the ragged shapes (16, 32, 48, 64 and
# 112 K-blocks; 16, 24, 32, 64 for vocabulary-sized N), a half block at the end, K split over two workgroups.
RAGGED = [(100, 64), (272, 64 * 5), (1000, 128 * 7), (2880, 64 * 65), (4112, 128 * 47), (300, 64 * 127), (272, 64 * 131),
          (5000, 128 * 33), (33000, 64 * 7), (32768, 64 * 51), (320, 128 * 113), (272, 64 * 449)]


@pytest.mark.parametrize("N,K", RAGGED)
def test_qmm_ragged_rows_at_any_alignment(ctx, N, K):
    """Every output form on bf16 rows that start at any element and are any distance apart, with NaN in the elements
    between them (they are never part of a sum), against the oracle; a row's bits depend neither on M nor on where the
    rows lie."""
    g = rng(N + K)
    w, s, b = int4_matrix(g, N, K)
    xb, xf = bf16_normal(g, (32, K))
    y0 = g.normal(0, 3, size=(32, N)).astype(np.float32)
    W = QMat.int4(ctx, w, s, b)
    try:
        ref = oracle.qmm_int4(xf, w, s, b)
        tol = REL_TOL * np.abs(ref).max() + 1e-6
        first = None
        for M in (1, 16, 17, 18, 32):
            for off, pad in ((0, 0), (0, 8), (8, 64), (1, 0), (0, 3)):
                ld = K + pad
                host = np.full(off + M * ld + 64, 0x7FC0, np.uint16)
                for r in range(M):
                    host[off + r * ld: off + r * ld + K] = xb[r]
                dx = ctx.to_device(host)
                for mode in (0, 1, 2):
                    dy = ctx.to_device(y0[:M]) if mode == 1 else ctx.buffer(M * N * (2 if mode == 2 else 4)).fill(0)
                    check(lib().ih_qmm_int4(ctx.handle, W.handle, dx.ptr + 2 * off, ld, M, dy.ptr, N, mode))
                    ctx.sync()
                    got = dy.download(np.uint16 if mode == 2 else np.float32, (M, N))
                    dy.free()
                    if mode == 0:
                        assert np.abs(got - ref[:M]).max() <= tol, (M, off, pad)
                        if first is None:
                            first = got
                        assert np.array_equal(got[0].view(np.uint32), first[0].view(np.uint32)), (M, off, pad)
                        plain = got
                    elif mode == 1:  # the sum of two fp32 values, rounded once
                        assert np.array_equal(got, y0[:M] + plain), (M, off, pad)
                    else:
                        assert np.array_equal(got, oracle.f32_to_bf16(plain)), (M, off, pad)
                dx.free()
    finally:
        W.free()


@pytest.mark.parametrize("mode", [0, 1, 2])
def test_qmm_output_over_its_own_rows(ctx, mode):
    """y in x's memory: every row is read before any output is stored, so the bits are those of separate buffers."""
    g = rng(31)
    M, N, K = 17, 4096, 4096
    w, s, b = int4_matrix(g, N, K)
    xb, _ = bf16_normal(g, (M, K))
    W = QMat.int4(ctx, w, s, b)
    dt = np.uint16 if mode == 2 else np.float32
    host = np.zeros(2 * M * K, np.uint16)  # room for fp32 rows; x is its first half
    host[:M * K] = xb.reshape(-1)
    y0 = host[:M * N * (1 if mode == 2 else 2)].view(dt).reshape(M, N)
    try:
        want = run_qmm(ctx, W, xb, M, out_mode=mode, y0=y0 if mode == 1 else None)
        dx = ctx.to_device(host)
        check(lib().ih_qmm_int4(ctx.handle, W.handle, dx.ptr, K, M, dx.ptr, N, mode))
        ctx.sync()
        got = dx.download(dt, (M, N))
        dx.free()
    finally:
        W.free()
    assert np.array_equal(got.view(np.uint8), want.view(np.uint8))


@pytest.mark.parametrize("N,K", [x for x in CFG1_SHAPES if x != (151936, 4096)] + TILED)
def test_qmm_more_rows_than_a_block(ctx, N, K):
    """18 … 32 rows through every launch shape: the first 17 rows have the bits of the 17-row product, the others those
    of a product of their own."""
    g = rng(N + K + 1)
    w = g.integers(0, 2**32, size=(N, K // 8), dtype=np.uint32)
    s = oracle.f32_to_bf16(np.abs(g.normal(0, 0.02, size=(N, K // 64))).astype(np.float32))
    xb, _ = bf16_normal(g, (32, K))
    W = QMat.int4(ctx, w, s, oracle.f32_to_bf16(-8.0 * oracle.bf16_to_f32(s)))
    try:
        want = np.concatenate([run_qmm(ctx, W, xb[:17].copy(), 17), run_qmm(ctx, W, xb[17:].copy(), 15)])
        assert np.isfinite(want).all()
        for m in (18, 32):
            got = run_qmm(ctx, W, xb[:m].copy(), m)
            assert np.array_equal(got.view(np.uint32), want[:m].view(np.uint32)), m
            got = run_qmm(ctx, W, xb[:m].copy(), m, out_mode=2)
            assert np.array_equal(got, oracle.f32_to_bf16(want[:m])), m
    finally:
        W.free()
