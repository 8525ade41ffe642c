"""GPU parity of the direct-to-LDS GEMM kernels at shapes that are not whole tiles: one
row, column or k past or short of a tile and of a K stage, operands and C at every
4-byte offset from a 16-byte boundary, C between guard floats that must keep their bits.

Bar: float64 on the same inputs with the reference's K-scaled tolerance (tol_gemm,
abs_tol_gemm); the fused launch bit-equal to the plain one followed by bias + activation.
"""
from __future__ import annotations

import numpy as np
import pytest

from tests.test_gpu_row_edges import _Out, _up

pytestmark = pytest.mark.gpu

TILES = [256, 128, 64, 32]


def _tile(m, t):
    return m.GemmTile(t, t, 32, t // 16, t // 16)


def _shapes(t):
    return [(1, t, 32), (t - 1, t + 1, 33), (t + 1, 2 * t - 1, 63), (t, t + 3, 64),
            (2 * t + 5, t, 95), (3, 2 * t + 2, 129), (t + 7, t + t // 2, 160),
            (5, t, 31), (5, t - 1, 64)]          # the last two: the staged kernel


@pytest.mark.parametrize("t", TILES)
def test_gemm_f32_tile_edges(gpu, orc, t):
    V = gpu.GemmVariant.kMfmaF32
    for M, N, K in _shapes(t):
        a = orc.fill_random(M * K, 11 + K).reshape(M, K)
        b = orc.fill_random(K * N, 12 + N).reshape(K, N)
        c = orc.fill_random(M * N, 13 + M).reshape(M, N)
        prod = a.astype(np.float64) @ b.astype(np.float64)
        for sa, sb, sc, alpha, beta in ((0, 0, 0, 1.0, 0.0), (1, 3, 2, -0.5, 1.5)):
            da, pa = _up(gpu, a, sa)
            db, pb = _up(gpu, b, sb)
            out = _Out(gpu, M * N, sc)
            full = out.buf.download()
            full[out.at:out.at + M * N] = np.nan if beta == 0.0 else c.ravel()
            out.buf.upload(full)
            st = gpu.launch_gemm_f32(pa, pb, out.ptr, M, N, K, alpha, beta, V, _tile(gpu, t))
            assert st.ok(), str(st)
            gpu.device_synchronize()
            want = alpha * prod + beta * c
            floor = max(1.0, abs(alpha)) * orc.abs_tol_gemm(K) + 2e-7 * abs(beta)
            r = orc.compare(out.get(), want.ravel(), orc.tol_gemm(K), floor)
            assert r.ok, f"{M}x{N}x{K} tile={t} shifts={sa},{sb},{sc}: {r}"
            del da, db


def _check_plain_and_fused(gpu, orc, shape, tile):
    M, N, K = shape
    V = gpu.GemmVariant.kMfmaF32
    a = orc.fill_random(M * K, 61 + K).reshape(M, K)
    b = orc.fill_random(K * N, 62 + N).reshape(K, N)
    c = orc.fill_random(M * N, 63 + M).reshape(M, N)
    bias = orc.fill_random(N, 64)
    prod = a.astype(np.float64) @ b.astype(np.float64)
    for sa, sb, sc, beta in ((0, 0, 0, 0.0), (1, 3, 2, 1.5)):
        da, pa = _up(gpu, a, sa)
        db, pb = _up(gpu, b, sb)
        out = _Out(gpu, M * N, sc)
        full = out.buf.download()
        full[out.at:out.at + M * N] = np.nan if beta == 0.0 else c.ravel()
        out.buf.upload(full)
        st = gpu.launch_gemm_f32(pa, pb, out.ptr, M, N, K, 0.75, beta, V, tile)
        assert st.ok(), str(st)
        gpu.device_synchronize()
        r = orc.compare(out.get(), (0.75 * prod + beta * c).ravel(), orc.tol_gemm(K),
                        orc.abs_tol_gemm(K) + 4e-7)
        assert r.ok, f"shifts={sa},{sb},{sc}: {r}"
        if beta == 0.0:
            dbias, pbias = _up(gpu, bias, 0)
            y, fused = _Out(gpu, M * N, 0), _Out(gpu, M * N, 0)
            for st in (gpu.launch_bias_act_f32(out.ptr, pbias, y.ptr, M, N, 3, 1),
                       gpu.launch_gemm_bias_act_f32(pa, pb, pbias, fused.ptr, M, N, K, 0.75, 3,
                                                    tile)):
                assert st.ok(), str(st)
            gpu.device_synchronize()
            assert np.array_equal(fused.get().view(np.uint32), y.get().view(np.uint32))
        del da, db


# 64 x 64 launches that run 128 x 64 tiles (1000 x 4096: four 64 x 64 tiles per CU) and
# 32 x 64 tiles (1531 x 1021: 1.5 per CU), whole and not.
@pytest.mark.parametrize("shape", [(1024, 4096, 64), (1000, 4093, 70), (901, 4096, 33),
                                   (1536, 1024, 96), (1531, 1021, 70), (1505, 1089, 32)],
                         ids=lambda s: "x".join(map(str, s)))
def test_64_tile_launch_picks(gpu, orc, shape):
    _check_plain_and_fused(gpu, orc, shape, _tile(gpu, 64))


# Launches of the small tiles that run the tile's own EDGE kernel: one 64 x 64 tile per CU,
# where 32 x 64 ones tie, and more 32 x 32 tiles than the few-tiles kernel takes.
OWN_EDGE = ([(64, (1000, 1023, k)) for k in (33, 64, 95, 161, 333)] +
            [(32, (500, 515, k)) for k in (64, 65, 95, 161, 319)])
# K of 32 to 63: with 16-byte operands (and at 32 x 32) the staged kernel, whole tiles of 64
# their own where 128 x 64 ones (960 rows) would not be whole.
SHORT_K = [(64, (996, 1020, 32)), (64, (996, 1020, 40)), (64, (960, 4096, 32)),
           (128, (260, 388, 32)), (256, (260, 516, 60)), (32, (500, 516, 60)), (32, (500, 515, 33))]


@pytest.mark.parametrize("t,shape", OWN_EDGE + SHORT_K,
                         ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else str(v))
def test_tile_own_kernels(gpu, orc, t, shape):
    _check_plain_and_fused(gpu, orc, shape, _tile(gpu, t))


@pytest.mark.parametrize("t", TILES)
@pytest.mark.parametrize("act", [0, 1, 2, 3])
def test_fused_tile_edges_match_the_pair(gpu, orc, t, act):
    V = gpu.GemmVariant.kMfmaF32
    for M, N, K in _shapes(t)[1:6]:
        a, b = orc.fill_random(M * K, 21 + K), orc.fill_random(K * N, 22 + N)
        bias = orc.fill_random(N, 23 + M)
        da, pa = _up(gpu, a, 1)
        db, pb = _up(gpu, b, 2)
        dbias, pbias = _up(gpu, bias, 0)
        c, y, fused = _Out(gpu, M * N, 0), _Out(gpu, M * N, 0), _Out(gpu, M * N, 3)
        tile = _tile(gpu, t)
        for st in (gpu.launch_gemm_f32(pa, pb, c.ptr, M, N, K, 0.75, 0.0, V, tile),
                   gpu.launch_bias_act_f32(c.ptr, pbias, y.ptr, M, N, act, 1),
                   gpu.launch_gemm_bias_act_f32(pa, pb, pbias, fused.ptr, M, N, K, 0.75, act,
                                                tile)):
            assert st.ok(), str(st)
        gpu.device_synchronize()
        assert np.array_equal(fused.get().view(np.uint32), y.get().view(np.uint32)), \
            f"{M}x{N}x{K} tile={t}"
        del da, db, dbias


@pytest.mark.parametrize("t,shape", [(t, (t + 1, t + 5, 45)) for t in TILES] +
                         [(64, (1000, 1023, 45)), (32, (500, 515, 77))],
                         ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else str(v))
def test_gemm_remainder_keeps_special_values_apart(gpu, orc, t, shape):
    """K % 32 != 0 pads both operands with zeros: infinities and NaN in the last columns of
    A, the last rows of B, and past the operands' ends reach their own outputs only.  (At t +
    1 x t + 5 the 64 x 64 launch runs 32 x 64 tiles and the 32 x 32 one the few-tiles kernel;
    the last two shapes run the tile's own EDGE kernel.)"""
    M, N, K = shape
    a = orc.fill_random(M * K, 31).reshape(M, K)
    b = orc.fill_random(K * N, 32).reshape(K, N)
    a[M - 1, 3], a[0, K - 1] = np.nan, np.inf
    b[K - 1, N - 1] = -np.inf
    want = np.einsum("mk,kn->mn", a.astype(np.float64), b.astype(np.float64))
    da, pa = _up(gpu, a, 0)
    db, pb = _up(gpu, b, 0)
    out = _Out(gpu, M * N, 0)
    st = gpu.launch_gemm_f32(pa, pb, out.ptr, M, N, K, 1.0, 0.0, gpu.GemmVariant.kMfmaF32,
                             _tile(gpu, t))
    assert st.ok(), str(st)
    gpu.device_synchronize()
    got = out.get().reshape(M, N)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    assert np.array_equal(got[np.isinf(want)], want[np.isinf(want)])
    fin = np.isfinite(want)
    assert orc.compare(got[fin], want[fin], orc.tol_gemm(K), orc.abs_tol_gemm(K)).ok


# (M, N, K) around the few-tiles kernel's tiles (16 x 16 while 256 of them hold the product,
# then 16 x 32 from K = 320 on, 32 x 32 from K = 1024 on, 16 x 64 up to 16 rows), K chunks
# (32, dealt to 8 waves) and limits (15 columns, more than 256 tiles: the tile kernels).
ROWS_SHAPES = [(1, 16, 1), (16, 17, 31), (17, 31, 32), (31, 33, 33), (32, 100, 255), (33, 64, 1024),
               (48, 77, 1031), (64, 259, 1056), (15, 4095, 257), (16, 4096, 256), (5, 4097, 1024),
               (16, 4128, 1027), (32, 8192, 1025), (3, 8193, 1055), (16, 16383, 1024),
               (65, 40, 300), (7, 15, 90), (255, 255, 70), (300, 217, 321), (193, 771, 1056),
               (512, 512, 1055), (2000, 33, 333), (257, 256, 64)]


@pytest.mark.parametrize("shape", ROWS_SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_few_rows(gpu, orc, shape):
    M, N, K = shape
    V = gpu.GemmVariant.kMfmaF32
    tile = _tile(gpu, 32)
    a = orc.fill_random(M * K, 41 + K).reshape(M, K)
    b = orc.fill_random(K * N, 42 + N).reshape(K, N)
    c = orc.fill_random(M * N, 43 + M).reshape(M, N)
    bias = orc.fill_random(N, 44)
    prod = a.astype(np.float64) @ b.astype(np.float64)
    rel, floor = orc.tol_gemm(K), orc.abs_tol_gemm(K) + 4e-7
    for sa, sb, sc, beta in ((0, 0, 0, 0.0), (1, 3, 2, 1.5)):
        da, pa = _up(gpu, a, sa)
        db, pb = _up(gpu, b, sb)
        out = _Out(gpu, M * N, sc)
        full = out.buf.download()
        full[out.at:out.at + M * N] = np.nan if beta == 0.0 else c.ravel()
        out.buf.upload(full)
        st = gpu.launch_gemm_f32(pa, pb, out.ptr, M, N, K, 0.75, beta, V, tile)
        assert st.ok(), str(st)
        gpu.device_synchronize()
        got = out.get()
        r = orc.compare(got, (0.75 * prod + beta * c).ravel(), rel, floor)
        assert r.ok, f"shifts={sa},{sb},{sc}: {r}"
        if beta == 0.0:
            # The fused launch has the bits of the pair.
            dbias, pbias = _up(gpu, bias, 0)
            y, fused = _Out(gpu, M * N, 0), _Out(gpu, M * N, 1)
            for st in (gpu.launch_bias_act_f32(out.ptr, pbias, y.ptr, M, N, 3, 1),
                       gpu.launch_gemm_bias_act_f32(pa, pb, pbias, fused.ptr, M, N, K, 0.75, 3,
                                                    tile)):
                assert st.ok(), str(st)
            gpu.device_synchronize()
            assert np.array_equal(fused.get().view(np.uint32), y.get().view(np.uint32))
        del da, db


def test_few_rows_repeat_their_bits(gpu, orc):
    """The same bits on every run (no state between launches)."""
    M, N, K = 16, 1000, 1003
    a, b = orc.fill_random(M * K, 51), orc.fill_random(K * N, 52)
    da, db = gpu.DeviceBuffer.from_array(a), gpu.DeviceBuffer.from_array(b)
    seen = []
    for _ in range(3):
        out = _Out(gpu, M * N, 0)
        st = gpu.launch_gemm_f32(da, db, out.ptr, M, N, K, 1.0, 0.0, gpu.GemmVariant.kMfmaF32,
                                 _tile(gpu, 32))
        assert st.ok(), str(st)
        gpu.device_synchronize()
        seen.append(out.get().view(np.uint32).copy())
    assert np.array_equal(seen[0], seen[1]) and np.array_equal(seen[0], seen[2])
