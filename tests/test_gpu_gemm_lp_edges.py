"""GPU parity of the 16-bit GEMM at shapes that are not whole tiles: the EDGE form of the
direct-to-LDS kernel, the WHOLE form of the register-staged one and the split-K kernel,
around their tiles, K steps and limits, with operands and C at every element offset, C
between guard values that must keep their bits.

Bars: quarter-multiple inputs make every sum exact in fp32, so the result is the oracle's
bit for bit; infinities and NaN reach their own outputs only.
"""
from __future__ import annotations

import numpy as np
import pytest

from tests.test_gpu_gemm_lp import BF16, DT_ID, DTS, F16, F32, _quarters

pytestmark = pytest.mark.gpu

GUARD = 16

# EDGE at 128 x 128 takes even N >= 128 and K >= 64 from 208 tiles on (from 80 on where K is
# at least 256, 100 with a 16-bit C; else the first five run split K), at 256 x 256 from 192
# tiles on; K % 64 is its first pair of steps (0, 2, 30, 32, 62 left over).
EDGE_128 = [(1279, 1024, 64), (1151, 1150, 66), (1025, 1154, 94), (10200, 130, 160),
            (129, 10112, 126), (1663, 2048, 64), (1919, 1790, 66), (1665, 2050, 94),
            (10200, 330, 160), (129, 13440, 126), (1151, 1150, 290)]
EDGE_256 = [(3073, 4000, 66), (3100, 4098, 128)]
# Whole 128 x 128 tiles, 80 of them or more, with K % 64 == 32: the direct-to-LDS 32x32x16
# kernel, 1, 3, 5 and 7 K steps of 32 (its 4-stage ring's prologue and tail).
DMA_32 = [(1280, 1024, 32), (1280, 1024, 96), (1152, 1280, 160), (1024, 1280, 224)]
# The register-staged kernel's WHOLE form: odd N or K, from 208 tiles of 128 or 192 of 256
# on; K % 64 of 0, 1, 32, 63 as the first stage, one and two stages, last tile columns of 1
# and 127 columns of their own.
WHOLE_128 = [(1921, 1665, 64), (1793, 1919, 65), (1665, 2049, 191), (13300, 129, 96),
             (129, 13311, 127), (1409, 2563, 321)]
WHOLE_256 = [(3073, 3841, 66), (3100, 4095, 127)]
# Split K: 16 and 32 rows (8 waves), 32 x 64 and 64 x 64 tiles (past 1024 of 32 x 64), odd
# widths, K around its 32-deep chunks dealt to 4 and 8 waves, none and several to a wave; the
# remainder with wave 0 or another, below 8, a multiple of 8 or not; N below 32:
# register-staged.
SPLIT = [(1, 32, 1), (16, 33, 31), (15, 8191, 33), (17, 100, 257), (32, 63, 256), (33, 63, 96),
         (33, 64, 32), (65, 131, 65), (200, 136, 264), (127, 1001, 127), (257, 9001, 63),
         (5, 8193, 70), (3001, 1501, 35), (40, 31, 64), (7, 5, 3), (33, 100, 7), (1, 64, 8),
         (65, 131, 41), (16, 4096, 1031), (32, 515, 2049), (17, 8191, 545), (100, 63, 1100),
         (70, 200, 1183), (2049, 2051, 271)]


# Past 1024 tiles of 32 x 64, K below 64 where rows are 16-byte aligned and below 8 elsewhere:
# the register-staged kernel, at 128 x 128 for the last two (441 and 476 tiles), else 64 x 64.
SHORT_K = [(2081, 1032, 8), (2460, 1608, 56), (2293, 1737, 7), (4097, 513, 1), (2166, 3544, 40),
           (2688, 2688, 56)]


def _check(m, orc, dt, out, M, N, K, tile, shifts, alpha, beta):
    rng = np.random.default_rng(M * 7 + N * 3 + K)
    a16 = orc.to_16(_quarters(rng, (M, K)), dt)
    b16 = orc.to_16(_quarters(rng, (K, N)), dt)
    cf = _quarters(rng, (M, N))
    cd = F32 if out == "f32" else dt
    ct = np.float32 if cd == F32 else np.uint16
    c = cf.ravel() if cd == F32 else orc.to_16(cf, dt).ravel()
    # The oracle's value in float64 (exact: quarter multiples), rounded as C is.
    want = alpha * (orc.from_16(a16, dt).reshape(M, K).astype(np.float64) @
                    orc.from_16(b16, dt).reshape(K, N).astype(np.float64)) + beta * cf
    want = want.astype(np.float32).ravel()
    want = want if cd == F32 else orc.to_16(want, dt).ravel()
    nan16 = 0x7FC0 if dt == BF16 else 0x7E00
    bufs = []

    def up(arr, shift):
        pad = np.full(GUARD, nan16, np.uint16)
        buf = m.DeviceBuffer.from_array(np.concatenate([pad, pad[:shift], arr.ravel(), pad]))
        bufs.append(buf)
        return buf.ptr + 2 * (GUARD + shift)

    pa, pb = up(a16, shifts[0]), up(b16, shifts[1])
    at = GUARD + shifts[2]
    mark = np.full(at + M * N + GUARD, 77, ct)
    mark[at:at + M * N] = c if beta != 0.0 else (np.nan if cd == F32 else nan16)
    dc = m.DeviceBuffer.from_array(mark)
    st = m.launch_gemm_lp(pa, pb, dc.ptr + at * mark.itemsize, dt, cd, M, N, K, alpha, beta, tile)
    assert st.ok(), str(st)
    m.device_synchronize()
    full = dc.download(mark.size, ct)
    where = f"{M}x{N}x{K} {DT_ID[dt]}->{out} {tile} shifts={shifts} beta={beta}"
    assert (full[:at] == 77).all() and (full[at + M * N:] == 77).all(), "wrote outside C: " + where
    got = full[at:at + M * N]
    bits = np.uint32 if cd == F32 else np.uint16
    bad = np.nonzero(got.view(bits) != want.view(bits))[0]
    assert bad.size == 0, f"{where}: {bad.size} wrong, first at {divmod(int(bad[0]), N)}"


@pytest.mark.parametrize("dt", DTS, ids=DT_ID.get)
@pytest.mark.parametrize("out", ["f32", "same"])
@pytest.mark.parametrize("shape", EDGE_128 + EDGE_256, ids=lambda s: "x".join(map(str, s)))
def test_edge_tiles(gpu, orc, dt, out, shape):
    tile = gpu.LP_TILES[0] if shape in EDGE_256 else gpu.LP_TILES[1]
    _check(gpu, orc, dt, out, *shape, tile, (0, 0, 0), 1.0, 0.0)
    _check(gpu, orc, dt, out, *shape, tile, (2, 4, 2), 0.5, 2.0)


@pytest.mark.parametrize("dt", DTS, ids=DT_ID.get)
@pytest.mark.parametrize("out", ["f32", "same"])
@pytest.mark.parametrize("shape", DMA_32, ids=lambda s: "x".join(map(str, s)))
def test_whole_tiles_of_32_deep_stages(gpu, orc, dt, out, shape):
    _check(gpu, orc, dt, out, *shape, gpu.LP_TILES[1], (0, 0, 0), 1.0, 0.0)
    _check(gpu, orc, dt, out, *shape, gpu.LP_TILES[1], (0, 0, 0), 0.5, 2.0)


@pytest.mark.parametrize("dt", DTS, ids=DT_ID.get)
@pytest.mark.parametrize("out", ["f32", "same"])
@pytest.mark.parametrize("shape", WHOLE_128 + WHOLE_256, ids=lambda s: "x".join(map(str, s)))
def test_whole_form_of_the_staged_kernel(gpu, orc, dt, out, shape):
    tile = gpu.LP_TILES[0] if shape in WHOLE_256 else gpu.LP_TILES[1]
    _check(gpu, orc, dt, out, *shape, tile, (0, 0, 0), 1.0, 0.0)
    _check(gpu, orc, dt, out, *shape, tile, (1, 3, 1), 0.5, 2.0)


@pytest.mark.parametrize("dt", DTS, ids=DT_ID.get)
@pytest.mark.parametrize("out", ["f32", "same"])
@pytest.mark.parametrize("shape", SPLIT, ids=lambda s: "x".join(map(str, s)))
def test_split_k(gpu, orc, dt, out, shape):
    _check(gpu, orc, dt, out, *shape, gpu.LP_TILES[2], (0, 0, 0), 1.0, 0.0)
    _check(gpu, orc, dt, out, *shape, gpu.LP_TILES[2], (1, 3, 1), 0.5, 2.0)


@pytest.mark.parametrize("dt", DTS, ids=DT_ID.get)
@pytest.mark.parametrize("out", ["f32", "same"])
@pytest.mark.parametrize("shape", SHORT_K, ids=lambda s: "x".join(map(str, s)))
def test_short_k(gpu, orc, dt, out, shape):
    tile = gpu.gemm_lp_default_tile(*shape)
    _check(gpu, orc, dt, out, *shape, tile, (0, 0, 0), 1.0, 0.0)
    _check(gpu, orc, dt, out, *shape, tile, (1, 3, 1), 0.5, 2.0)


@pytest.mark.parametrize("dt", DTS, ids=DT_ID.get)
@pytest.mark.parametrize("out", ["f32", "same"])
@pytest.mark.parametrize("shape", [(300, 24, 72), (70, 8, 128), (513, 16, 8)],
                         ids=lambda s: "x".join(map(str, s)))
def test_narrow_products_on_every_tile(gpu, orc, dt, out, shape):
    """Below 32 columns: the register-staged kernel at the requested tile, 16 bytes a load
    and element by element."""
    for tile in gpu.LP_TILES:
        _check(gpu, orc, dt, out, *shape, tile, (0, 0, 0), 1.0, 0.0)
        _check(gpu, orc, dt, out, *shape, tile, (1, 3, 1), 0.5, 2.0)


def test_remainders_keep_special_values_apart(gpu, orc):
    """The K remainder pads both operands with zeros: infinities and NaN in the last columns
    of A and the last rows of B reach their own outputs only."""
    for M, N, K, tile in ((1663, 2050, 70, gpu.LP_TILES[1]), (1279, 1026, 70, gpu.LP_TILES[1]),
                          (1921, 1665, 131, gpu.LP_TILES[1]), (37, 131, 45, gpu.LP_TILES[2])):
        rng = np.random.default_rng(K)
        a, b = _quarters(rng, (M, K)), _quarters(rng, (K, N))
        a[M - 1, 3], a[0, K - 1] = np.nan, np.inf
        b[K - 1, N - 1] = -np.inf
        b[K - 1, 0] = 0.25
        a16, b16 = orc.to_16(a, F16), orc.to_16(b, F16)
        with np.errstate(invalid="ignore"):
            want = (np.einsum("mk,kn->mn", a.astype(np.float64), b.astype(np.float64))
                    .astype(np.float32))
        da, db = gpu.DeviceBuffer.from_array(a16), gpu.DeviceBuffer.from_array(b16)
        dc = gpu.DeviceBuffer(M * N * 4)
        st = gpu.launch_gemm_lp(da, db, dc, F16, F32, M, N, K, 1.0, 0.0, tile)
        assert st.ok(), str(st)
        gpu.device_synchronize()
        got = dc.download(M * N).reshape(M, N)
        assert np.array_equal(np.isnan(got), np.isnan(want))
        ok = ~np.isnan(want)
        assert np.array_equal(got[ok], want[ok])


@pytest.mark.parametrize("along", ["rows", "columns"])
def test_extents_up_to_int32_max(gpu, orc, along):
    """INT32_MAX rows or columns are accepted (extent + tile - 1 is past an int there): an
    outer product with one column or row, whose every value is half the long operand's."""
    n, period = 2**31 - 1, 1000003
    M, N = (n, 1) if along == "rows" else (1, n)
    tile = gpu.gemm_lp_default_tile(M, N, 1)
    pattern = orc.to_16(((np.arange(period) * 7) % 1021 / 4.0).astype(np.float32), F16)
    want = orc.to_16(orc.from_16(pattern, F16) * np.float32(0.5), F16)
    copy = gpu.lib().mcke_rt_memcpy_async
    x, y = gpu.DeviceBuffer(2 * n), gpu.DeviceBuffer(2 * (n + GUARD))
    half = gpu.DeviceBuffer.from_array(orc.to_16(np.full(1, 0.5, np.float32), F16))
    head = gpu.DeviceBuffer.from_array(pattern)
    assert copy(x.ptr, head.ptr, 2 * period, 2, None) == 0
    done = 2 * period
    while done < 2 * n:                     # the part that is there, again behind itself
        take = min(done, 2 * n - done)
        assert copy(x.ptr + done, x.ptr, take, 2, None) == 0
        done += take
    mark = gpu.DeviceBuffer.from_array(np.full(GUARD, 77, np.uint16))
    assert copy(y.ptr + 2 * n, mark.ptr, 2 * GUARD, 2, None) == 0
    a, b = (x, half) if along == "rows" else (half, x)
    st = gpu.launch_gemm_lp(a, b, y, F16, F16, M, N, 1, 1.0, 0.0, tile)
    assert st.ok(), str(st)
    gpu.device_synchronize()
    chunk = np.empty(32 * period, np.uint16)
    tiled = np.tile(want, 32)
    for at in range(0, n, chunk.size):
        part = chunk[:min(chunk.size, n - at)]
        assert copy(part.ctypes.data, y.ptr + 2 * at, part.nbytes, 1, None) == 0
        gpu.device_synchronize()
        assert np.array_equal(part, tiled[:part.size]), f"in [{at}, {at + part.size})"
    tail = np.empty(GUARD, np.uint16)
    assert copy(tail.ctypes.data, y.ptr + 2 * n, tail.nbytes, 1, None) == 0
    gpu.device_synchronize()
    assert (tail == 77).all()
