"""GPU parity of the row kernels where their split of a row can go wrong: widths at the
edges of each lane layout, rows and base addresses at every offset from a 16-byte
boundary (x and y apart), fewer rows than a workgroup owns, against the CPU oracle.
Every output buffer has guard floats around it that must keep their bits.

Bars: softmax rel 1e-5 + abs 1e-6 (the fixed-shape tests' bar); max exact; sums in
float64 within 2^-24 times the longest chain of adds a lane and its combine can make
(cols / 32 + 16 at most for these layouts), relative to the row's sum of magnitudes;
bias + activation bit-equal to the capped launch, which walks rows in chunks, and past 4096
workgroups with the row kernel; there also against the oracle at abs 1e-6 + rel 1e-6.
"""
from __future__ import annotations

import numpy as np
import pytest

from tests.gpu_util import f32

pytestmark = pytest.mark.gpu

GUARD = 8
MARK = np.float32(-77.25)


class _Out:
    """`n` floats at `shift` floats past a 16-byte boundary, between guard floats."""

    def __init__(self, m, n, shift):
        self.n, self.at = n, GUARD + shift
        self.buf = m.DeviceBuffer.from_array(np.full(n + 2 * GUARD + 4, MARK, np.float32))
        self.ptr = self.buf.ptr + 4 * self.at

    def get(self):
        full = self.buf.download()
        assert (full[:self.at] == MARK).all() and (full[self.at + self.n:] == MARK).all(), \
            "wrote outside the output"
        return full[self.at:self.at + self.n]


def _up(m, x, shift):
    # The floats around x are NaN: a read past either end that reached a result shows.
    pad = np.full(GUARD + 4, np.nan, np.float32)
    buf = m.DeviceBuffer.from_array(np.concatenate([pad[:GUARD + shift], f32(x), pad]))
    return buf, buf.ptr + 4 * (GUARD + shift)


# (x, y) offsets in floats; GUARD is a multiple of 4, so (0, 0) is the aligned one.
SHIFTS = [(0, 0), (1, 1), (3, 2), (0, 3)]
SOFTMAX_COLS = [1, 2, 3, 5, 35, 36, 39, 67, 68, 71, 131, 259, 260, 263, 515, 519, 1027, 1031,
                2055, 4103, 8195, 8200, 16387, 16391, 32768, 32771,
                32776, 65536, 65539, 65540, 65543]


@pytest.mark.parametrize("cols", SOFTMAX_COLS)
def test_softmax_width_edges(gpu, orc, cols):
    rows = 37 if cols < 4096 else 3
    x = orc.fill_normal(rows * cols, 0x50F7 + cols, 0.0, 2.0)
    x[cols - 1] += 30.0
    want = orc.row_softmax(x, rows, cols)
    for sx, sy in SHIFTS:
        buf, px = _up(gpu, x, sx)
        out = _Out(gpu, rows * cols, sy)
        st = gpu.launch_row_softmax_f32(px, out.ptr, rows, cols, gpu.SoftmaxVariant.kOnlineOnePass)
        assert st.ok(), str(st)
        gpu.device_synchronize()
        r = orc.compare(out.get(), want, 1e-5, 1e-6)
        assert r.ok, f"cols={cols} shift={sx},{sy}: {r}"
        del buf


REDUCE_COLS = [1, 2, 5, 7, 31, 128, 131, 132, 133, 256, 259, 260, 263, 515, 516, 519, 1027, 1028,
               1031, 2048, 2051, 2052, 2055, 4095, 4099]


@pytest.mark.parametrize("cols", REDUCE_COLS)
@pytest.mark.parametrize("kind", [0, 1, 2])
def test_row_reduce_width_edges(gpu, orc, cols, kind):
    rows = 77
    x = orc.fill_normal(rows * cols, 0x2ED0 + cols, 0.0, 1.0).reshape(rows, cols)
    if kind == 1:
        x[3] = -np.inf
        x[4, cols // 2] = np.nan if cols > 1 else x[4, 0]
    x64 = x.astype(np.float64)
    if kind == 1:
        want = np.fmax.reduce(x64, axis=1)
        bar = np.zeros(rows)
    else:
        want = x64.sum(axis=1)
        bar = (cols / 32 + 16) * 2.0 ** -24 * np.abs(x64).sum(axis=1)
        if kind == 2:
            want, bar = want / cols, bar / cols + 2.0 ** -24 * np.abs(want / cols)
    V = gpu.ReduceVariant
    for sx, _ in SHIFTS[:3]:
        buf, px = _up(gpu, x, sx)
        for variant in (V.kWarpShuffle, V.kTwoPass):
            out = _Out(gpu, rows, 1)
            if variant == V.kTwoPass:
                nbytes = gpu.row_reduce_workspace_bytes(rows, cols, variant)
                ws = gpu.DeviceBuffer(max(4, nbytes))
                st = gpu.launch_row_reduce_f32(px, out.ptr, rows, cols, kind, variant, ws, nbytes,
                                               None)
            else:
                st = gpu.launch_row_reduce_f32(px, out.ptr, rows, cols, kind, variant)
            assert st.ok(), str(st)
            gpu.device_synchronize()
            got = out.get().astype(np.float64)
            same = got == want
            with np.errstate(invalid="ignore"):
                assert (same | (np.abs(got - want) <= bar)).all(), \
                    f"cols={cols} kind={kind} {variant!r} shift={sx}"
        del buf


@pytest.mark.parametrize("cols", [100003, 65537])
def test_split_sum_at_any_alignment(gpu, orc, cols):
    """The split form's chunks start where the row does, plus a multiple of 4 floats."""
    rows, V = 3, gpu.ReduceVariant.kTwoPass
    x = orc.fill_random(rows * cols, 0x5B11 + cols, 0.0, 1.0).reshape(rows, cols)
    want = x.astype(np.float64).sum(axis=1)
    nbytes = gpu.row_reduce_workspace_bytes(rows, cols, V)
    ws = gpu.DeviceBuffer(nbytes)
    for sx in range(4):
        buf, px = _up(gpu, x, sx)
        out = _Out(gpu, rows, 0)
        st = gpu.launch_row_reduce_f32(px, out.ptr, rows, cols, 0, V, ws, nbytes, None)
        assert st.ok(), str(st)
        gpu.device_synchronize()
        assert np.allclose(out.get(), want, rtol=1e-6, atol=0.0), f"shift={sx}"
        del buf


@pytest.mark.parametrize("act", [0, 1, 2, 3])
@pytest.mark.parametrize("cols", [1, 2, 3, 5, 63, 100, 129, 252, 255, 257, 260, 1000, 4095])
def test_bias_act_any_width_matches_the_row_kernel(gpu, orc, cols, act):
    rows = 301 if cols < 64 else 37
    x = orc.fill_normal(rows * cols, 0xB1A5 + cols, 0.0, 2.0)
    x[0], x[-1] = np.inf, -np.inf
    bias = orc.fill_random(cols, 0xB1A6 + cols, -0.5, 0.5)
    db, pb = _up(gpu, bias, 0)
    dx, px = _up(gpu, x, 0)
    widest = min(gpu.max_vector_width_f32(p, cols) for p in (px, pb))
    ref = _Out(gpu, rows * cols, 0)
    st = gpu.launch_bias_act_f32(px, pb, ref.ptr, rows, cols, act, 1, None, rows)
    assert st.ok(), str(st)
    gpu.device_synchronize()
    want = ref.get().view(np.uint32)
    for vw in (w for w in (1, 2, 4) if w <= widest):
        out = _Out(gpu, rows * cols, 0)
        st = gpu.launch_bias_act_f32(px, pb, out.ptr, rows, cols, act, vw)
        assert st.ok(), str(st)
        gpu.device_synchronize()
        assert np.array_equal(out.get().view(np.uint32), want), f"vw={vw}"
    for sx, sy, sb in ((1, 2, 3), (3, 0, 1)):
        d2, p2 = _up(gpu, x, sx)
        b2, q2 = _up(gpu, bias, sb)
        out = _Out(gpu, rows * cols, sy)
        st = gpu.launch_bias_act_f32(p2, q2, out.ptr, rows, cols, act, 1)
        assert st.ok(), str(st)
        gpu.device_synchronize()
        assert np.array_equal(out.get().view(np.uint32), want), f"shift={sx},{sy},{sb}"
    del db, dx


@pytest.mark.parametrize("act", [0, 1, 2, 3])
@pytest.mark.parametrize("cols", [100, 256])
def test_bias_act_kernels_of_many_rows_agree(gpu, orc, cols, act):
    """4101 rows: capped launches walk them with the row kernel (7 workgroup rows, and one
    per row), the others run as one flat array or, at vw = 4 and 256 columns, as whole 1 KiB
    strips."""
    rows = 4101
    x = orc.fill_normal(rows * cols, 0xB1A7 + cols, 0.0, 2.0)
    bias = orc.fill_random(cols, 0xB1A8 + cols, -0.5, 0.5)
    want = orc.bias_act(x, bias, rows, cols, act)
    dx, px = _up(gpu, x, 0)
    db, pb = _up(gpu, bias, 0)
    seen = None
    for vw in (1, 2, 4):
        for cap in (7, rows, 0):
            out = _Out(gpu, rows * cols, 0)
            st = gpu.launch_bias_act_f32(px, pb, out.ptr, rows, cols, act, vw, None, cap)
            assert st.ok(), str(st)
            gpu.device_synchronize()
            got = out.get()
            if seen is None:
                seen = got.view(np.uint32).copy()
                r = orc.compare(got, want, 1e-6, 1e-6)
                assert r.ok, str(r)
            assert np.array_equal(got.view(np.uint32), seen), f"vw={vw} cap={cap}"
    del dx, db
