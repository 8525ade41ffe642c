"""GPU parity of the row kernels where their split of a row can go wrong: widths at the
edges of each lane layout, rows and base addresses at every offset from a 16-byte
boundary (x and y apart), fewer rows than a workgroup owns, against the CPU oracle.
Every output buffer has guard floats around it that must keep their bits.

Bars: softmax rel 1e-5 + abs 1e-6 (the fixed-shape tests' bar); max exact; sums in
float64 within 2^-24 times the longest chain of adds a lane and its combine can make
(cols / 32 + 16 at most for these layouts), relative to the row's sum of magnitudes;
bias + activation bit-equal to the capped launch, which walks rows with the row kernel.
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
                2055, 4103, 8195, 8200, 16387, 16391, 32771, 32776, 65536, 65539, 65540, 65543]


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
