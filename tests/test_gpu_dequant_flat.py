"""flh_dequant on flat units of 256 outputs, bitwise against the oracle: partial
last units (32-weight blocks), a workgroup's last units, odd addresses."""
import numpy as np
import pytest

from oracle import Q8_0, Q5_0, Q4_K, Q6_K, IQ2_XXS, IQ3_XXS
from util import sane_rows
from test_gpu_parity import bits, say

pytestmark = pytest.mark.gpu

K = [(1, 256), (3, 768), (17, 1024), (70, 4096)]
B32 = [(1, 32), (3, 96), (5, 224), (7, 288), (33, 2080)] + K


@pytest.mark.parametrize("shift", [0, 1, 2])
@pytest.mark.parametrize("fmt,rows,cols", [(f, r, c) for f in (Q8_0, Q5_0) for r, c in B32] +
                         [(f, r, c) for f in (Q4_K, Q6_K, IQ2_XXS, IQ3_XXS) for r, c in K])
def test_dequant_bitwise(flh, orc, gpu, fmt, rows, cols, shift):
    say("dequant", fmt, rows, cols, shift)
    w = sane_rows(fmt, rows, cols, np.random.default_rng(fmt * 100 + rows))
    dw = flh.DeviceBuffer.from_array(np.concatenate([np.zeros(shift, np.uint8), w]), gpu)
    guard = np.full(rows * cols + 64, 7.0, np.float32)
    out = flh.DeviceBuffer.from_array(guard, gpu)
    flh.dequant(fmt, dw.ptr + shift, rows, cols, out, gpu)
    got = out.download(np.float32, guard.size, gpu)
    assert np.array_equal(bits(got[:rows * cols]), bits(orc.dequant(fmt, w, rows, cols).ravel()))
    assert np.all(got[rows * cols:] == 7.0)


@pytest.mark.parametrize("fmt,rows", [(IQ2_XXS, (1 << 20) + 3), (Q8_0, (1 << 20) - 1)])
def test_dequant_past_one_launch(flh, orc, gpu, fmt, rows):
    """2^35 outputs: more than one launch's 2^24 - 1 workgroups of 2048 outputs, and one
    row fewer than that.  The matrix repeats 5 rows, and so do its outputs."""
    cols, rep = 32768, 5
    say("dequant", fmt, rows)
    w = sane_rows(fmt, rep, cols, np.random.default_rng(fmt))
    rb = w.size // rep
    want = orc.dequant(fmt, w, rep, cols)
    dw, out = flh.DeviceBuffer(rows * rb), flh.DeviceBuffer(rows * cols * 4)
    dw.upload(w, gpu)
    have = rep
    while have < rows:                                            # doubled
        n = min(have, rows - have)
        flh.copy(dw.ptr + have * rb, dw, n * rb, gpu)
        have += n
    n = 2 * rep
    flh.check(flh.lib().flh_zero(out.ptr + (rows - n) * cols * 4, n * cols * 4, gpu.handle))
    flh.dequant(fmt, dw, rows, cols, out, gpu)
    edge = ((1 << 24) - 1) * 2048 // cols                         # the row that a second launch begins in
    for r0 in (0, rows // 2, min(edge, rows) - rep, rows - n):
        part = flh.DeviceBuffer(n * cols * 4)
        m = min(n, rows - r0)
        flh.copy(part, out.ptr + r0 * cols * 4, m * cols * 4, gpu)
        got = part.download(np.float32, m * cols, gpu).reshape(m, cols)
        assert np.array_equal(bits(got), bits(want[(np.arange(m) + r0) % rep])), r0
    dw.close()
    out.close()
