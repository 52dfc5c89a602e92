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
