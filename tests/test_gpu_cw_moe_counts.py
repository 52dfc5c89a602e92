"""Grouped experts with uneven counts: every form of the launch (4, 8, 16 columns,
and a second pass beyond 16 pairs) at its edges in one call, bitwise against the
oracle; and the several-column lane kernel that the matrix-core one replaces on
most shapes."""
import numpy as np
import pytest

from oracle import Q8_0, Q5_0, Q4_K, Q6_K, IQ2_XXS, IQ3_XXS, col_stride_floats, row_bytes
from util import activations, sane_rows, tuned
from test_gpu_parity import bits, dev_cols, say
from test_gpu_cw_iq import check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fmt", [Q8_0, Q5_0, Q4_K, Q6_K, IQ2_XXS, IQ3_XXS])
@pytest.mark.parametrize("rows,cols", [(50, 1280), (700, 2048)])
def test_uneven_experts(flh, orc, gpu, fmt, rows, cols):
    say("uneven experts", fmt, rows, cols)
    counts = [1, 4, 5, 8, 9, 16, 17, 0, 33, 2]
    rng = np.random.default_rng(fmt + rows)
    ids = rng.permutation(np.repeat(np.arange(len(counts)), counts)).astype(np.uint32)
    n, eb = len(ids), rows * row_bytes(fmt, cols)
    w = sane_rows(fmt, len(counts) * rows, cols, rng)
    xs = activations(n, cols, rng, outliers=True)
    st = (col_stride_floats(cols) + 3) & ~3
    y0 = rng.standard_normal(n * rows).astype(np.float32)
    dx, _ = dev_cols(flh, gpu, xs, st)
    flh.act_q8(dx, cols, gpu, nx=n, xstride=st)
    dw, dy = flh.DeviceBuffer.from_array(w, gpu), flh.DeviceBuffer.from_array(y0, gpu)
    flh.moe_dot(fmt, dw, eb, rows, cols, flh.DeviceBuffer.from_array(ids, gpu), n, 1, len(counts), dx, st, False, dy, rows,
                gpu)
    got = dy.download(np.float32, y0.size, gpu)
    xq, want = orc.act_q8_cols(xs, st), y0.copy()
    for i, e in enumerate(ids):
        orc.stream_dot(fmt, w[e * eb:(e + 1) * eb], rows, cols, xq[i * st:], want[i * rows:(i + 1) * rows], xstride=st,
                       ystride=rows, i8_mask=0x7F)
    assert np.array_equal(bits(got), bits(want))


@pytest.mark.parametrize("rows,cols,nx", [(100, 2048, 2), (257, 4096, 5), (65, 6144, 8), (40, 8192, 16)])
@pytest.mark.parametrize("fmt", [Q8_0, Q5_0, IQ2_XXS, IQ3_XXS])
def test_lane_kernel(flh, orc, gpu, fmt, rows, cols, nx):
    say("lane kernel", fmt, rows, cols, nx)
    with tuned(flh, FLH_CW="0"):
        check(flh, orc, gpu, fmt, rows, cols, nx, pad=1)
