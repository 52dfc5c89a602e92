"""F32 rows on a workgroup per row (k_dot_f32small), bitwise against the
oracle's fast fp32 order at the edges of its tiles (4096 columns), column
groups (4) and routing lines."""
import numpy as np
import pytest

from oracle import F32, col_stride_floats
from util import activations, normal_weights
from test_gpu_parity import bits, dev_cols, say

pytestmark = pytest.mark.gpu

CASES = [(1, 16, 1), (3, 15, 2), (5, 64, 4), (7, 4095, 1), (2, 4096, 5), (9, 4097, 3), (4, 4112, 16), (3, 8192, 4),
         (2, 12289, 2), (64, 2048, 8), (512, 272, 16), (513, 272, 16), (2048, 48, 3), (2049, 48, 3), (5000, 512, 1),
         # either side of the routing lines: rows and lengths of one column, narrow rows of several
         (2048, 100, 1), (2049, 100, 1), (4096, 768, 1), (4096, 1024, 1), (1536, 512, 3), (1537, 1276, 3), (2048, 1280, 3), (16384, 1024, 1), (16385, 1024, 1),
         (20000, 2047, 1), (20000, 2048, 1), (1280, 500, 4), (1281, 500, 3), (1281, 512, 4), (2048, 512, 3)]


@pytest.mark.parametrize("rows,cols,nx", CASES)
def test_f32_small_bitwise(flh, orc, gpu, rows, cols, nx):
    say("f32 small", rows, cols, nx)
    rng = np.random.default_rng(rows * 31 + cols + nx)
    w = normal_weights(rows, cols, rng, std=0.5).view(np.uint8).reshape(-1)
    y0 = rng.standard_normal(nx * rows).astype(np.float32)
    xs = activations(nx, cols, rng, outliers=True)
    st = col_stride_floats(cols)
    dx, hx = dev_cols(flh, gpu, xs, st)
    dy = flh.DeviceBuffer.from_array(y0, gpu)
    dw = flh.DeviceBuffer.from_array(w, gpu)
    flh.stream_dot(F32, dw, rows, cols, dx, dy, gpu, nx=nx, xstride=st, ystride=rows)
    want = y0.copy()
    orc.stream_dot(F32, w, rows, cols, hx, want, nx=nx, xstride=st, ystride=rows, fast=True, threads=8)
    assert np.array_equal(bits(dy.download(np.float32, y0.size, gpu)), bits(want))


@pytest.mark.parametrize("rows", [(1 << 24) - 1, 1 << 24, (1 << 24) + 37])
def test_f32_rows_past_one_launch(flh, orc, gpu, rows):
    """2^24 rows of one column: a workgroup of 256 threads per row is more than a
    launch holds.  The matrix repeats 4099 rows, and so do its outputs."""
    say("f32 rows", rows)
    cols, rep = 16, 4099
    rng = np.random.default_rng(rows)
    w = normal_weights(rep, cols, rng, std=0.5)
    xs = activations(1, cols, rng)
    dx, hx = dev_cols(flh, gpu, xs, col_stride_floats(cols))
    dw = flh.DeviceBuffer.from_array(np.resize(w, (rows, cols)), gpu)
    dy = flh.DeviceBuffer(4 * rows)
    dy.zero(gpu)
    flh.stream_dot(F32, dw, rows, cols, dx, dy, gpu)
    want = np.zeros(rep, np.float32)
    orc.stream_dot(F32, w.view(np.uint8).reshape(-1), rep, cols, hx, want, fast=True, threads=8)
    got = dy.download(np.float32, rows, gpu)
    dw.close()
    assert np.array_equal(bits(got), bits(np.resize(want, rows)))
