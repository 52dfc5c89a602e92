"""Activation columns at 4-byte boundaries (quantised elsewhere and copied) on the
chain-per-wave kernel, dense and grouped, bitwise against the oracle: every
offset from a 16-byte boundary, column strides that move it, whole and partial
last chunks (1-4 superblocks), through the default routing."""
import numpy as np
import pytest

from oracle import Q4_K, Q6_K, col_stride_floats, row_bytes
from util import activations, sane_rows
from test_gpu_parity import bits, say

pytestmark = pytest.mark.gpu


def columns(flh, orc, gpu, xs, cols, off, gap):
    """Quantised columns `off` floats into a buffer that ends with the last one."""
    st = (col_stride_floats(cols) + 3) & ~3
    xq = orc.act_q8_cols(xs, st)
    used, ust = flh.x_alloc_bytes(cols) // 4, st + gap
    buf = np.zeros(off + (len(xs) - 1) * ust + used, np.float32)
    for p in range(len(xs)):
        buf[off + p * ust:off + p * ust + used] = xq[p * st:p * st + used]
    return flh.DeviceBuffer.from_array(buf, gpu), xq, st, ust


@pytest.mark.parametrize("off,gap", [(1, 0), (2, 1), (3, 2), (0, 3)])
@pytest.mark.parametrize("rows,cols,nx", [(40, 256, 3), (100, 512, 16), (33, 768, 8), (300, 1024, 5), (4100, 1280, 9)])
@pytest.mark.parametrize("fmt", [Q4_K, Q6_K])
def test_dense(flh, orc, gpu, fmt, rows, cols, nx, off, gap):
    say("cw unaligned", fmt, rows, cols, nx, off, gap)
    rng = np.random.default_rng(rows + cols + off)
    w, y0 = sane_rows(fmt, rows, cols, rng), rng.standard_normal(nx * rows).astype(np.float32)
    dx, xq, st, ust = columns(flh, orc, gpu, activations(nx, cols, rng, outliers=True), cols, off, gap)
    dw, dy = flh.DeviceBuffer.from_array(w, gpu), flh.DeviceBuffer.from_array(y0, gpu)
    flh.stream_dot(fmt, dw, rows, cols, dx.ptr + 4 * off, dy, gpu, nx=nx, xstride=ust, ystride=rows)
    want = y0.copy()
    orc.stream_dot(fmt, w, rows, cols, xq, want, nx=nx, xstride=st, ystride=rows, threads=8)
    assert np.array_equal(bits(dy.download(np.float32, y0.size, gpu)), bits(want))


@pytest.mark.parametrize("off,gap", [(1, 0), (2, 1), (3, 2), (0, 3)])
@pytest.mark.parametrize("rows,cols,ntok,top_k,experts,per_slot", [
    (40, 256, 4, 2, 3, False), (33, 1536, 3, 6, 64, True), (100, 768, 24, 2, 2, False), (50, 1280, 16, 8, 16, True)])
@pytest.mark.parametrize("fmt", [Q4_K, Q6_K])
def test_grouped(flh, orc, gpu, fmt, rows, cols, ntok, top_k, experts, per_slot, off, gap):
    say("cw moe unaligned", fmt, rows, cols, ntok, top_k, experts, off, gap)
    rng = np.random.default_rng(rows + cols + off)
    pairs, eb = ntok * top_k, rows * row_bytes(fmt, cols)
    nxc = pairs if per_slot else ntok
    ids = np.concatenate([rng.permutation(experts)[:top_k] for _ in range(ntok)]).astype(np.uint32)
    w, y0 = sane_rows(fmt, experts * rows, cols, rng), rng.standard_normal(pairs * rows).astype(np.float32)
    dx, xq, st, ust = columns(flh, orc, gpu, activations(nxc, cols, rng, outliers=True), cols, off, gap)
    dw, dy = flh.DeviceBuffer.from_array(w, gpu), flh.DeviceBuffer.from_array(y0, gpu)
    flh.moe_dot(fmt, dw, eb, rows, cols, flh.DeviceBuffer.from_array(ids, gpu), ntok, top_k, experts, dx.ptr + 4 * off, ust,
                per_slot, dy, rows, gpu)
    want = y0.copy()
    for i, e in enumerate(ids):
        p = i if per_slot else i // top_k
        orc.stream_dot(fmt, w[e * eb:(e + 1) * eb], rows, cols, xq[p * st:], want[i * rows:(i + 1) * rows], xstride=st,
                       ystride=rows)
    assert np.array_equal(bits(dy.download(np.float32, y0.size, gpu)), bits(want))
