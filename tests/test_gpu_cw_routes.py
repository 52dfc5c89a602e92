"""The lines between the chain-per-wave kernel and the formats' other kernels: on
either side of each, the default routing, the kernel by force (FLH_CW=2) and
without it (FLH_CW=0) give the oracle's bits, dense and grouped."""
import numpy as np
import pytest

from oracle import Q8_0, Q5_0, Q4_K, Q6_K, IQ2_XXS, IQ3_XXS, col_stride_floats, row_bytes
from util import activations, sane_rows, tuned
from test_gpu_parity import bits, dev_cols, say

pytestmark = pytest.mark.gpu

DENSE = [(Q4_K, 16400, 768, 9), (Q4_K, 8200, 1280, 9), (Q4_K, 20500, 1280, 5), (Q4_K, 2048, 8448, 5), (Q4_K, 2049, 8448, 5),
         (Q4_K, 256, 2304, 2), (Q4_K, 257, 2304, 2),
         (Q6_K, 4080, 8448, 2), (Q6_K, 4081, 8448, 2), (Q6_K, 2048, 2304, 3), (Q6_K, 2049, 2304, 4), (Q6_K, 1024, 3072, 8),
         (Q6_K, 1025, 3072, 5), (Q6_K, 256, 8448, 5), (Q6_K, 257, 8448, 8),
         (Q8_0, 2048, 6144, 2), (Q8_0, 2049, 6144, 2), (Q8_0, 256, 4352, 8), (Q8_0, 257, 4352, 5), (Q5_0, 2048, 2304, 2),
         (Q5_0, 1024, 8192, 6), (Q5_0, 1025, 8192, 5), (Q5_0, 1024, 8192, 7),
         (IQ2_XXS, 1024, 1280, 2), (IQ2_XXS, 1025, 1280, 2), (IQ3_XXS, 16400, 4096, 2), (IQ2_XXS, 2048, 4096, 4),
         (IQ3_XXS, 2049, 4096, 3), (IQ2_XXS, 2048, 8192, 6), (IQ3_XXS, 2048, 8192, 7), (IQ2_XXS, 256, 1280, 3),
         (IQ2_XXS, 2048, 16384, 1),
         (IQ3_XXS, 2049, 16384, 1), (IQ2_XXS, 2048, 8448, 1), (IQ3_XXS, 816, 2304, 4), (IQ2_XXS, 817, 2304, 4), (IQ3_XXS, 1024, 8448, 3), (IQ2_XXS, 1025, 8448, 4)]


@pytest.mark.parametrize("fmt,rows,cols,nx", DENSE)
def test_dense(flh, orc, gpu, fmt, rows, cols, nx):
    say("cw routes", fmt, rows, cols, nx)
    rng = np.random.default_rng(fmt + rows + cols + nx)
    w, xs = sane_rows(fmt, rows, cols, rng), activations(nx, cols, rng, outliers=True)
    y0 = rng.standard_normal(nx * rows).astype(np.float32)
    st = (col_stride_floats(cols) + 3) & ~3
    dx, _ = dev_cols(flh, gpu, xs, st)
    flh.act_q8(dx, cols, gpu, nx=nx, xstride=st)
    dw, want = flh.DeviceBuffer.from_array(w, gpu), y0.copy()
    orc.stream_dot(fmt, w, rows, cols, orc.act_q8_cols(xs, st), want, nx=nx, xstride=st, ystride=rows, i8_mask=0x7F, threads=8)
    for mode in "102":
        dy = flh.DeviceBuffer.from_array(y0, gpu)
        with tuned(flh, FLH_CW=mode):
            flh.stream_dot(fmt, dw, rows, cols, dx, dy, gpu, nx=nx, xstride=st, ystride=rows, i8_mask=0x7F)
            assert np.array_equal(bits(dy.download(np.float32, y0.size, gpu)), bits(want)), mode


@pytest.mark.parametrize("fmt", [Q8_0, Q5_0, Q4_K, Q6_K, IQ2_XXS, IQ3_XXS])
def test_longer_rows_are_refused(flh, gpu, fmt):
    """More than 16384 columns are refused whatever the rows and columns (as
    every other kernel of these formats refuses them), dense and grouped."""
    say("cw refused", fmt)
    cols, rows, E = 16640, 4200, 2
    w, x = flh.DeviceBuffer(rows * row_bytes(fmt, cols)), flh.DeviceBuffer(16 * flh.x_alloc_bytes(cols) + 256)
    y, ids = flh.DeviceBuffer(16 * rows * 4), flh.DeviceBuffer.from_array(np.array([0, 1, 1, 0], np.uint32), gpu)
    st = (col_stride_floats(cols) + 3) & ~3
    for r, nx in ((rows, 1), (rows, 2), (rows, 8), (33, 4), (rows, 16)):
        with pytest.raises(flh.FlhError):
            flh.stream_dot(fmt, w, r, cols, x, y, gpu, nx=nx, xstride=st, ystride=r, i8_mask=0x7F)
    for n, k in ((2, 2), (2, 1)):
        with pytest.raises(flh.FlhError):
            flh.moe_dot(fmt, w, 16 * row_bytes(fmt, cols), 16, cols, ids, n, k, E, x, st, False, y, 16, gpu)


@pytest.mark.parametrize("fused", [False, True])
@pytest.mark.parametrize("rows,cols,ntok,top_k,experts", [
    (64, 1024, 16, 4, 16), (256, 1024, 16, 8, 64), (257, 1024, 8, 2, 8), (1024, 2048, 2, 2, 8), (300, 2048, 4, 2, 8),
    (300, 2048, 8, 4, 64), (300, 2048, 3, 6, 64), (40, 8448, 2, 2, 4), (600, 1280, 2, 4, 16)])
@pytest.mark.parametrize("fmt", [Q8_0, Q5_0, Q6_K, IQ2_XXS, IQ3_XXS])
def test_grouped(flh, orc, gpu, fmt, rows, cols, ntok, top_k, experts, fused):
    say("cw moe routes", fmt, rows, cols, ntok, top_k, experts, fused)
    rng = np.random.default_rng(fmt + rows + cols + ntok)
    pairs, eb = ntok * top_k, rows * row_bytes(fmt, cols)
    logits = rng.standard_normal((ntok, experts)).astype(np.float32)
    ids = np.argsort(-logits, axis=1, kind="stable")[:, :top_k].astype(np.uint32)
    w, xs = sane_rows(fmt, experts * rows, cols, rng), activations(ntok, cols, rng, outliers=True)
    y0 = rng.standard_normal(pairs * rows).astype(np.float32)
    st = (col_stride_floats(cols) + 3) & ~3
    dx, _ = dev_cols(flh, gpu, xs, st)
    flh.act_q8(dx, cols, gpu, nx=ntok, xstride=st)
    dw, di, dg = flh.DeviceBuffer.from_array(w, gpu), flh.DeviceBuffer.from_array(ids, gpu), flh.DeviceBuffer(4 * pairs)
    dl, want, xq = flh.DeviceBuffer.from_array(logits, gpu), y0.copy(), orc.act_q8_cols(xs, st)
    for i, e in enumerate(ids.reshape(-1)):
        orc.stream_dot(fmt, w[e * eb:(e + 1) * eb], rows, cols, xq[i // top_k * st:], want[i * rows:(i + 1) * rows], xstride=st,
                       ystride=rows, i8_mask=0x7F)
    for mode in "102":
        dy = flh.DeviceBuffer.from_array(y0, gpu)
        with tuned(flh, FLH_CW=mode):
            if fused:
                flh.router_moe_dot(fmt, dw, eb, rows, cols, dl, ntok, experts, top_k, 1, 1.0, di, dg, dx, st, False, dy, rows, gpu)
            else:
                flh.moe_dot(fmt, dw, eb, rows, cols, di, ntok, top_k, experts, dx, st, False, dy, rows, gpu)
            assert np.array_equal(bits(dy.download(np.float32, y0.size, gpu)), bits(want)), mode
