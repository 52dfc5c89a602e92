"""IQ2_XXS and IQ3_XXS on the chain-per-wave matrix-core kernel, bitwise against
the oracle where its plan can go wrong: one row, partial 16-row tiles, several
tiles per workgroup, partial last chunks (1 to 3 of 4 superblocks), rows at
every 2-byte offset from a 16-byte boundary, 1-16 columns, grouped experts."""
import numpy as np
import pytest

from oracle import IQ2_XXS, IQ3_XXS, col_stride_floats, row_bytes
from util import activations, sane_rows, tuned
from test_gpu_parity import bits, dev_cols, say

pytestmark = pytest.mark.gpu

FMTS = [IQ2_XXS, IQ3_XXS]
MASK = 0x7F


def check(flh, orc, gpu, fmt, rows, cols, nx, pad=0, slot=False, shift=0):
    rng = np.random.default_rng(fmt * 1000 + rows + cols + nx)
    rb, ys = rows * row_bytes(fmt, cols), rows + pad
    w = sane_rows(fmt, rows * (3 if slot else 1), cols, rng)
    y0 = rng.standard_normal((nx - 1) * ys + rows).astype(np.float32)
    xs = activations(nx, cols, rng, outliers=True)
    st = (col_stride_floats(cols) + 3) & ~3
    dx, hx = dev_cols(flh, gpu, xs, st)
    flh.act_q8(dx, cols, gpu, nx=nx, xstride=st)
    dy = flh.DeviceBuffer.from_array(y0, gpu)
    dw = flh.DeviceBuffer.from_array(np.concatenate([np.zeros(shift, np.uint8), w]), gpu)
    ids = flh.DeviceBuffer.from_array(np.array([2], np.uint32), gpu) if slot else None
    flh.stream_dot(fmt, dw.ptr + shift, rows, cols, dx, dy, gpu, nx=nx, xstride=st, ystride=ys, id_slot=ids,
                   estride=rb if slot else 0, i8_mask=MASK)
    want = y0.copy()
    orc.stream_dot(fmt, w[2 * rb:] if slot else w, rows, cols, orc.act_q8_cols(xs, st), want, nx=nx, xstride=st,
                   ystride=ys, threads=8, i8_mask=MASK)
    assert np.array_equal(bits(dy.download(np.float32, y0.size, gpu)), bits(want))


@pytest.mark.parametrize("rows,cols,nx", [
    (1, 256, 1), (15, 512, 2), (16, 768, 3), (17, 1024, 4), (33, 1280, 5), (100, 2304, 8), (300, 2816, 16),
    (4096, 1024, 2), (8200, 256, 7), (16500, 512, 1), (9000, 1792, 9), (70, 14336, 6), (40, 16384, 1)])
@pytest.mark.parametrize("fmt", FMTS)
@pytest.mark.parametrize("wgs", [0, 1])                # workgroups per CU (0: the default)
def test_cw_iq_bitwise(flh, orc, gpu, wgs, fmt, rows, cols, nx):
    say("cw iq", fmt, rows, cols, nx, wgs)
    with tuned(flh, FLH_CW="2,%d" % wgs):
        check(flh, orc, gpu, fmt, rows, cols, nx, pad=nx % 3)


@pytest.mark.parametrize("rows,cols,nx", [(300, 2048, 1), (300, 2304, 1), (300, 4096, 2), (5000, 4096, 16)])
@pytest.mark.parametrize("fmt", FMTS)
def test_default_route(flh, orc, gpu, fmt, rows, cols, nx):
    say("cw iq route", fmt, rows, cols, nx)
    check(flh, orc, gpu, fmt, rows, cols, nx, slot=rows == 300)


@pytest.mark.parametrize("shift", [2, 4, 6, 8, 10, 14])
@pytest.mark.parametrize("fmt", FMTS)
def test_cw_iq_offsets(flh, orc, gpu, fmt, shift):
    say("cw iq offset", fmt, shift)
    with tuned(flh, FLH_CW="2"):
        check(flh, orc, gpu, fmt, 37, 1280, 5, shift=shift)


@pytest.mark.parametrize("fmt", FMTS)
@pytest.mark.parametrize("ntok,top_k,experts,rows,cols,per_slot", [
    (1, 2, 8, 100, 768, False), (1, 2, 8, 100, 2048, True), (2, 1, 3, 37, 256, False), (4, 6, 64, 100, 768, True),
    (8, 2, 8, 300, 2048, False), (16, 8, 16, 33, 1280, True), (24, 2, 2, 50, 512, False), (128, 2, 200, 17, 1024, False)])
def test_cw_iq_moe(flh, orc, gpu, fmt, ntok, top_k, experts, rows, cols, per_slot):
    say("cw iq moe", fmt, ntok, top_k, experts, rows, cols, per_slot)
    rng = np.random.default_rng(fmt + ntok + rows)
    eb = rows * row_bytes(fmt, cols)
    w = sane_rows(fmt, experts * rows, cols, rng)
    ids = np.stack([rng.permutation(experts)[:top_k] for _ in range(ntok)]).astype(np.uint32)
    nxc, pairs = ntok * top_k if per_slot else ntok, ntok * top_k
    xs = activations(nxc, cols, rng, outliers=True)
    st = (col_stride_floats(cols) + 3) & ~3
    y0 = rng.standard_normal(pairs * rows).astype(np.float32)
    dx, _ = dev_cols(flh, gpu, xs, st)
    flh.act_q8(dx, cols, gpu, nx=nxc, xstride=st)
    dw, dy = flh.DeviceBuffer.from_array(w, gpu), flh.DeviceBuffer.from_array(y0, gpu)
    flh.moe_dot(fmt, dw, eb, rows, cols, flh.DeviceBuffer.from_array(ids, gpu), ntok, top_k, experts, dx, st, per_slot,
                dy, rows, gpu)
    got = dy.download(np.float32, y0.size, gpu)
    xq, want = orc.act_q8_cols(xs, st), y0.copy()
    for i, e in enumerate(ids.reshape(-1)):
        p = i if per_slot else i // top_k
        orc.stream_dot(fmt, w[e * eb:(e + 1) * eb], rows, cols, xq[p * st:], want[i * rows:(i + 1) * rows], xstride=st,
                       ystride=rows, i8_mask=MASK)
    assert np.array_equal(bits(got), bits(want))
