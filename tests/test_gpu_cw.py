"""Several columns on the chain-per-wave matrix-core kernel (k_dot_cw), bitwise
against the oracle at the edges of its plan: one row, partial 16-row tiles,
several tiles per workgroup, partial last chunks (512 columns for Q8_0 / Q5_0,
1024 for the K formats), fewer superblocks than chains, 2-16 columns, the
expert slot, and Q6_K rows at every 2-byte offset from a 16-byte boundary."""
import numpy as np
import pytest

from oracle import Q8_0, Q5_0, Q4_K, Q6_K, col_stride_floats, row_bytes
from util import activations, sane_rows, tuned
from test_gpu_parity import bits, dev_cols, say

pytestmark = pytest.mark.gpu

FMTS = [Q8_0, Q5_0, Q4_K, Q6_K]
SHAPES = [(1, 256, 2), (15, 512, 3), (16, 768, 4), (17, 1024, 5), (33, 1280, 8), (100, 2304, 9), (300, 2816, 16),
          (4096, 1024, 2), (8200, 256, 7), (16500, 512, 4), (9000, 1792, 16), (70, 14336, 8), (40, 16384, 3)]


def check(flh, orc, gpu, fmt, rows, cols, nx, pad=0, slot=False, shift=0):
    rng = np.random.default_rng(fmt * 1000 + rows + cols + nx)
    rb = rows * row_bytes(fmt, cols)
    w = sane_rows(fmt, rows * (3 if slot else 1), cols, rng)
    ys = rows + pad
    y0 = rng.standard_normal((nx - 1) * ys + rows).astype(np.float32)
    xs = activations(nx, cols, rng, outliers=True)
    st = (col_stride_floats(cols) + 3) & ~3
    dx, hx = dev_cols(flh, gpu, xs, st)
    flh.act_q8(dx, cols, gpu, nx=nx, xstride=st)
    dy = flh.DeviceBuffer.from_array(y0, gpu)
    dw = flh.DeviceBuffer.from_array(np.concatenate([np.zeros(shift, np.uint8), w]), gpu)
    ids = flh.DeviceBuffer.from_array(np.array([2], np.uint32), gpu) if slot else None
    flh.stream_dot(fmt, dw.ptr + shift, rows, cols, dx, dy, gpu, nx=nx, xstride=st, ystride=ys, id_slot=ids,
                   estride=rb if slot else 0)
    want = y0.copy()
    orc.stream_dot(fmt, w[2 * rb:] if slot else w, rows, cols, orc.act_q8_cols(xs, st), want, nx=nx, xstride=st,
                   ystride=ys, threads=8)
    assert np.array_equal(bits(dy.download(np.float32, y0.size, gpu)), bits(want))


@pytest.mark.parametrize("rows,cols,nx", SHAPES)
@pytest.mark.parametrize("fmt", FMTS)
@pytest.mark.parametrize("wgs", [0, 1])                # workgroups per CU (0: the default)
def test_cw_bitwise(flh, orc, gpu, wgs, fmt, rows, cols, nx):
    say("cw", fmt, rows, cols, nx, wgs)
    with tuned(flh, FLH_CW="2,%d" % wgs):
        check(flh, orc, gpu, fmt, rows, cols, nx, pad=nx % 3)


@pytest.mark.parametrize("rows,cols", [(4080, 4352), (4081, 4352), (4100, 4096), (4111, 8448), (4097, 14592)])
@pytest.mark.parametrize("fmt", [Q8_0, Q5_0])
def test_one_wide_column(flh, orc, gpu, fmt, rows, cols):
    """One column on either side of the line (more than 4096 columns, a tile per CU)."""
    say("cw one column", fmt, rows, cols)
    check(flh, orc, gpu, fmt, rows, cols, 1)


@pytest.mark.parametrize("fmt", FMTS)
def test_cw_expert_slot(flh, orc, gpu, fmt):
    say("cw slot", fmt)
    with tuned(flh, FLH_CW="2"):
        check(flh, orc, gpu, fmt, 160, 2048, 6, slot=True)


@pytest.mark.parametrize("shift", [2, 4, 6, 10, 14])
def test_cw_q6_offsets(flh, orc, gpu, shift):
    say("cw q6 offset", shift)
    with tuned(flh, FLH_CW="2"):
        check(flh, orc, gpu, Q6_K, 37, 1280, 5, shift=shift)


@pytest.mark.parametrize("fmt", FMTS)
@pytest.mark.parametrize("ntok,top_k,experts,rows,cols,per_slot", [
    (2, 1, 3, 37, 256, False), (4, 6, 64, 100, 768, True), (8, 2, 8, 300, 2048, False), (16, 8, 16, 33, 1280, True),
    (24, 2, 2, 50, 512, False), (128, 2, 200, 17, 1024, False)])
def test_cw_moe_bitwise(flh, orc, gpu, fmt, ntok, top_k, experts, rows, cols, per_slot):
    """Grouped experts: one to many pairs per expert (several passes of 4, 8 or
    16 columns), workgroups without rows, unrouted experts."""
    say("cw moe", fmt, ntok, top_k, experts, rows, cols, per_slot)
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
    with tuned(flh, FLH_CW="2"):
        flh.moe_dot(fmt, dw, eb, rows, cols, flh.DeviceBuffer.from_array(ids, gpu), ntok, top_k, experts, dx, st, per_slot,
                    dy, rows, gpu)
        got = dy.download(np.float32, y0.size, gpu)
    xq, want = orc.act_q8_cols(xs, st), y0.copy()
    for i, e in enumerate(ids.reshape(-1)):
        p = i if per_slot else i // top_k
        orc.stream_dot(fmt, w[e * eb:(e + 1) * eb], rows, cols, xq[p * st:], want[i * rows:(i + 1) * rows], xstride=st,
                       ystride=rows, i8_mask=0x7F)
    assert np.array_equal(bits(got), bits(want))
