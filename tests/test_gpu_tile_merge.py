"""Row tiles that follow a fused norm / quantisation task join its launch:
bitwise the one-matrix result, and a tile whose output lies over the norm's
input keeps its place in the order."""
import numpy as np
import pytest

from oracle import Q4_K, Q6_K, col_stride_floats, row_bytes
from util import activations, sane_rows
from test_gpu_parity import bits, say
from test_gpu_tasks import mk

pytestmark = pytest.mark.gpu


PAD = 128                                            # floats in front of the input column


def table(flh, gpu, fmt, cols, cuts, norm, w, x, wn, over=False):
    """[RMSNORM] ACT_Q8 and the row tiles [cuts] of one matrix; over: the output
    starts PAD floats before the input column x.  Returns the output and the
    activation column."""
    T, st, rb, rows = flh.TaskKind, col_stride_floats(cols), row_bytes(fmt, cols), cuts[-1]
    buf = np.zeros(PAD + st, np.float32)
    buf[PAD:PAD + cols] = x
    db = flh.DeviceBuffer.from_array(buf, gpu)
    dx = db.ptr + 4 * PAD
    dn = flh.DeviceBuffer.from_array(np.zeros(st, np.float32), gpu)
    dwn = flh.DeviceBuffer.from_array(wn, gpu)
    dw = flh.DeviceBuffer.from_array(w, gpu)
    dy = flh.DeviceBuffer.from_array(np.zeros(rows, np.float32), gpu)
    a = dn.ptr if norm else dx
    y = db.ptr if over else dy.ptr
    tasks, p = [], flh.HostBuffer(256)
    if norm:
        v = p.view(flh.RmsNormP)
        v.wnorm, v.x, v.y, v.eps, v.n = dwn.ptr, dx, dn.ptr, 1e-5, cols
        tasks.append(mk(flh, T.RMSNORM, aux=p.ptr))
    tasks.append(mk(flh, T.ACT_Q8, x=a, y=a + flh.xq_offset(cols), rows=cols // 32, cols=cols))
    for r0, r1 in zip([0] + cuts[:-1], cuts):
        tasks.append(mk(flh, T.STREAM_DOT, fmt=fmt, w=dw.ptr + r0 * rb, w_bytes=(r1 - r0) * rb, x=a, y=y + 4 * r0,
                        rows=r1 - r0, cols=cols, nx=1))
    flh.exec_tasks(tasks, gpu)
    act = dn.download(np.float32, st, gpu) if norm else db.download(np.float32, st, gpu, offset=4 * PAD)
    return (db if over else dy).download(np.float32, rows, gpu), act


@pytest.mark.parametrize("fmt,cols,cuts,norm", [(Q4_K, 1024, [512, 1024, 1536], True), (Q4_K, 4096, [1, 700, 701], True),
                                                (Q4_K, 2816, [64, 128], False), (Q6_K, 1024, [300, 301, 900], False),
                                                (Q6_K, 2048, [512, 600], True)])
def test_merged_tiles_bitwise(flh, orc, gpu, fmt, cols, cuts, norm):
    say("tile merge", fmt, cols, cuts, norm)
    rng = np.random.default_rng(cols + len(cuts))
    w, x = sane_rows(fmt, cuts[-1], cols, rng), activations(1, cols, rng, outliers=True)[0]
    wn = (1 + 0.1 * rng.standard_normal(cols)).astype(np.float32)
    got, act = table(flh, gpu, fmt, cols, cuts, norm, w, x, wn)
    one, act1 = table(flh, gpu, fmt, cols, cuts[-1:], norm, w, x, wn)
    assert np.array_equal(bits(got), bits(one)) and np.array_equal(bits(act), bits(act1))
    want = np.zeros(cuts[-1], np.float32)
    orc.stream_dot(fmt, w, cuts[-1], cols, act, want, xstride=act.size, ystride=cuts[-1])
    assert np.array_equal(bits(got), bits(want))


def test_tile_over_the_norm_input_stays_out(flh, orc, gpu):
    """The second tile's outputs lie over the norm's input column: it runs after
    the first tile's launch has read that column."""
    cols, cuts = 1024, [PAD, 2 * PAD]
    rng = np.random.default_rng(5)
    w, x = sane_rows(Q4_K, 2 * PAD, cols, rng), activations(1, cols, rng)[0]
    wn = np.ones(cols, np.float32)
    ref, _ = table(flh, gpu, Q4_K, cols, cuts, True, w, x, wn)
    got, _ = table(flh, gpu, Q4_K, cols, cuts, True, w, x, wn, over=True)
    want = ref.copy()
    want[PAD:] += x[:PAD]
    assert np.array_equal(bits(got), bits(want))
