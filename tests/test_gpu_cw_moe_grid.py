"""Grouped experts on fewer workgroups than experts (a device of few CUs: FLH_CW's
third value caps the grid): every routed expert is still computed, bitwise."""
import numpy as np
import pytest

from oracle import Q8_0, Q4_K, col_stride_floats, row_bytes
from util import activations, sane_rows, tuned
from test_gpu_parity import bits, dev_cols, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cap,ntok,top_k,experts", [(64, 16, 8, 128), (64, 65, 1, 65), (7, 4, 2, 8), (1, 2, 1, 2), (255, 128, 2, 256)])
@pytest.mark.parametrize("fmt", [Q8_0, Q4_K])
def test_every_expert_is_computed(flh, orc, gpu, fmt, cap, ntok, top_k, experts):
    say("cw moe grid", fmt, cap, ntok, top_k, experts)
    rows, cols, rng = 33, 512, np.random.default_rng(experts + cap)
    pairs, eb = ntok * top_k, rows * row_bytes(fmt, cols)
    ids = rng.permutation(np.resize(np.arange(experts), pairs)).astype(np.uint32)   # all of them, if there are pairs enough
    w = sane_rows(fmt, experts * rows, cols, rng)
    xs = activations(ntok, cols, rng, outliers=True)
    st = (col_stride_floats(cols) + 3) & ~3
    y0 = rng.standard_normal(pairs * rows).astype(np.float32)
    dx, _ = dev_cols(flh, gpu, xs, st)
    flh.act_q8(dx, cols, gpu, nx=ntok, xstride=st)
    dw, dy = flh.DeviceBuffer.from_array(w, gpu), flh.DeviceBuffer.from_array(y0, gpu)
    with tuned(flh, FLH_CW="2,0,%d" % cap):
        flh.moe_dot(fmt, dw, eb, rows, cols, flh.DeviceBuffer.from_array(ids, gpu), ntok, top_k, experts, dx, st, False, dy,
                    rows, gpu)
        got = dy.download(np.float32, y0.size, gpu)
    xq, want = orc.act_q8_cols(xs, st), y0.copy()
    for i, e in enumerate(ids):
        orc.stream_dot(fmt, w[e * eb:(e + 1) * eb], rows, cols, xq[i // top_k * st:], want[i * rows:(i + 1) * rows], xstride=st,
                       ystride=rows)
    assert np.array_equal(bits(got), bits(want))
