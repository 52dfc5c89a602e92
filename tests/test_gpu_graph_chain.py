"""Captured graphs: short chains of kernels (launched one by one on replay), at
and past the lines of 5 kernels, 7 that stream some weights and 16 that stream many, and a capture with a copy node (the runtime's
form).  Every replay equals the eager result, with eager work, a change of the
inputs and synchronizations between the replays, on the captured stream and on
another one."""
import numpy as np
import pytest

from oracle import Q4_K, col_stride_floats
from util import activations, sane_rows
from test_gpu_parity import bits, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("layers,more,copy", [(0, 0, False), (1, 0, False), (1, 1, False), (1, 2, False), (2, 0, False),
                                              (1, 0, True), (5, 0, False), (5, 0, True), (6, 0, False), (9, 0, False)])
def test_replays_equal_eager(flh, gpu, layers, more, copy):
    replays(flh, gpu, layers, more, copy, 96, 512)


@pytest.mark.parametrize("layers,more,rows", [(1, 2, 1024), (2, 0, 1024), (2, 1, 1024), (2, 1, 12288), (5, 0, 12288),
                                              (5, 1, 12288)])
def test_replays_of_larger_matrices(flh, gpu, layers, more, rows):
    """Dots of 2.3 and 27 MiB: chains of 6 and 7 kernels past 0.5 MiB a kernel and one
    too long for that, of 8 and 16 past 12 MiB and one too long."""
    replays(flh, gpu, layers, more, False, rows, 4096)


def replays(flh, gpu, layers, more, copy, rows, cols):
    """1 + 3 * layers + more launches (and a copy): zero, then ACT_Q8, dot, dot."""
    say("graph chain", layers, more, copy)
    rng = np.random.default_rng(layers)
    st = col_stride_floats(cols)
    xb = np.zeros(st, np.float32)
    dx = flh.DeviceBuffer.from_array(xb, gpu)
    dw = [flh.DeviceBuffer.from_array(sane_rows(Q4_K, rows, cols, rng), gpu) for _ in range(max(layers, 1))]
    dy, dz = flh.DeviceBuffer(4 * rows * 2 * max(layers, 1)), flh.DeviceBuffer(4 * rows)
    out = rows * 2 * max(layers, 1)

    def issue(s):
        dy.zero(s)
        for l in range(layers):
            flh.act_q8(dx, cols, s)
            for k in range(2):
                flh.stream_dot(Q4_K, dw[l], rows, cols, dx, dy.ptr + 4 * rows * (2 * l + k), s)
        for _ in range(more):
            flh.stream_dot(Q4_K, dw[0], rows, cols, dx, dy, s)
        if copy:
            flh.copy(dz, dy, 4 * rows, s)

    g = flh.Graph.capture(gpu)
    with g:
        issue(gpu)
    other = flh.Stream()
    for i in range(4):
        xb[:cols] = activations(1, cols, rng)[0]
        dx.upload(xb, gpu)
        issue(gpu)
        want = dy.download(np.float32, out, gpu)
        dy.upload(np.full(out, 3.0, np.float32), gpu)
        gpu.sync()
        s = other if i == 2 else gpu
        g.launch(s)
        s.sync()
        assert np.array_equal(bits(dy.download(np.float32, out, gpu)), bits(want)), i
        if copy:
            assert np.array_equal(bits(dz.download(np.float32, rows, gpu)), bits(want[:rows]))
    g.close()
    other.close()
