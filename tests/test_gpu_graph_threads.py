"""Graphs over the same buffers, replayed by several threads onto one stream: each
replay is whole (its clear, quantisation and dots in a row), so what is left is
the result of one."""
import threading

import numpy as np
import pytest

from oracle import Q4_K, col_stride_floats
from util import activations, sane_rows
from test_gpu_parity import bits, say

pytestmark = pytest.mark.gpu


def test_replays_stay_whole(flh, gpu):
    say("graph threads")
    rows, cols, rng = 64, 512, np.random.default_rng(5)
    xb = np.zeros(col_stride_floats(cols), np.float32)
    xb[:cols] = activations(1, cols, rng)[0]
    dx, dw = flh.DeviceBuffer.from_array(xb, gpu), flh.DeviceBuffer.from_array(sane_rows(Q4_K, rows, cols, rng), gpu)
    dy = flh.DeviceBuffer(4 * rows)

    def issue():
        dy.zero(gpu)
        flh.act_q8(dx, cols, gpu)
        for _ in range(4):
            flh.stream_dot(Q4_K, dw, rows, cols, dx, dy, gpu)

    issue()
    want = dy.download(np.float32, rows, gpu)
    graphs = [flh.Graph.capture(gpu) for _ in range(3)]
    for g in graphs:
        with g:
            issue()
    for _ in range(10):
        ts = [threading.Thread(target=lambda g=g: [g.launch(gpu) for _ in range(20)]) for g in graphs]
        for t in ts:
            t.start()
        for t in ts:
            t.join()
        gpu.sync()
        assert np.array_equal(bits(dy.download(np.float32, rows, gpu)), bits(want))
    for g in graphs:
        g.close()
