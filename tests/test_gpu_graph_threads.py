"""Graphs over the same buffers, replayed by several threads onto one stream: each
replay is whole (its clear, quantisation and dots in a row), so what is left is
the result of one."""
import ctypes
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


def test_replays_stay_whole_among_other_work(flh, gpu):
    """A graph that the runtime replays (it holds a copy) and eager calls, from
    another thread onto the same stream over the same buffers: what they read of a
    short chain's output is always that of a whole replay."""
    say("graph threads, other work")
    rows, cols, reps, rng = 64, 512, 150, np.random.default_rng(6)
    xb = np.zeros(col_stride_floats(cols), np.float32)
    xb[:cols] = activations(1, cols, rng)[0]
    dx, dw = flh.DeviceBuffer.from_array(xb, gpu), flh.DeviceBuffer.from_array(sane_rows(Q4_K, rows, cols, rng), gpu)
    dy, dz, seen = flh.DeviceBuffer(4 * rows), flh.DeviceBuffer(4 * rows), flh.DeviceBuffer(4 * rows * 2 * reps)
    short, other = flh.Graph.capture(gpu), flh.Graph.capture(gpu)
    with short:
        dy.zero(gpu)
        flh.act_q8(dx, cols, gpu)
        for _ in range(3):
            flh.stream_dot(Q4_K, dw, rows, cols, dx, dy, gpu)
    with other:
        flh.copy(dz, dy, 4 * rows, gpu)
    short.launch(gpu)
    want = dy.download(np.float32, rows, gpu)
    errors = []

    def look():
        try:
            for i in range(reps):
                other.launch(gpu)
                flh.copy(seen.ptr + 8 * rows * i, dz, 4 * rows, gpu)
                flh.copy(seen.ptr + 8 * rows * i + 4 * rows, dy, 4 * rows, gpu)
        except Exception as e:
            errors.append(e)

    th = threading.Thread(target=look)
    th.start()
    while th.is_alive():
        short.launch(gpu)
    th.join()
    got = seen.download(np.float32, rows * 2 * reps, gpu).reshape(2 * reps, rows)
    assert not errors, errors
    assert np.array_equal(bits(got), bits(np.broadcast_to(want, got.shape)))
    short.close()
    other.close()


def test_replays_on_other_streams(flh, gpu):
    """Streams that were not made by this library take the runtime's form."""
    say("graph, other streams")
    rows, cols, rng = 64, 512, np.random.default_rng(7)
    xb = np.zeros(col_stride_floats(cols), np.float32)
    xb[:cols] = activations(1, cols, rng)[0]
    dx, dw = flh.DeviceBuffer.from_array(xb, gpu), flh.DeviceBuffer.from_array(sane_rows(Q4_K, rows, cols, rng), gpu)
    dy, g = flh.DeviceBuffer(4 * rows), flh.Graph.capture(gpu)
    with g:
        dy.zero(gpu)
        flh.act_q8(dx, cols, gpu)
        flh.stream_dot(Q4_K, dw, rows, cols, dx, dy, gpu)
    g.launch(gpu)
    want = dy.download(np.float32, rows, gpu)
    handle, hip = ctypes.c_void_p(), flh.lib()                    # (the runtime's symbols are found through the library's)
    assert hip.hipStreamCreateWithFlags(ctypes.byref(handle), 1) == 0   # 1: hipStreamNonBlocking
    theirs, null = flh.Stream.__new__(flh.Stream), flh.Stream.__new__(flh.Stream)
    theirs.handle, null.handle = handle.value, None
    gpu.sync()
    for s in (theirs, null, gpu):
        for _ in range(3):
            dy.upload(np.full(rows, 3.0, np.float32), gpu)
            g.launch(s)
            s.sync()
            assert np.array_equal(bits(dy.download(np.float32, rows, gpu)), bits(want))
    assert hip.hipStreamDestroy(handle) == 0
    g.close()
