"""The scratch of calls that bring none: qk_matmul at M > 8 from more streams
than there are blocks, from threads that share a stream, on recreated streams,
across block sizes, under capture and after a release, each result equal bit
for bit to qk_matmul_ws on a workspace of its own."""
from __future__ import annotations

import ctypes
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

Q4, Q6 = 12, 14


class Case:
    def __init__(self, qk, oracle, qtype, K, N, M, seed):
        self.qk, self.args = qk, (qtype, K, N, M)
        self.w = qk.DeviceBuffer.from_array(oracle.synth_superblocks(qtype, N, K, seed, 0.01, 0.01))
        self.x = qk.DeviceBuffer.from_array(oracle.synth_normal(M * K, seed + 1))
        self.y = qk.DeviceBuffer(4 * M * N)
        need = qk.matmul_workspace_size(qtype, K, N, M)
        ws = qk.DeviceBuffer(need)
        self.run(None, ws, need)
        qk.synchronize()
        self.want = self.y.download(np.uint32)
        self.y.fill(0)

    def run(self, stream, ws=None, need=0):
        qtype, K, N, M = self.args
        if ws is None:
            self.qk.matmul(self.x, self.w, qtype, K, N, self.y, M, stream)
        else:
            self.qk.matmul_ws(self.x, self.w, qtype, K, N, self.y, M, ws, need, stream)

    def check(self):
        assert np.array_equal(self.y.download(np.uint32), self.want)
        self.y.fill(0)


# scratch below, at and past the 16 and 64 MiB classes: 0.6, 15.2, 17, 40 and 80 MiB
SHAPES = [(Q4, 2560, 256, 33), (Q6, 9728, 64, 400), (Q4, 4096, 96, 1040), (Q4, 9728, 64, 1040), (Q6, 9728, 32, 2060)]


def test_streams_and_sizes(gpu, oracle):
    cases = [Case(gpu, oracle, *SHAPES[i % len(SHAPES)], 20261201 + i) for i in range(11)]
    streams = [gpu.Stream() for _ in cases]
    for _ in range(3):
        for c, s in zip(cases, streams):
            c.run(s.ptr)
        gpu.synchronize()
        for c in cases:
            c.check()
        for s in streams:
            s.destroy()
        streams = [gpu.Stream() for _ in cases]
    gpu.release_scratch()
    for c in cases:  # one stream, every size in turn
        c.run(streams[0].ptr)
    gpu.synchronize()
    for c in cases:
        c.check()
    for s in streams:
        s.destroy()


def test_threads_sharing_a_stream(gpu, oracle):
    cases = [Case(gpu, oracle, *SHAPES[i % 3], 20261301 + i) for i in range(6)]
    stream = gpu.Stream()
    errors = []

    def work(c):
        try:
            for _ in range(20):
                c.run(stream.ptr)
        except Exception as e:  # noqa: BLE001
            errors.append(e)

    threads = [threading.Thread(target=work, args=(c,)) for c in cases]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    gpu.synchronize()
    assert not errors
    for c in cases:
        c.check()
    stream.destroy()


def test_captured_calls_beside_eager_ones(gpu, oracle):
    """A call recorded on a stream that already has a cached block, replayed
    on a second stream while that first stream makes eager calls of the same
    size, with nothing between them in a round: the graph shares no block."""
    a, b, c = (Case(gpu, oracle, Q4, 2560, 1024, 500 + i, 20261401 + i) for i in range(3))
    eager, replay = gpu.Stream(), gpu.Stream()
    a.run(eager.ptr)  # leaves the stream a block
    graph = gpu.Graph.capture(eager, lambda: a.run(eager.ptr))
    gpu.synchronize()
    for _ in range(6):
        for _ in range(4):
            graph.launch(replay.ptr)
            b.run(eager.ptr)
            c.run(eager.ptr)
        gpu.synchronize()
        for case in (a, b, c):
            case.check()
    graph.destroy()
    for s in (eager, replay):
        s.destroy()


@pytest.mark.parametrize("others", [0, 8])
def test_calls_while_another_stream_is_captured(gpu, oracle, others):
    """Calls on other streams, from this thread and another, neither end nor
    enter a capture, with no block allocated yet and with every block last
    used by a further stream."""
    gpu.release_scratch()
    cases = [Case(gpu, oracle, Q4, 2560, 256, 33 + i, 20261501 + i) for i in range(3)]
    used = [gpu.Stream() for _ in range(others)]
    for s in used:
        cases[0].run(s.ptr)
    gpu.synchronize()
    streams = [gpu.Stream() for _ in cases]
    errors = []

    def eager(i):
        try:
            cases[i].run(streams[i].ptr)
        except Exception as e:  # noqa: BLE001
            errors.append(e)

    def record():
        cases[0].run(streams[0].ptr)
        thread = threading.Thread(target=eager, args=(1,))
        thread.start()
        thread.join()
        eager(2)

    graph = gpu.Graph.capture(streams[0], record)
    gpu.synchronize()
    assert not errors
    cases[1].check()
    cases[2].check()
    cases[0].y.fill(0)
    for _ in range(3):
        graph.launch(streams[0].ptr)
        gpu.synchronize()
        cases[0].check()
        assert not cases[1].y.download(np.uint32).any() and not cases[2].y.download(np.uint32).any()
    graph.destroy()
    for s in used + streams:
        s.destroy()


def _free_bytes(qk):
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert qk.load().hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


def test_release_gives_the_blocks_back(gpu, oracle):
    """8 streams hold a block each; once qk_release_scratch has returned their
    memory is free on the device, and later calls run as before. (The pool takes
    and gives 2 MiB pieces, some of which it may have had: half a block of slack.)"""
    most = 8 * (16 << 20) - (8 << 20)
    case = Case(gpu, oracle, Q4, 2560, 256, 33, 20261601)
    streams = [gpu.Stream() for _ in range(8)]
    gpu.release_scratch()
    before = _free_bytes(gpu)
    for s in streams:
        case.run(s.ptr)
    gpu.synchronize()
    held = _free_bytes(gpu)
    assert before - held >= most
    case.check()
    gpu.release_scratch()
    assert _free_bytes(gpu) - held >= most
    case.run(streams[0].ptr)
    gpu.synchronize()
    case.check()
    for s in streams:
        s.destroy()


def test_per_thread_stream_holds_no_block(gpu, oracle):
    """The per-thread default stream's handle (2) names a stream of each
    thread: a block kept under it would make one thread's call wait for
    another's, so its calls keep none; two threads' results are right."""
    per_thread = 2
    cases = [Case(gpu, oracle, Q4, 2560, 256, 33 + i, 20261701 + i) for i in range(2)]
    cases[0].run(per_thread)  # (what the runtime itself allocates at first use)
    gpu.synchronize()
    gpu.release_scratch()
    gpu.synchronize()
    before = _free_bytes(gpu)
    errors = []

    def work(c):
        try:
            for _ in range(8):
                c.run(per_thread)
        except Exception as e:  # noqa: BLE001
            errors.append(e)

    threads = [threading.Thread(target=work, args=(c,)) for c in cases]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    gpu.synchronize()
    assert not errors
    assert before - _free_bytes(gpu) < 16 << 20
    for c in cases:
        c.check()
