"""The native operators give the interpreter up: another thread runs while one of them is under way, and threads on streams of
their own get the results of one thread."""
import sys
import threading
import time

import pytest
import torch

import modular_amd as mx
from modular_amd import _lib, synth

pytestmark = pytest.mark.gpu


def test_another_thread_runs_during_native_calls(dev):
    """With a switch interval that never runs out, the counting thread only gets its turn where the calls give the lock up."""
    x = synth.activations(64, 1024, seed=1, device=dev)
    native, interval = _lib.native(), sys.getswitchinterval()
    turns, stop, ready = [0], threading.Event(), threading.Event()

    def count():
        ready.set()
        while not stop.is_set():
            turns[0] += 1
            time.sleep(0)                       # (hands the lock back)

    thread = threading.Thread(target=count)
    thread.start()
    ready.wait()
    sys.setswitchinterval(1000.0)
    try:
        before = turns[0]
        for _ in range(2000):
            native.quantize(x, 128, True, 1200.0)
        during = turns[0] - before
    finally:
        sys.setswitchinterval(interval)
        stop.set()
        thread.join()
    torch.cuda.synchronize()
    assert during > 0


def test_threads_on_their_own_streams(dev):
    cfg = mx.blockwise_fp8_config()
    w, ws = (t.to(dev) for t in synth.quantize_weight_block(synth.weights_f32(1024, 2048, seed=2)))
    xs = [synth.activations(m, 2048, seed=m, device=dev) for m in (1, 40, 130, 300)]
    want = [mx.quantized_matmul(x, w, ws, None, cfg) for x in xs]
    torch.cuda.synchronize()
    got = [[] for _ in xs]

    def work(i):
        stream = torch.cuda.Stream(dev)
        with torch.cuda.stream(stream):
            for _ in range(20):
                got[i].append(mx.quantized_matmul(xs[i], w, ws, None, cfg))
        stream.synchronize()

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(xs))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for i, results in enumerate(got):
        assert len(results) == 20 and all(torch.equal(y, want[i]) for y in results), f"{xs[i].shape[0]} tokens"
