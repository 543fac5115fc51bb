"""Calls of the C++ host path launch without Python's interpreter lock: another thread gets on while they do."""
import sys
import threading
import time

import pytest
import torch

from nanoquant_amd import ops, packing

pytestmark = pytest.mark.gpu
CALLS = 500


def _packed(dev, n, r, m):
    signs = lambda a, b: torch.randint(0, 2, (a, b), dtype=torch.int8, device=dev) * 2 - 1
    scale = lambda k: torch.rand(k, device=dev).half() + 0.01
    return packing.marlin_nanoquant_packer(signs(n, r), signs(r, m), scale(n), scale(r), scale(m))


def _decode_args(dev):
    words = lambda a, b: torch.randint(-2 ** 31, 2 ** 31 - 1, (a, b), dtype=torch.int32, device=dev)
    half = lambda k: torch.rand(k, device=dev).half()
    return half(512), words(256, 16), half(256), words(512, 8), half(512)


@pytest.mark.parametrize("call", ["gemm_group", "gemm_group_sum", "gemm_bias", "gemv_bias"])
def test_another_thread_runs_during_a_call(dev, call):
    x, term = torch.rand(40, 512, device=dev).half(), _packed(dev, 512, 256, 512)
    decode = _decode_args(dev)
    run = {"gemm_group": lambda: ops.gemm_group_forward(x, [term]),
           "gemm_group_sum": lambda: ops.gemm_group_sum_forward(x, [[term, term]]),
           "gemm_bias": lambda: ops.gemm_forward_with_bias(x, *term, None),
           "gemv_bias": lambda: ops.gemv_forward_with_bias(x[:8], *decode, None)}[call]
    run()
    torch.cuda.synchronize()
    print(f"lock during {call}", flush=True)
    turns, stop = [0], threading.Event()

    def other():
        while not stop.is_set():
            turns[0] += 1
            time.sleep(0)
    # no thread is asked to give the lock up: the other one gets turns only while a call has let go of it.  Some 30 a call where
    # the call allocates and launches without the lock; next to none where it does not.
    interval = sys.getswitchinterval()
    thread = threading.Thread(target=other)
    sys.setswitchinterval(3600.0)
    try:
        thread.start()
        before = turns[0]
        for _ in range(CALLS):
            run()
        got = turns[0] - before
    finally:
        stop.set()
        sys.setswitchinterval(interval)
        thread.join()
    torch.cuda.synchronize()
    assert got > CALLS, got
