"""hipStreamPerThread is one handle for a stream per thread: calls on it from several
threads overlap, so each thread has a workspace (split-K partials, counters) of its
own, and an ended thread's serves the next one.
"""
import ctypes
import os
import threading
import time

import numpy as np
import pytest

import oracle as O
from juno_amd import _lib
from juno_amd import matvec as mv
from test_gpu_wide_batch import upload, weights

pytestmark = pytest.mark.gpu
P = ctypes.c_void_p
PER_THREAD = P(2)  # hipStreamPerThread


def workspace(L):
    cap, base = ctypes.c_size_t(), P()
    assert L.jh_stream_workspace_info(0, PER_THREAD, ctypes.byref(cap), ctypes.byref(base)) == 0
    return base.value


def in_threads(fns):
    out, errors = [None] * len(fns), []

    def body(i):
        try:
            out[i] = fns[i]()
        except BaseException as e:  # noqa: BLE001 - reported by the test
            errors.append(e)

    ts = [threading.Thread(target=body, args=(i,)) for i in range(len(fns))]
    for t in ts:
        t.start()
    for t in ts:
        t.join(60)
    assert not errors, errors
    # a joined thread still has its thread-local destructors to run
    end = time.monotonic() + 20
    while any(os.path.exists(f"/proc/self/task/{t.native_id}") for t in ts):
        assert time.monotonic() < end
        time.sleep(0.01)
    return out


@pytest.mark.parametrize("B", [2, 16, 100])
def test_a_workspace_per_thread(B):
    import torch
    L = _lib.load()
    rows, cols = (6656, 4096) if B == 2 else (2048, 4096)  # K split
    raw = weights(O.Q4_K, rows, cols, 30)
    rng = np.random.default_rng(31)
    X = [torch.from_numpy(rng.standard_normal((B, cols)).astype(np.float32)).cuda() for _ in range(3)]
    Y = [torch.zeros(B, rows, device="cuda") for _ in X]
    with upload(O.Q4_K, rows, cols, raw) as dev:
        kernel, ksplit = ctypes.c_int(), ctypes.c_int()
        assert L.jh_qmatvec_batched_plan(1, (P * 1)(dev.handle), B, ctypes.byref(kernel), ctypes.byref(ksplit)) == 0
        assert kernel.value == 1 and ksplit.value > 1
        refs = []
        for x, y in zip(X, Y):
            assert L.jh_qmatvec_batched_dev(dev.handle, P(x.data_ptr()), B, P(y.data_ptr()), 0, rows, None) == 0
            torch.cuda.synchronize()
            refs.append(y.clone())
            y.zero_()
        torch.cuda.synchronize()
        meet = threading.Barrier(len(X))

        def work(i):
            meet.wait(30)
            for _ in range(40):
                rc = L.jh_qmatvec_batched_dev(dev.handle, P(X[i].data_ptr()), B, P(Y[i].data_ptr()), 0, rows, PER_THREAD)
                assert rc == 0, _lib.last_error()
            base = workspace(L)
            meet.wait(30)  # no thread ends, and gives its workspace back, before all have theirs
            return base

        first = in_threads([lambda i=i: work(i) for i in range(len(X))])
        torch.cuda.synchronize()
        assert None not in first and len(set(first)) == len(X)
        for y, ref in zip(Y, refs):
            assert torch.equal(y, ref)
        # the threads have ended: the next ones take their workspaces and allocate none
        second = in_threads([lambda i=i: work(i) for i in range(len(X))])
        torch.cuda.synchronize()
        assert set(second) == set(first)
        for y, ref in zip(Y, refs):
            assert torch.equal(y, ref)


def test_a_captured_workspace_is_not_handed_on():
    """A graph captured on a thread's stream keeps that workspace's addresses, so it is
    not the next thread's after the thread has ended."""
    import torch
    L = _lib.load()
    rows, cols, B = 2048, 4096, 16
    raw = weights(O.Q4_K, rows, cols, 32)
    x, y = torch.randn(B, cols, device="cuda"), torch.zeros(B, rows, device="cuda")
    torch.cuda.synchronize()
    with upload(O.Q4_K, rows, cols, raw) as dev:

        def call():
            assert L.jh_qmatvec_batched_dev(dev.handle, P(x.data_ptr()), B, P(y.data_ptr()), 0, rows, PER_THREAD) == 0

        def capture():
            call()
            g = P()
            assert L.hipStreamBeginCapture(PER_THREAD, 1) == 0  # thread-local mode
            call()
            assert L.hipStreamEndCapture(PER_THREAD, ctypes.byref(g)) == 0
            return workspace(L), g

        def eager():
            call()
            return workspace(L)

        (base, g), = in_threads([capture])
        others = [in_threads([eager])[0] for _ in range(4)]
        torch.cuda.synchronize()
        assert base and base not in others
        assert L.hipGraphDestroy(g) == 0


@pytest.mark.parametrize("B", [2, 16])
def test_host_calls_give_their_workspace_back(B):
    """Host-pointer calls run on a stream per thread; its workspace (8 MB and more) ends
    with the thread."""
    import torch
    rows, cols, n = 6656, 4096, 8
    raw = weights(O.Q4_K, rows, cols, 33)
    X = np.random.default_rng(34).standard_normal((B, cols)).astype(np.float32)
    meet = threading.Barrier(n)
    be = mv.GpuContext.shared(0).create_mat_vec()
    with upload(O.Q4_K, rows, cols, raw) as dev:

        def work():
            y = np.asarray(be.sgemv_batched(dev, X, 0, rows)).copy()
            meet.wait(30)  # all alive at once
            return y

        want = in_threads([work] * n)
        torch.cuda.synchronize()
        free0 = torch.cuda.mem_get_info()[0]
        got = in_threads([work] * n)
        torch.cuda.synchronize()
        assert all(np.array_equal(a.view(np.uint32), want[0].view(np.uint32)) for a in want + got)
        held = []

        def hold():
            be.sgemv_batched(dev, X, 0, rows)
            meet.wait(30)
            if not held:
                held.append(torch.cuda.mem_get_info()[0])
            meet.wait(30)

        in_threads([hold] * n)
        torch.cuda.synchronize()
        assert free0 - held[0] >= n << 22  # theirs while they live
        assert free0 - torch.cuda.mem_get_info()[0] < 8 << 20
