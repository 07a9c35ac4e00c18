"""A stream's first batched call allocates its workspace.  It may come while another
thread captures a graph on a stream of its own (in the default, global mode): the call
is taken, and the capture goes on.
"""
import ctypes
import threading

import numpy as np
import pytest

import oracle as O
from juno_amd import _lib
from test_gpu_wide_batch import check, fresh_stream, upload, weights

pytestmark = pytest.mark.gpu
P = ctypes.c_void_p


@pytest.mark.parametrize("B,rows,cols", [(2, 6656, 4096), (16, 2048, 4096), (100, 2048, 4096)])
def test_first_call_while_another_thread_captures(B, rows, cols):
    import torch
    L = _lib.load()
    raw = weights(O.Q4_K, rows, cols, 60)
    X = np.random.default_rng(61).standard_normal((B, cols)).astype(np.float32)
    x, y, z = torch.from_numpy(X).cuda(), torch.zeros(B, rows, device="cuda"), torch.zeros(B, rows, device="cuda")
    eager_stream, capture_stream = fresh_stream(), fresh_stream()
    with upload(O.Q4_K, rows, cols, raw) as dev:

        def call(out, s):
            assert L.jh_qmatvec_batched_dev(dev.handle, P(x.data_ptr()), B, P(out.data_ptr()), 0, rows, s) == 0, _lib.last_error()

        call(y, P(capture_stream.cuda_stream))  # its workspace
        torch.cuda.synchronize()
        want = y.clone()
        y.zero_()
        z.zero_()
        torch.cuda.synchronize()
        graph = P()
        assert L.hipStreamBeginCapture(P(capture_stream.cuda_stream), 0) == 0  # global mode
        call(y, P(capture_stream.cuda_stream))
        errors = []

        def other():
            try:
                call(z, P(eager_stream.cuda_stream))
            except BaseException as e:  # noqa: BLE001 - reported below
                errors.append(e)

        t = threading.Thread(target=other)
        t.start()
        t.join(60)
        assert L.hipStreamEndCapture(P(capture_stream.cuda_stream), ctypes.byref(graph)) == 0
        assert not errors, errors
        torch.cuda.synchronize()
        assert torch.equal(z, want)
        exe = P()
        assert L.hipGraphInstantiate(ctypes.byref(exe), graph, None, None, 0) == 0
        for _ in range(3):
            y.zero_()
            torch.cuda.synchronize()
            assert L.hipGraphLaunch(exe, P(capture_stream.cuda_stream)) == 0
            torch.cuda.synchronize()
            assert torch.equal(y, want)
        assert L.hipGraphExecDestroy(exe) == 0 and L.hipGraphDestroy(graph) == 0
    check(z.cpu().numpy(), X, O.dequantize(O.Q4_K, raw, rows, cols).reshape(rows, cols).astype(np.float64), B)
