"""More than 64 vectors captured on a stream that has no workspace: the MFMA kernels
without a split of K, not the fp32 kernels.  A row's sums do not depend on the other
rows, so the captured call has the bits of an eager call on a taller matrix of the
same rows, which is planned without a split.
"""
import ctypes

import numpy as np
import pytest

import oracle as O
from juno_amd import _lib
from test_gpu_wide_batch import fresh_stream, upload, weights

pytestmark = pytest.mark.gpu
P = ctypes.c_void_p


def ksplit(dev, B):
    kernel, ks = ctypes.c_int(), ctypes.c_int()
    assert _lib.load().jh_qmatvec_batched_plan(1, (P * 1)(dev.handle), B, ctypes.byref(kernel), ctypes.byref(ks)) == 0
    return ks.value


@pytest.mark.parametrize("qtype,rows,of,cols,B", [
    (O.Q6_K, 300, 12000, 4096, 65), (O.Q6_K, 300, 12000, 4096, 100), (O.Q3_K, 300, 12000, 4096, 65),
    (O.Q3_K, 300, 12000, 4096, 100), (O.Q8_0, 10240, 12800, 8192, 100)])  # Q8_0: split, in chunks of 64; whole, of 32
def test_captured_first(qtype, rows, of, cols, B):
    import torch
    L = _lib.load()
    raw = weights(qtype, 100, cols, 40).reshape(100, -1)
    x = torch.from_numpy(np.random.default_rng(41).standard_normal((B, cols)).astype(np.float32)).cuda()
    y, tall = torch.zeros(B, rows, device="cuda"), torch.zeros(B, of, device="cuda")
    tile = np.tile(raw, (-(-of // 100), 1))
    with upload(qtype, rows, cols, tile[:rows].reshape(-1)) as dev, upload(qtype, of, cols, tile[:of].reshape(-1)) as many:
        assert ksplit(dev, B) > 1 and ksplit(many, B) == 1
        assert L.jh_qmatvec_batched_dev(many.handle, P(x.data_ptr()), B, P(tall.data_ptr()), 0, of, None) == 0
        torch.cuda.synchronize()
        st = fresh_stream()
        g = torch.cuda.CUDAGraph()

        def call():
            assert L.jh_qmatvec_batched_dev(dev.handle, P(x.data_ptr()), B, P(y.data_ptr()), 0, rows,
                                            P(st.cuda_stream)) == 0, _lib.last_error()

        with torch.cuda.stream(st):
            g.capture_begin()
            call()
            g.capture_end()
            for _ in range(3):
                y.zero_()
                g.replay()
                assert torch.equal(y, tall[:, :rows].contiguous())
                call()  # eager, with the split and the stream's workspace
        st.synchronize()
