"""The host-pointer GEMVs around the sizes where their copies change: y stored into
host memory by the kernel (up to 128 KB), copied by a kernel (up to 256 KB) or by
DMA; x by a kernel (up to 256 KB) or by DMA; sizes that are no multiple of four.
Against the device-pointer call of the same kernels, bit for bit."""
import numpy as np
import pytest

import oracle as O
from juno_amd import matvec as mv
from test_gpu_numerics import run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,cols,B", [
    (1, 32, 1), (3, 64, 1), (255, 64, 2), (32768, 32, 1), (32769, 32, 1), (65536, 32, 1), (65537, 32, 1),
    (1025, 64, 32), (5, 65536, 1), (5, 65568, 1), (3, 32768, 3)])
def test_host_call_equals_device_call(rows, cols, B):
    rng = np.random.default_rng(rows + cols + B)
    raw = O.quantize(O.Q8_0, (rng.standard_normal(rows * cols) * 0.02).astype(np.float32))
    X = rng.standard_normal((B, cols)).astype(np.float32)
    be = mv.GpuContext.shared(0).create_mat_vec()
    with be.upload_quant(mv.QuantizedTensor("w", O.Q8_0, rows * cols, raw.tobytes()), rows, cols) as dev:
        want = run(dev, X, rows)
        for _ in range(2):  # the staging buffers kept from the first call
            got = be.sgemv_batched(dev, X, 0, rows) if B > 1 else be.sgemv_quant(dev, X[0], 0, rows)[None, :]
            assert np.array_equal(np.asarray(got).reshape(B, rows).view(np.uint32), want.view(np.uint32))
