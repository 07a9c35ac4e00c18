"""Quantizing and dequantizing more than 2^34 elements (a lane makes four: 2^32 lanes
or more, of which one launch does not run all), against the bytes of a short pattern of whole
rows that the array repeats."""
import numpy as np
import pytest

import oracle as O
from juno_amd import matvec as mv
from test_oracle_q2q3 import random_blocks

pytestmark = pytest.mark.gpu
COLS = 8192
ROWS = (1 << 34) // COLS + 3


@pytest.mark.parametrize("qtype", [O.Q8_0, O.Q4_K])
def test_quantize_large(qtype):
    import torch
    x = (np.random.default_rng(70).standard_normal(COLS) * 0.02).astype(np.float32)
    want = torch.from_numpy(O.quantize(qtype, x)).cuda()
    src = torch.from_numpy(x).cuda().expand(ROWS, COLS).contiguous()
    dst = torch.zeros(ROWS, want.numel(), device="cuda", dtype=torch.uint8)
    torch.cuda.synchronize()
    mv.quantize_dev(qtype, src.data_ptr(), src.numel(), dst.data_ptr(), 0)
    torch.cuda.synchronize()
    del src
    same = all(bool((part == want).all()) for part in dst.split(1 << 16))
    del dst
    torch.cuda.empty_cache()
    assert same


def test_dequantize_large():
    import torch
    raw = random_blocks(O.Q2_K, 1, COLS, 71)
    want = torch.from_numpy(O.dequantize(O.Q2_K, raw, 1, COLS).reshape(-1)).cuda()
    be = mv.GpuContext.shared(0).create_mat_vec()
    with be.upload_quant(mv.QuantizedTensor("w", O.Q2_K, ROWS * COLS, raw.tobytes() * ROWS), ROWS, COLS) as dev:
        out = torch.zeros(ROWS, COLS, device="cuda")
        torch.cuda.synchronize()
        be.dequantize_dev(dev, out.data_ptr(), 0)
        torch.cuda.synchronize()
    same = all(bool((part.view(torch.int32) == want.view(torch.int32)).all()) for part in out.split(1 << 16))
    del out
    torch.cuda.empty_cache()
    assert same
