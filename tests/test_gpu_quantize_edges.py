"""The device quantizers and dequantizers byte for byte against the oracle where
their lanes and roundings can go wrong: one block, a last wave that is not full,
values half way between two quants, infinities, NaN, constant and zero blocks,
subnormal scales, and outputs that are not 16-byte aligned."""
import ctypes

import numpy as np
import pytest

import oracle as O
from juno_amd import _lib
from juno_amd import matvec as mv
from test_oracle_q2q3 import random_blocks

pytestmark = pytest.mark.gpu


def values(kind, n):
    rng = np.random.default_rng(n)
    x = (rng.standard_normal(n) * 0.02).astype(np.float32)
    if kind == "halves":  # multiples of half a quant step of a range of 15, with its ends in every sub-block
        x = (rng.integers(0, 31, n) * 0.5).astype(np.float32)
        x[::16], x[1::16] = 0.0, 15.0
        x = x - np.float32(7.5)
    elif kind == "special":
        x[::7], x[1::61], x[2::83], x[3::97] = 0.0, np.inf, -np.inf, np.nan
        x[-32:] = np.nan
    elif kind == "flat":
        x = np.repeat(rng.standard_normal(n // 32).astype(np.float32), 32)
        x[: n // 2] = -np.abs(x[: n // 2])
        x[:32] = -0.0
    elif kind == "ends":  # +-max everywhere: the products round just beside the largest quant
        x = np.sign(x) * np.repeat(np.abs(x[::32]) + np.float32(3e-6), 32)
    elif kind == "tiny":
        x = x * np.float32(2.0 ** -18)
        x[: n // 2] *= np.float32(2.0 ** -110)
    return x


@pytest.mark.parametrize("qtype", [O.Q4_K, O.Q5_K, O.Q6_K, O.Q8_0])
@pytest.mark.parametrize("kind", ["normal", "halves", "special", "flat", "ends", "tiny"])
@pytest.mark.parametrize("n", [32, 256, 288, 1280, 256 * 1001])
def test_quantize_bytes(qtype, kind, n):
    import torch
    if n % O.QK[qtype]:
        pytest.skip("not a whole number of blocks")
    x = values(kind, n)
    want = O.quantize(qtype, x)
    for off in (0, 2):  # the packed image at an address that is even only
        src = torch.from_numpy(np.concatenate([np.zeros(1, np.float32), x])).cuda()[1:]  # 4-byte aligned
        dst = torch.zeros(want.size + off, device="cuda", dtype=torch.uint8)[off:]
        mv.quantize_dev(qtype, src.data_ptr(), n, dst.data_ptr(), 0)
        torch.cuda.synchronize()
        assert np.array_equal(dst.cpu().numpy(), want), (qtype, kind, n, off)


@pytest.mark.parametrize("qtype", [O.Q4_K, O.Q5_K, O.Q6_K, O.Q8_0, O.Q2_K, O.Q3_K])
@pytest.mark.parametrize("rows,cols", [(1, 256), (3, 512), (77, 1280)])
def test_dequantize_bits(qtype, rows, cols):
    import torch
    L = _lib.load()
    if qtype in (O.Q2_K, O.Q3_K):
        raw = random_blocks(qtype, rows, cols, 5)
    else:
        raw = O.quantize(qtype, values("normal", rows * cols))
    want = O.dequantize(qtype, raw, rows, cols).reshape(-1)
    be = mv.GpuContext.shared(0).create_mat_vec()
    with be.upload_quant(mv.QuantizedTensor("w", qtype, rows * cols, raw.tobytes()), rows, cols) as dev:
        buf = torch.full((rows * cols + 2,), 7.0, device="cuda")
        out = buf[1:]  # 4-byte aligned
        be.dequantize_dev(dev, out.data_ptr(), 0)
        tok = torch.tensor([rows - 1], device="cuda", dtype=torch.int32)
        row = torch.full((cols + 1,), 7.0, device="cuda")
        assert L.jh_embed_dev(dev.handle, ctypes.c_void_p(tok.data_ptr()), ctypes.c_void_p(row[1:].data_ptr()),
                                         None) == 0, _lib.last_error()
        torch.cuda.synchronize()
    got = buf.cpu().numpy()
    assert np.array_equal(got[1:-1].view(np.uint32), want.view(np.uint32))
    assert got[0] == 7.0 and got[-1] == 7.0
    assert np.array_equal(row[1:].cpu().numpy().view(np.uint32), want[-cols:].view(np.uint32))
