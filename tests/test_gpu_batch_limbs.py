"""The batched kernels' x operand at its edges: the batch sizes where its layout
changes (both limbs in one MFMA up to 16 columns, two column groups from 33), and
activations whose block sums or scales leave fp16's range if they are not scaled --
all of one sign near the block's maximum, and very small.

Tolerance: the sums run in fp32 with about 40 roundings of a partial sum per output
(32 MFMAs, the folds, the super-blocks), each at most 2^-24 of sum_c |w_rc x_c|:
2^-18 of it is allowed.  x = hi + lo drops at most 2^-24 of the column's largest
|x| per element, in random directions, and a format with a min forms each weight
from parts no larger than the row's largest weight: 2^-18 of the root sum of
squares of those terms, some 30 standard deviations, is allowed.  Losing the lo
limbs would cost 2^-13 of it, and a sum out of range is off by its whole size.
"""
import numpy as np
import pytest

import oracle as O
from juno_amd import matvec as mv
from test_gpu_numerics import run
from test_oracle_q2q3 import random_blocks

pytestmark = pytest.mark.gpu

TYPES = [O.Q4_K, O.Q5_K, O.Q6_K, O.Q8_0, O.Q2_K, O.Q3_K]


@pytest.mark.parametrize("qtype", TYPES)
@pytest.mark.parametrize("B", [3, 15, 16, 17, 32, 33, 64])
@pytest.mark.parametrize("kind", ["constant", "tiny", "normal"])
def test_limb_layouts(qtype, B, kind):
    rows, cols = 300, 1024
    rng = np.random.default_rng(B * 100 + qtype)
    raw = random_blocks(qtype, rows, cols, B) if qtype in (O.Q2_K, O.Q3_K) else O.quantize(
        qtype, (rng.standard_normal(rows * cols) * 0.02 + 0.01).astype(np.float32))
    deq = O.dequantize(qtype, raw, rows, cols).astype(np.float64).reshape(rows, cols)
    X = {"constant": np.ones((B, cols)) * (1.0 + np.arange(B))[:, None] / B,
         "tiny": rng.standard_normal((B, cols)) * 2.0 ** -118,
         "normal": rng.standard_normal((B, cols))}[kind].astype(np.float32)
    be = mv.GpuContext.shared(0).create_mat_vec()
    with be.upload_quant(mv.QuantizedTensor("w", qtype, rows * cols, raw.tobytes()), rows, cols) as dev:
        Y = run(dev, X, rows).astype(np.float64)
    assert np.all(np.isfinite(Y))
    ref = X.astype(np.float64) @ deq.T
    S = np.abs(X.astype(np.float64)) @ np.abs(deq).T
    rss = np.sqrt(cols) * np.abs(deq).max(1)[None, :] * np.abs(X).max(1).astype(np.float64)[:, None]
    bound = 2.0 ** -18 * (S + rss) + 1e-44
    worst = np.max(np.abs(Y - ref) / bound)
    print(qtype, B, kind, "worst / bound", worst, flush=True)
    assert worst <= 1.0


@pytest.mark.parametrize("qtype", TYPES)
@pytest.mark.parametrize("B", [3, 17, 33, 65])
def test_sums_of_x_past_the_largest_float(qtype, B):
    """x of one sign from 2^124 on: 16 of them together are past the largest float, the
    results are not.  The bound is the other test's."""
    rows, cols = 70, 256
    rng = np.random.default_rng(B * 100 + qtype)
    raw = random_blocks(qtype, rows, cols, B) if qtype in (O.Q2_K, O.Q3_K) else O.quantize(
        qtype, (rng.standard_normal(rows * cols) * 0.002 + 0.001).astype(np.float32))
    deq = O.dequantize(qtype, raw, rows, cols).astype(np.float64).reshape(rows, cols)
    keep = np.abs(deq).sum(1) <= 7.0  # rows whose terms together stay below the largest float
    assert keep.any() and (qtype in (O.Q2_K, O.Q3_K) or keep.all())
    deq[~keep] = 0.0
    X = (np.ldexp(1.0 + rng.random((B, cols)), 124)).astype(np.float32)
    be = mv.GpuContext.shared(0).create_mat_vec()
    with be.upload_quant(mv.QuantizedTensor("w", qtype, rows * cols, raw.tobytes()), rows, cols) as dev:
        Y = run(dev, X, rows).astype(np.float64)
    assert np.all(np.isfinite(Y[:, keep]))
    ref = X.astype(np.float64) @ deq.T
    S = np.abs(X.astype(np.float64)) @ np.abs(deq).T
    rss = np.sqrt(cols) * np.abs(deq).max(1)[None, :] * np.abs(X).max(1).astype(np.float64)[:, None]
    assert np.all(np.abs(Y - ref)[:, keep] <= 2.0 ** -18 * (S + rss)[:, keep])
