"""x that two fp16 limbs on one scale per 256 columns cannot hold -- an element far
above the rest of its block over a zero weight, infinities, NaN -- where the batched
kernels stand in for the fp32 ones: two vectors on a large matrix, and more than 64,
in chunks of 32 and of 64 columns.

Tolerance of the finite case: an element is used exactly or with at least 10 bits,
and four neighbours together with at least 23, so what is left is the sums' rounding:
2^-18 of sum_c |w_rc x_c| over the columns whose weight is not zero (some 40
roundings of partial sums of 2^-24 each).  The other cases are compared with the fp32
kernels (two vectors on a small matrix), value for value where one is not finite.
"""
import ctypes

import numpy as np
import pytest

import oracle as O
from juno_amd import _lib
from juno_amd import matvec as mv
from test_gpu_numerics import run, weights_zero_at
from test_gpu_wide_batch import upload
from test_oracle_q2q3 import random_blocks

pytestmark = pytest.mark.gpu

# rows of the packed image, copies of it below each other, cols, B
TWO = (325, 20, 4096, 2)
WIDE32 = (300, 1, 1024, 65)
WIDE64 = (290, 70, 512, 100)
CASES = [(t, *TWO) for t in (O.Q4_K, O.Q5_K, O.Q8_0)] + [
    (t, *WIDE32) for t in (O.Q4_K, O.Q5_K, O.Q6_K, O.Q8_0, O.Q2_K, O.Q3_K)] + [
    (t, *WIDE64) for t in (O.Q4_K, O.Q8_0, O.Q2_K)]


def planned(dev, B):
    kernel, ksplit = ctypes.c_int(), ctypes.c_int()
    assert _lib.load().jh_qmatvec_batched_plan(1, (ctypes.c_void_p * 1)(dev.handle), B, ctypes.byref(kernel),
                                               ctypes.byref(ksplit)) == 0
    return kernel.value


def packed(qtype, rows, copies, cols, big, seed):
    """Weights that are zero in every row at the columns `big` (Q2_K, Q3_K: in the
    rows where they come out zero), and their values."""
    raw = random_blocks(qtype, rows, cols, seed) if qtype in (O.Q2_K, O.Q3_K) else O.quantize(
        qtype, weights_zero_at(qtype, rows, cols, big, seed, whole_subblock=False))
    deq = O.dequantize(qtype, raw, rows, cols).astype(np.float64).reshape(rows, cols)
    return np.tile(raw.reshape(rows, -1), (copies, 1)).reshape(-1), deq


@pytest.mark.parametrize("big", [1e9, 1e12])
@pytest.mark.parametrize("qtype,rows,copies,cols,B", CASES)
def test_outlier_over_zero_weight(qtype, rows, copies, cols, B, big):
    rng = np.random.default_rng(7)
    at = np.arange(0, cols, 512) + rng.integers(0, 256, cols // 512)
    raw, deq = packed(qtype, rows, copies, cols, at, 70 + qtype)
    X = rng.standard_normal((B, cols)).astype(np.float32)
    X[::2, at] = big
    with upload(qtype, rows * copies, cols, raw) as dev:
        assert planned(dev, B)
        Y = run(dev, X, rows * copies).reshape(B, copies, rows)
    zero = np.all(deq[:, at] == 0.0, axis=1) if qtype not in (O.Q2_K, O.Q3_K) else np.full(rows, False)
    if not zero.any():  # one outlier alone, and the rows that have no weight there
        at = at[:1]
        X[::2] = rng.standard_normal(X[::2].shape).astype(np.float32)
        X[::2, at] = big
        with upload(qtype, rows * copies, cols, raw) as dev:
            Y = run(dev, X, rows * copies).reshape(B, copies, rows)
        zero = deq[:, at[0]] == 0.0
    assert zero.sum() >= 2
    ref, S = X.astype(np.float64) @ deq[zero].T, np.abs(X.astype(np.float64)) @ np.abs(deq[zero]).T
    worst = np.max(np.abs(Y[:, :, zero] - ref[:, None]) / (2.0 ** -18 * S[:, None]))
    print(qtype, B, big, "rows", zero.sum(), "worst / bound", worst, flush=True)
    assert worst <= 1.0


@pytest.mark.parametrize("qtype,rows,copies,cols,B", CASES)
def test_not_finite(qtype, rows, copies, cols, B):
    """Infinities and NaN in some of the vectors: those come out as the fp32 kernels
    give them, and the others as without them, bit for bit."""
    rng = np.random.default_rng(8)
    raw = random_blocks(qtype, rows, cols, 9) if qtype in (O.Q2_K, O.Q3_K) else O.quantize(
        qtype, (rng.standard_normal(rows * cols) * 0.02).astype(np.float32))
    X = rng.standard_normal((B, cols)).astype(np.float32)
    Z = X.copy()
    Z[0, [3, cols - 7]] = np.inf, np.inf
    bad = [0]
    if B > 2:
        Z[B - 1, 300] = -np.inf
        Z[5, 77] = np.nan
        Z[6, [10, 200]] = np.inf, -np.inf
        bad += [5, 6, B - 1]
    good = [j for j in range(B) if j not in bad]
    with upload(qtype, rows * copies, cols, np.tile(raw.reshape(rows, -1), (copies, 1)).reshape(-1)) as dev:
        assert planned(dev, B)
        Y, W = run(dev, X, rows * copies).reshape(B, copies, rows), run(dev, Z, rows * copies).reshape(B, copies, rows)
    assert np.array_equal(W[good].view(np.uint32), Y[good].view(np.uint32))
    with upload(qtype, rows, cols, raw) as dev:
        assert not planned(dev, 2)
        for j in bad:
            ref = run(dev, Z[[j, good[0]]], rows)[0]
            assert not np.isfinite(ref).any()
            got = W[j]
            assert np.array_equal(np.isnan(got), np.broadcast_to(np.isnan(ref), got.shape)), (j, qtype)
            assert np.all((got == ref) | np.isnan(ref)), (j, qtype)
    if qtype in (O.Q8_0, O.Q6_K):
        assert np.isinf(W[0]).any()
