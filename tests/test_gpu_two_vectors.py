"""Two vectors on either side of the size from which they take the MFMA kernels,
single matrices, row ranges, a group and the SwiGLU pair, eager and captured on a
stream without a workspace; and what is refused without scratch buffers.

Tolerance as for the other batches: 2^-18 of the absolute sum of a row's terms plus
2^-18 of their root sum of squares at the column's largest |x|.
"""
import ctypes

import numpy as np
import pytest

import oracle as O
from juno_amd import _lib
from juno_amd import matvec as mv
from test_gpu_wide_batch import check, fresh_stream, upload, weights

pytestmark = pytest.mark.gpu
P = ctypes.c_void_p




@pytest.mark.parametrize("captured", [False, True])
@pytest.mark.parametrize("qtype,rows,cols,lo,mfma", [
    (O.Q4_K, 6347, 4096, 0, False), (O.Q4_K, 6348, 4096, 0, True), (O.Q4_K, 1950, 14336, 37, False),
    (O.Q4_K, 2600, 14336, 37, True), (O.Q5_K, 4096, 8704, 0, False), (O.Q5_K, 4097, 8192, 0, True),
    (O.Q8_0, 8465, 3072, 0, True), (O.Q8_0, 7161, 3072, 0, False), (O.Q8_0, 7162, 3072, 0, True),
    (O.Q8_0, 13000, 2080, 0, False), (O.Q5_K, 33100, 1024, 300, True), (O.Q6_K, 6500, 4096, 0, False)])
def test_two_vectors(qtype, rows, cols, lo, mfma, captured):
    import torch
    L = _lib.load()
    kernel, ksplit = ctypes.c_int(), ctypes.c_int()
    assert L.jh_qmatvec_batched_plan_shape(qtype, cols, lo, rows, 2, ctypes.byref(kernel), ctypes.byref(ksplit)) == 0
    assert (kernel.value > 0) == mfma
    raw = weights(qtype, rows, cols, 3)
    X = np.random.default_rng(4).standard_normal((2, cols)).astype(np.float32)
    n = rows - lo
    with upload(qtype, rows, cols, raw) as dev:
        dx, y, z = torch.from_numpy(X).cuda(), torch.zeros(2, n, device="cuda"), torch.zeros(2, n, device="cuda")
        st = fresh_stream() if captured else torch.cuda.current_stream()
        torch.cuda.synchronize()
        with torch.cuda.stream(st):
            g = torch.cuda.CUDAGraph()
            if captured:
                g.capture_begin()
            assert L.jh_qmatvec_batched_dev(dev.handle, P(dx.data_ptr()), 2, P(y.data_ptr()), lo, rows, P(st.cuda_stream)) == 0
            if captured:
                g.capture_end()
                for _ in range(3):
                    y.zero_()
                    g.replay()
            assert L.jh_qmatvec_batched_noalloc_dev(dev.handle, P(dx.data_ptr()), 2, P(z.data_ptr()), lo, rows,
                                                    P(st.cuda_stream)) == 0, _lib.last_error()
        st.synchronize()
        if not captured:
            assert torch.equal(y, z)
    deq = O.dequantize(qtype, raw, rows, cols).reshape(rows, cols)[lo:].astype(np.float64)
    check(y.cpu().numpy(), X, deq, (qtype, rows, cols, captured))


@pytest.mark.parametrize("rows,cols,fused", [(4096, 2560, True), (5120, 2560, True), (3417, 2048, False), (3418, 2048, True)])
@pytest.mark.parametrize("captured", [False, True])
def test_two_vector_swiglu(rows, cols, fused, captured):
    import torch
    L = _lib.load()
    raws = [weights(O.Q4_K, rows, cols, 8 + i) for i in range(2)]
    X = np.random.default_rng(6).standard_normal((2, cols)).astype(np.float32)
    with upload(O.Q4_K, rows, cols, raws[0]) as gate, upload(O.Q4_K, rows, cols, raws[1]) as up:
        dx = torch.from_numpy(X).cuda()
        out, a, b = (torch.zeros(2, rows, device="cuda") for _ in range(3))
        st = fresh_stream() if captured else torch.cuda.current_stream()
        torch.cuda.synchronize()

        def call(pa, pb):
            return L.jh_qmatvec_batched_swiglu_dev(gate.handle, up.handle, P(dx.data_ptr()), 2, P(out.data_ptr()), pa, pb,
                                                   P(st.cuda_stream))

        assert call(None, None) == _lib.JH_EINVAL  # two vectors need the scratch buffers, whatever the kernel
        with torch.cuda.stream(st):
            g = torch.cuda.CUDAGraph()
            if captured:
                g.capture_begin()
            assert call(P(a.data_ptr()), P(b.data_ptr())) == 0, _lib.last_error()
            if captured:
                g.capture_end()
                for _ in range(3):
                    out.zero_()
                    g.replay()
        st.synchronize()
        Y = out.cpu().numpy().astype(np.float64)
        if not captured:  # the pair kernel leaves the scratch buffers alone
            assert bool((a == 0).all() and (b == 0).all()) == fused
    dg, du = (O.dequantize(O.Q4_K, r, rows, cols).reshape(rows, cols).astype(np.float64) for r in raws)
    x64 = X.astype(np.float64)
    u, v = x64 @ dg.T, x64 @ du.T
    silu = u / (1.0 + np.exp(-u))
    # the two sums' errors carried through silu (slope at most 1.1) and the product, and the product's own rounding
    eps = [2.0 ** -18 * (np.abs(x64) @ np.abs(d).T + np.sqrt(cols) * np.abs(d).max(1)[None] * np.abs(x64).max(1)[:, None])
           for d in (dg, du)]
    bound = 1.1 * eps[0] * np.abs(v) + np.abs(silu) * eps[1] + 2 * eps[0] * eps[1] + 2.0 ** -20 * np.abs(silu * v)
    assert np.max(np.abs(Y - silu * v) / bound) <= 1.0


@pytest.mark.parametrize("rows,mfma", [((3400, 17, 0), False), ((3400, 19, 0), True), ((1024, 1024, 1371), True)])
def test_two_vector_group(rows, mfma):
    """A group on either side of its limit (14 M weights), all members at the bar of one."""
    import torch
    L, cols = _lib.load(), 4096
    rows = [r for r in rows if r]
    raws = [weights(t, r, cols, 50 + i) for i, (t, r) in enumerate(zip((O.Q4_K, O.Q8_0, O.Q5_K), rows))]
    devs = [upload(t, r, cols, w) for t, r, w in zip((O.Q4_K, O.Q8_0, O.Q5_K), rows, raws)]
    n = len(devs)
    hs = (P * n)(*[d.handle for d in devs])
    kernel, ksplit = ctypes.c_int(), ctypes.c_int()
    assert L.jh_qmatvec_batched_plan(n, hs, 2, ctypes.byref(kernel), ctypes.byref(ksplit)) == 0
    assert (kernel.value > 0) == mfma
    X = np.random.default_rng(51).standard_normal((2, cols)).astype(np.float32)
    dx, ys = torch.from_numpy(X).cuda(), [torch.zeros(2, r, device="cuda") for r in rows]
    torch.cuda.synchronize()
    assert L.jh_qmatvec_batched_group_dev(n, hs, (P * n)(*[dx.data_ptr()] * n), 2, (P * n)(*[y.data_ptr() for y in ys]), None) == 0
    torch.cuda.synchronize()
    for t, r, w, y in zip((O.Q4_K, O.Q8_0, O.Q5_K), rows, raws, ys):
        check(y.cpu().numpy(), X, O.dequantize(t, w, r, cols).reshape(r, cols).astype(np.float64), (t, r, mfma))
    for d in devs:
        d.close()


@pytest.mark.parametrize("B", [2, 3, 17])
@pytest.mark.parametrize("rows,cols", [(2600, 2048), (10753, 2048), (3073, 5120)])
def test_swiglu_pair_has_the_groups_bits(rows, cols, B):
    """The pair kernel against the grouped call and silu * up, also where the pair's
    rows together fill another number of row tiles than each matrix's do, and below the
    pair's limit."""
    import torch
    L = _lib.load()
    raws = [weights(O.Q4_K, rows, cols, 80 + i) for i in range(2)]
    x = torch.from_numpy(np.random.default_rng(81).standard_normal((B, cols)).astype(np.float32)).cuda()
    out, a, b, want = (torch.zeros(B, rows, device="cuda") for _ in range(4))
    torch.cuda.synchronize()
    with upload(O.Q4_K, rows, cols, raws[0]) as gate, upload(O.Q4_K, rows, cols, raws[1]) as up:
        assert L.jh_qmatvec_batched_swiglu_dev(gate.handle, up.handle, P(x.data_ptr()), B, P(out.data_ptr()), P(a.data_ptr()),
                                               P(b.data_ptr()), None) == 0, _lib.last_error()
        torch.cuda.synchronize()
        assert L.jh_qmatvec_batched_group_dev(2, (P * 2)(gate.handle, up.handle), (P * 2)(x.data_ptr(), x.data_ptr()), B,
                                              (P * 2)(a.data_ptr(), b.data_ptr()), None) == 0, _lib.last_error()
        assert L.jh_silu_mul_dev(P(a.data_ptr()), P(b.data_ptr()), B * rows, P(want.data_ptr()), None) == 0
        torch.cuda.synchronize()
    assert torch.equal(out, want)
