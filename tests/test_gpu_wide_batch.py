"""More than 64 vectors: the MFMA kernels in column chunks (64 columns, with Q6_K or
Q3_K in the launch 32), at the edges of the chunks, ragged row tiles, K split and
not, one matrix and groups of mixed formats.

Tolerance as for the smaller batches: 2^-18 of the absolute sum of a row's terms
(some 40 roundings of partial sums) plus 2^-18 of their root sum of squares at the
column's largest |x| (the 22-bit split of x, 30 standard deviations).
"""
import ctypes

import numpy as np
import pytest

import oracle as O
from juno_amd import _lib
from juno_amd import matvec as mv
from test_gpu_numerics import run
from test_oracle_q2q3 import random_blocks

pytestmark = pytest.mark.gpu

TYPES = [O.Q4_K, O.Q5_K, O.Q6_K, O.Q8_0, O.Q2_K, O.Q3_K]


def weights(qtype, rows, cols, seed):
    if qtype in (O.Q2_K, O.Q3_K):
        return random_blocks(qtype, rows, cols, seed)
    return O.quantize(qtype, (np.random.default_rng(seed).standard_normal(rows * cols) * 0.02).astype(np.float32))


def check(Y, X, deq, label):
    ref = X.astype(np.float64) @ deq.T
    S = np.abs(X.astype(np.float64)) @ np.abs(deq).T
    rss = np.sqrt(deq.shape[1]) * np.abs(deq).max(1)[None, :] * np.abs(X).max(1).astype(np.float64)[:, None]
    worst = np.max(np.abs(Y.astype(np.float64) - ref) / (2.0 ** -18 * (S + rss)))
    print(label, "worst / bound", worst, flush=True)
    assert worst <= 1.0


def fresh_stream():
    """A stream that has never been used (torch's streams come round again from a pool,
    with the workspace of their earlier use); it stays for the process."""
    import torch
    s = ctypes.c_void_p()
    assert _lib.load().hipStreamCreateWithFlags(ctypes.byref(s), 1) == 0  # non-blocking
    return torch.cuda.ExternalStream(s.value)


def upload(qtype, rows, cols, raw):
    return mv.GpuContext.shared(0).create_mat_vec().upload_quant(
        mv.QuantizedTensor("w", qtype, rows * cols, raw.tobytes()), rows, cols)


@pytest.mark.parametrize("qtype", TYPES)
@pytest.mark.parametrize("rows,cols,B", [(300, 256, 65), (300, 2048, 96), (257, 1024, 97), (31, 4096, 128), (520, 512, 130)])
def test_wide_batch(qtype, rows, cols, B):
    raw = weights(qtype, rows, cols, B)
    deq = O.dequantize(qtype, raw, rows, cols).astype(np.float64).reshape(rows, cols)
    X = np.random.default_rng(B).standard_normal((B, cols)).astype(np.float32)
    L = _lib.load()
    with upload(qtype, rows, cols, raw) as dev:
        Y = run(dev, X, rows)
        check(Y, X, deq, (qtype, rows, cols, B))
        # without allocation: the same kernels, bit for bit
        import torch
        dx, dy = torch.from_numpy(X).cuda(), torch.empty(B, rows, device="cuda")
        rc = L.jh_qmatvec_batched_noalloc_dev(dev.handle, ctypes.c_void_p(dx.data_ptr()), B,
                                              ctypes.c_void_p(dy.data_ptr()), 0, rows, None)
        assert rc == 0, _lib.last_error()
        torch.cuda.synchronize()
        assert np.array_equal(dy.cpu().numpy().view(np.uint32), Y.view(np.uint32))


@pytest.mark.parametrize("types", [(O.Q4_K, O.Q4_K, O.Q6_K), (O.Q4_K, O.Q8_0), (O.Q5_K, O.Q2_K, O.Q4_K, O.Q8_0)])
@pytest.mark.parametrize("captured", [False, True])
def test_wide_group(types, captured):
    """A group in one launch; and captured on a stream that has no workspace yet, where
    nothing may be allocated: the call is taken all the same."""
    import torch
    cols, B, rows = 1024, 100, [300, 64, 257, 33][:len(types)]
    raws = [weights(t, r, cols, 7 + i) for i, (t, r) in enumerate(zip(types, rows))]
    X = np.random.default_rng(5).standard_normal((B, cols)).astype(np.float32)
    devs = [upload(t, r, cols, w) for t, r, w in zip(types, rows, raws)]
    n, P, L = len(types), ctypes.c_void_p, _lib.load()
    dx = torch.from_numpy(X).cuda()
    ys = [torch.zeros(B, r, device="cuda") for r in rows]
    st = fresh_stream() if captured else torch.cuda.current_stream()
    torch.cuda.synchronize()

    def call():
        rc = L.jh_qmatvec_batched_group_dev(n, (P * n)(*[d.handle for d in devs]), (P * n)(*[dx.data_ptr()] * n), B,
                                            (P * n)(*[y.data_ptr() for y in ys]), P(st.cuda_stream))
        assert rc == 0, _lib.last_error()

    with torch.cuda.stream(st):
        if captured:
            g = torch.cuda.CUDAGraph()
            with torch.cuda.graph(g, stream=st):
                call()
            for _ in range(3):
                for y in ys:
                    y.zero_()
                g.replay()
        else:
            call()
    st.synchronize()
    for t, r, w, y in zip(types, rows, raws, ys):
        check(y.cpu().numpy(), X, O.dequantize(t, w, r, cols).astype(np.float64).reshape(r, cols), (t, r, captured))
    for d in devs:
        d.close()


def layout(qtype, rows, cols, B):
    out = (ctypes.c_int * 13)()
    assert _lib.load().jh_qmatvec_batched_layout_shape(qtype, cols, 0, rows, B, out, 13) == 0
    return dict(zip(("kernel", "ksplit", "ksb", "columns", "chunks"), out))


@pytest.mark.parametrize("qtype", [O.Q4_K, O.Q5_K, O.Q8_0, O.Q2_K])
@pytest.mark.parametrize("rows,cols,B", [(20300, 512, 100), (20300, 512, 127), (20300, 1024, 128), (20300, 1024, 130)])
def test_chunks_of_64(qtype, rows, cols, B):
    """Where the planner takes chunks of 64 columns: full ones, and last ones of 36, 63
    and 2."""
    assert layout(qtype, rows, cols, B)["columns"] == 64
    raw = weights(qtype, rows, cols, B)
    X = np.random.default_rng(B).standard_normal((B, cols)).astype(np.float32)
    with upload(qtype, rows, cols, raw) as dev:
        Y = run(dev, X, rows)
    check(Y, X, O.dequantize(qtype, raw, rows, cols).astype(np.float64).reshape(rows, cols), (qtype, rows, cols, B))


def test_group_in_chunks_of_64():
    import torch
    types, rows, cols, B = (O.Q4_K, O.Q8_0, O.Q5_K, O.Q2_K), (10200, 5100, 257, 4700), 512, 100
    assert layout(O.Q4_K, 256 * sum(-(-r // 256) for r in rows), cols, B)["columns"] == 64  # the group's row tiles
    raws = [weights(t, r, cols, 17 + i) for i, (t, r) in enumerate(zip(types, rows))]
    X = np.random.default_rng(18).standard_normal((B, cols)).astype(np.float32)
    devs = [upload(t, r, cols, w) for t, r, w in zip(types, rows, raws)]
    n, P = len(types), ctypes.c_void_p
    dx, ys = torch.from_numpy(X).cuda(), [torch.zeros(B, r, device="cuda") for r in rows]
    torch.cuda.synchronize()
    assert _lib.load().jh_qmatvec_batched_group_dev(n, (P * n)(*[d.handle for d in devs]), (P * n)(*[dx.data_ptr()] * n), B,
                                                    (P * n)(*[y.data_ptr() for y in ys]), None) == 0
    torch.cuda.synchronize()
    for t, r, w, y in zip(types, rows, raws, ys):
        check(y.cpu().numpy(), X, O.dequantize(t, w, r, cols).astype(np.float64).reshape(r, cols), (t, r))
    for d in devs:
        d.close()


@pytest.mark.parametrize("qtype", TYPES)
@pytest.mark.parametrize("cols", [1024, 4096])
def test_no_less_exact_than_the_fp32_kernels(qtype, cols):
    """The error of 96 vectors against 64 bits, in the norm, is no larger than that of
    the kernels that took such batches before (two vectors at a time: on a small matrix
    they still do)."""
    rows, B = 520, 96
    raw = weights(qtype, rows, cols, 90)
    X = np.random.default_rng(91).standard_normal((B, cols)).astype(np.float32)
    assert layout(qtype, rows, cols, B)["kernel"] == 1 and layout(qtype, rows, cols, 2)["kernel"] == 0
    with upload(qtype, rows, cols, raw) as dev:
        Y = run(dev, X, rows).astype(np.float64)
        Z = np.concatenate([run(dev, X[b:b + 2], rows) for b in range(0, B, 2)]).astype(np.float64)
    ref = X.astype(np.float64) @ O.dequantize(qtype, raw, rows, cols).astype(np.float64).reshape(rows, cols).T
    ours, fp32 = (np.linalg.norm(v - ref) / np.linalg.norm(ref) for v in (Y, Z))
    print(qtype, cols, "error", ours, "fp32 kernels", fp32, flush=True)
    assert ours <= fp32


@pytest.mark.parametrize("qtype,rows,cols", [(O.Q8_0, 12800, 8192), (O.Q2_K, 10240, 4096)])
def test_no_less_exact_where_k_is_not_split(qtype, rows, cols):
    """The same for long walks of one workgroup, on the first rows (row ranges of 640,
    which two vectors take on the fp32 kernels)."""
    B = 100
    assert layout(qtype, rows, cols, B)["ksplit"] == 1
    raw = weights(qtype, 640, cols, 92)
    X = np.random.default_rng(93).standard_normal((B, cols)).astype(np.float32)
    with upload(qtype, rows, cols, np.tile(raw.reshape(640, -1), (rows // 640, 1)).reshape(-1)) as dev:
        Y = run(dev, X, rows)[:, :640].astype(np.float64)
    assert layout(qtype, 640, cols, 2)["kernel"] == 0
    with upload(qtype, 640, cols, raw) as dev:
        Z = np.concatenate([run(dev, X[b:b + 2], 640) for b in range(0, B, 2)]).astype(np.float64)
    ref = X.astype(np.float64) @ O.dequantize(qtype, raw, 640, cols).astype(np.float64).reshape(640, cols).T
    ours, fp32 = (np.linalg.norm(v - ref) / np.linalg.norm(ref) for v in (Y, Z))
    print(qtype, rows, cols, "error", ours, "fp32 kernels", fp32, flush=True)
    assert ours <= fp32
