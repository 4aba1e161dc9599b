"""GPU parity of the fused dequant-GEMV (IWeightTensor.MatMul) against the oracle's float64
GEMV on the same blocks.  Tolerance: max|y - y_ref| / max|y_ref| <= 1e-3 (the stated bar for
the quantized GEMV), and the kernel is additionally held to 2e-5, which fp32 accumulation of
K <= 11008 terms meets with margin."""
import numpy as np
import pytest

import oracle as O
from tests.helpers import ALL_TYPES as TYPES, quantized, random_blocks, rel_err

pytestmark = pytest.mark.gpu

TOL = 1e-3
TIGHT = 2e-5


def _dev(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def _gemv(qt, blocks, N, K, x, m=1):
    import torch

    from smallmind_amd.quantization import GpuWeightTensor
    w = GpuWeightTensor(qt, N, K, blocks)
    xd = _dev(x.reshape(m, K))
    out = torch.empty((m, N), dtype=torch.float32, device="cuda")
    w.mat_mul(xd, out, m, K, N)
    y = out.cpu().numpy()
    w.close()
    return y


SHAPES = [(2, 256), (48, 512), (2560, 2048), (2048, 5632), (1000, 768), (3, 3072), (1030, 8192), (1024, 11008),
          (700, 8192), (1100, 6144), (1024, 16384),
          # tall matrices of rows up to 32 chunks: each half of a wave takes its own rows
          # (a ragged last row group at 9001 rows, full half-waves at K = 1024)
          (9001, 768), (8200, 256), (8192, 1024)]


@pytest.mark.parametrize("name", list(TYPES))
@pytest.mark.parametrize("N,K", SHAPES)
def test_gemv_vs_oracle_realistic(gpu, name, N, K):
    qt = TYPES[name]
    if K % O.BLOCK_ELEMS[qt]:
        pytest.skip("row length not a multiple of the block")
    W = quantized(qt, (N, K), seed=N * 7 + K)
    x = np.random.default_rng(K).normal(0, 1, K).astype(np.float32)
    y = _gemv(qt, W, N, K, x)[0]
    ref = O.gemv_f64(qt, W, N, K, x)
    err = rel_err(y, ref)
    assert err <= TOL and err <= TIGHT, err


@pytest.mark.parametrize("name", list(TYPES))
def test_gemv_vs_oracle_random_bytes(gpu, name):
    qt = TYPES[name]
    N, K = 130, 2048
    W = random_blocks(qt, N * K // O.BLOCK_ELEMS[qt], 77)
    x = np.random.default_rng(1).normal(0, 1, K).astype(np.float32)
    y = _gemv(qt, W, N, K, x)[0]
    ref = O.gemv_f64(qt, W, N, K, x)
    # per-row relative error: random fp16 scales give rows of wildly different magnitude
    Wf = O.dequant(qt, W, N * K).reshape(N, K).astype(np.float64)
    scale = np.abs(Wf) @ np.abs(x.astype(np.float64))
    assert np.all(np.abs(y - ref) <= TIGHT * scale + 1e-30)


@pytest.mark.parametrize("N,K", [(4096, 4096), (11008, 4096), (4096, 11008)])
def test_q4_0_gemv_benchmark_shapes(gpu, N, K):
    """the three Q4_0 GEMV shapes, reference nibble semantics."""
    W = quantized(O.Q4_0, (N, K), seed=N + K)
    x = np.random.default_rng(3).normal(0, 1, K).astype(np.float32)
    y = _gemv(O.Q4_0, W, N, K, x)[0]
    err = rel_err(y, O.gemv_f64(O.Q4_0, W, N, K, x))
    assert err <= TOL and err <= TIGHT, err


@pytest.mark.parametrize("name", list(TYPES))
def test_matmul_m_rows_equals_gemv_rows(gpu, name):
    """Below the matrix-core threshold (m < 4) every activation row is one GEMV pass."""
    qt = TYPES[name]
    N, K, m = 300, 512, 3
    W = quantized(qt, (N, K), seed=5)
    X = np.random.default_rng(6).normal(0, 1, (m, K)).astype(np.float32)
    Y = _gemv(qt, W, N, K, X, m=m)
    for r in range(m):
        assert np.array_equal(Y[r], _gemv(qt, W, N, K, X[r])[0])
        assert rel_err(Y[r], O.gemv_f64(qt, W, N, K, X[r])) <= TIGHT


@pytest.mark.parametrize("name", list(TYPES))
@pytest.mark.parametrize("m,N,K", [(4, 272, 512), (16, 2560, 2048), (37, 300, 768),
                                   (64, 1000, 2048), (100, 48, 5632), (16, 40, 160),
                                   (20, 8200, 256), (9, 300, 8192),
                                   # one token tile: on tall K-quant matrices the row-split
                                   # kernel with 1, 3 and 8 super-blocks per row (the LDS ring
                                   # partly filled, full, wrapping) and a ragged last row
                                   # group; the K-split kernel at 1 and 12 super-blocks
                                   (6, 300, 256), (5, 8300, 256), (12, 8200, 768),
                                   (13, 5000, 2048), (7, 4000, 3072), (8, 9000, 2048),
                                   # K >= 8192 above 8 tokens: the tile's tokens split over two
                                   # workgroups (the second with 1, 3 and 8 tokens)
                                   (16, 2100, 8192), (11, 1000, 11008),
                                   # one token tile on K-quant matrices of 16385-49152 rows:
                                   # 192-row workgroups, the last one ragged
                                   (16, 30000, 512), (7, 17000, 256),
                                   # prefill-chunk tiles: 512 / 1100 tokens on few-row, long-K
                                   # and other matrices (every 5th row checked); from 1024 tokens
                                   # the XCD panel order (1100: one token group per panel;
                                   # 2600 x 2048 at 1504 tokens: 47 token groups in panels of 3
                                   # for the K-quants, a partial last panel, 82 row tiles of
                                   # which the last is ragged)
                                   (511, 2048, 2048), (517, 2560, 2048), (1100, 1040, 5632),
                                   (1504, 2600, 2048)])
def test_matmul_matrix_core_path_vs_oracle(gpu, name, m, N, K):
    """m >= 4 rows: bf16 MFMA on exact integer codes and three-part activations; held to the
    same bounds as the GEMV, row by row (ragged m and N exercise the tile padding)."""
    qt = TYPES[name]
    if K % O.BLOCK_ELEMS[qt]:
        pytest.skip("row length not a multiple of the block")
    W = quantized(qt, (N, K), seed=m * 31 + N + K)
    X = np.random.default_rng(m + K).normal(0, 1, (m, K)).astype(np.float32)
    X[m // 2] *= 1e-3        # rows of very different magnitude in one tile
    Y = _gemv(qt, W, N, K, X, m=m)
    rows = range(m) if m <= 128 else sorted(set(range(0, m, 5)) | {m // 2, m - 1})
    for r in rows:
        err = rel_err(Y[r], O.gemv_f64(qt, W, N, K, X[r]))
        assert err <= TOL and err <= TIGHT, (r, err)


@pytest.mark.parametrize("name", list(TYPES))
def test_matmul_matrix_core_random_bytes(gpu, name):
    """Every code value and random (finite) scales through the matrix-core path."""
    qt = TYPES[name]
    N, K, m = 96, 2048, 20
    W = random_blocks(qt, N * K // O.BLOCK_ELEMS[qt], 91)
    X = np.random.default_rng(2).normal(0, 1, (m, K)).astype(np.float32)
    Y = _gemv(qt, W, N, K, X, m=m)
    Wf = O.dequant(qt, W, N * K).reshape(N, K).astype(np.float64)
    for r in range(m):
        ref = O.gemv_f64(qt, W, N, K, X[r])
        scale = np.abs(Wf) @ np.abs(X[r].astype(np.float64))
        assert np.all(np.abs(Y[r] - ref) <= TIGHT * scale + 1e-30), r


@pytest.mark.parametrize("name", [n for n in TYPES if n not in ("F16", "F32")])
@pytest.mark.parametrize("m,N,K", [(1025, 4100, 256),     # 64 x 64 wave tiles; one super-block, one token in the last tile
                                   (1100, 4160, 768),     # three super-blocks, whole row groups
                                   (700, 3100, 512),      # two waves of 64 x 32
                                   (517, 3600, 768),      # K split in two: 2 + 1 super-blocks
                                   (1030, 200, 2304),     # K split in four: 3 + 3 + 3 + 0 super-blocks
                                   (641, 70, 2048),       # few rows, many tokens (the K-split kernel)
                                   # the K-quants with mins reach the same shapes at these sizes
                                   (1313, 4100, 256), (1300, 4160, 768),
                                   (1030, 800, 2304),     # K split in four, the last part empty
                                   (6101, 70, 2048),      # few rows on the tile kernel
                                   (195, 16300, 256)])    # one workgroup of four waves per CU
def test_matmul_tile_kernel_vs_float64(gpu, name, m, N, K):
    """The tile kernel (long prompts) at the edges of its tiles and K splits, on random bytes (every
    code, scale and min value, fp16 scales of any magnitude) and rows of very different size.  Bound
    per output: fp32 accumulation of K products whose magnitudes sum to |w| . |x| (the sub-block
    sums carry a code offset of at most 4 code widths); the GEMM bound of this file."""
    import torch
    qt = TYPES[name]
    W = random_blocks(qt, N * K // O.BLOCK_ELEMS[qt], m + N)
    X = np.random.default_rng(m + K).normal(0, 1, (m, K)).astype(np.float32)
    X[m // 2] *= 1e-3
    X[3] *= 1e4
    Y = _dev(_gemv(qt, W, N, K, X, m=m)).double()
    Wf = _dev(O.dequant(qt, W, N * K).reshape(N, K)).double()
    Xd = _dev(X).double()
    ref, scale = Xd @ Wf.t(), Xd.abs() @ Wf.abs().t()
    worst = float(((Y - ref).abs() / (TIGHT * scale + 1e-30)).max())
    assert worst <= 1.0, worst


@pytest.mark.parametrize("name,m,N,K", [("Q8_0", 5, 40, 544),     # one span of 64 eight-element items and one of 4
                                        ("Q4_0", 16, 40, 4128),   # nine spans, the last of 4 items
                                        ("Q5_K", 13, 40, 8448),   # padding tokens in the last group of four
                                        ("Q4_K", 2500, 40, 2304),   # spans of 128 items, the last of 32
                                        ("Q4_K", 2500, 400, 2304),  # the same with sub-block sums
                                        ("Q6_K", 2500, 400, 2304)])  # with sums of half sub-blocks
def test_matmul_activation_spans_vs_float64(gpu, name, m, N, K):
    """Activation parts written by several workgroups per row, at ragged last spans; the GEMM bound
    of this file per output."""
    qt = TYPES[name]
    W = quantized(qt, (N, K), seed=m + K)
    X = np.random.default_rng(m + K).normal(0, 1, (m, K)).astype(np.float32)
    Y = _dev(_gemv(qt, W, N, K, X, m=m)).double()
    Wf = _dev(O.dequant(qt, W, N * K).reshape(N, K)).double()
    Xd = _dev(X).double()
    ref, scale = Xd @ Wf.t(), Xd.abs() @ Wf.abs().t()
    worst = float(((Y - ref).abs() / (TIGHT * scale + 1e-30)).max())
    assert worst <= 1.0, worst


def test_fused_equals_dequant_then_matmul(gpu):
    """The reference's live equivalence check (ExpandedQuantizationTests.cs:229-250): fused
    quantized matmul == dequantize then fp32 matmul."""
    import torch

    from smallmind_amd.quantization import GpuWeightTensor
    for qt in TYPES.values():
        N, K = 256, 1024
        W = quantized(qt, (N, K), seed=qt)
        x = np.random.default_rng(qt).normal(0, 1, K).astype(np.float32)
        w = GpuWeightTensor(qt, N, K, W)
        Wf = w.to_float32().double()
        ref = (Wf @ _dev(x).double()).cpu().numpy()
        out = torch.empty((1, N), dtype=torch.float32, device="cuda")
        w.mat_mul(_dev(x), out, 1, K, N)
        assert rel_err(out.cpu().numpy()[0], ref) <= 1e-5
        w.close()


def test_matmul_dimension_mismatch_raises(gpu):
    import torch

    from smallmind_amd.quantization import GpuWeightTensor
    w = GpuWeightTensor(O.Q8_0, 64, 256, quantized(O.Q8_0, (64, 256), 1))
    x = torch.zeros(256, device="cuda")
    y = torch.zeros(64, device="cuda")
    with pytest.raises(ValueError):
        w.mat_mul(x, y, 1, 128, 64)
    with pytest.raises(ValueError):
        w.mat_mul(x, y, 1, 256, 32)
    w.close()


def test_weight_create_refuses_matrices_past_4_gib(gpu):
    """A weight whose blocks would exceed the 4 GiB the kernels address (32-bit byte offsets) is
    refused at creation, before any allocation or copy: rows large enough to wrap the size
    arithmetic, and a plainly too large Q8_0 matrix.  The source pointer is never read."""
    import ctypes

    from smallmind_amd import _lib
    L = _lib.load()
    src = np.zeros(64, np.uint8)
    for rows, cols in [(2**60, 32), (2**33, 32), (2**20, 16384)]:
        w = ctypes.c_void_p()
        rc = L.smx_weight_create(int(O.Q8_0), ctypes.c_int64(rows), ctypes.c_int64(cols),
                                        src.ctypes.data_as(ctypes.c_void_p), 0, ctypes.byref(w))
        assert rc == -5 and not w.value, (rows, cols, rc)
        assert b"4 GiB" in L.smx_last_error()


@pytest.mark.parametrize("name", ["Q4_K", "Q8_0", "Q6_K"])
def test_host_memory_matmul_matches_oracle_and_device_api(gpu, name):
    """IWeightTensor.MatMul with the reference's host operands (smx_weight_matmul_host): numpy
    arrays in and out, m = 1 (GEMV) and m = 16 (matrix-core GEMM) against the oracle's float64
    GEMV; a run of calls with growing and shrinking m (the staging and the GEMM scratch are kept
    per weight and grow) gives the device entry point's bits; ToFloat32 into host memory is the
    oracle's dequantization bit for bit."""
    import torch

    from smallmind_amd.quantization import GpuWeightTensor
    qt = TYPES[name]
    N, K = 384, 2048
    W = quantized(qt, (N, K), seed=91)
    w = GpuWeightTensor(qt, N, K, W)
    rng = np.random.default_rng(5)
    for m in (1, 16, 40, 4, 16, 2):
        x = rng.normal(0, 1, (m, K)).astype(np.float32)
        y = w.mat_mul_host(x, m, K, N)
        yd = torch.empty((m, N), dtype=torch.float32, device="cuda")
        w.mat_mul(_dev(x), yd, m, K, N)
        torch.cuda.synchronize()
        assert np.array_equal(y, yd.cpu().numpy()), m
        if m in (1, 16):
            for r in range(m):
                assert rel_err(y[r], O.gemv_f64(qt, W, N, K, x[r])) <= TIGHT, (m, r)
    assert np.array_equal(w.to_float32_host().reshape(-1), O.dequant(qt, W, N * K))
    with pytest.raises(Exception):
        w.mat_mul_host(np.zeros((2, K + 32), np.float32), 2, K + 32, N)   # k != Cols
    w.close()


def test_weight_scratch_reuse_across_streams_and_threads(gpu):
    """The GEMM scratch of one weight serves calls on two streams from two threads: each call
    waits for the previous use, so every product is right."""
    import threading

    import torch

    from smallmind_amd.quantization import GpuWeightTensor
    qt, N, K, m = O.Q4_K, 256, 4096, 24
    W = quantized(qt, (N, K), seed=17)
    w = GpuWeightTensor(qt, N, K, W)
    xs = [np.random.default_rng(i).normal(0, 1, (m, K)).astype(np.float32) for i in range(2)]
    refs = [np.stack([O.gemv_f64(qt, W, N, K, x[r]) for r in range(m)]) for x in xs]
    errors = []

    def run(i):
        try:
            s = torch.cuda.Stream()
            with torch.cuda.stream(s):
                xd = _dev(xs[i])
                out = torch.empty((m, N), dtype=torch.float32, device="cuda")
                for _ in range(20):
                    w.mat_mul(xd, out, m, K, N)
                s.synchronize()
                if rel_err(out.cpu().numpy(), refs[i]) > TIGHT:
                    errors.append(i)
            for _ in range(5):
                if rel_err(w.mat_mul_host(xs[i], m, K, N), refs[i]) > TIGHT:
                    errors.append(10 + i)
        except Exception as e:   # noqa: BLE001
            errors.append(e)

    ts = [threading.Thread(target=run, args=(i,)) for i in range(2)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not errors, errors
    w.close()
