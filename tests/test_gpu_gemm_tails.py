"""The GEMM tile kernels over 1 to 9 K steps: four stages are filled ahead, groups of
four steps follow, and what is left runs without fetching; steps past the last one
must neither be fetched into a stage still read nor counted by a wait."""
from __future__ import annotations

import numpy as np
import pytest

from test_gpu_gemm_tiles import assert_product, operands

pytestmark = pytest.mark.gpu


def k_of(step, steps, tail):
    return step * (steps - 1) + (step if tail == 0 else tail)


@pytest.mark.parametrize("M,N,step", [(72, 88, 128), (400, 1000, 64), (1800, 2056, 64)])  # 32, 64, 128
@pytest.mark.parametrize("steps", range(1, 10))
@pytest.mark.parametrize("tail", [0, 8, 6, 5])  # whole; 16-byte, 4-byte and 2-byte aligned rows
@pytest.mark.parametrize("tr", [0, 1])
def test_gemm_f16_steps(ipus, oracle, ctx, M, N, step, steps, tail, tr):
    K = k_of(step, steps, tail)
    a, b, af, bf = operands(ipus, oracle, M, N, K, 0, tr, 1, True)
    pad = np.full(4096, 0x7E00, np.uint16)  # NaN after the operands
    da, db = (ctx.upload(np.concatenate([x, pad])) for x in (a, b))
    out = ctx.upload(np.full(M * N + 8, 0x7E00, np.uint16))
    ctx.launch("ipu_stack_gemm_f16", out, [da, db], [1, M, N, K, 0, tr, 0, 0])
    raw = out.download(np.uint16)
    assert np.all(raw[M * N:] == 0x7E00)
    rows = np.unique(np.concatenate([np.arange(0, M, 7), [M - 1]]))
    got = oracle.f16_to_f32(raw[:M * N]).reshape(1, M, N)[:, rows]
    assert_product(got, af[:, rows], bf, K)
    for x in (da, db, out):
        x.free()


@pytest.mark.parametrize("M,N,step", [(72, 88, 64), (712, 1200, 32)])  # 32, 64
@pytest.mark.parametrize("steps", range(1, 10))
@pytest.mark.parametrize("tail", [0, 4, 7])
@pytest.mark.parametrize("tl", [0, 1])
def test_gemm_f32_steps(ipus, ctx, M, N, step, steps, tail, tl):
    K = k_of(step, steps, tail)
    a, b = ipus.synth_f32(M * K, 77, 1, 0, 1.0), ipus.synth_f32(K * N, 77, 2, 0, 1.0)
    pad = np.full(4096, np.nan, np.float32)
    da, db = (ctx.upload(np.concatenate([x, pad])) for x in (a, b))
    out = ctx.upload(np.full(M * N + 8, 9.0, np.float32))
    ctx.launch("ipu_stack_gemm_f32", out, [da, db], [1, M, N, K, tl, 0, 0, 0])
    raw = out.download(np.float32)
    assert np.all(raw[M * N:] == 9.0)
    a64 = a.astype(np.float64).reshape((K, M) if tl else (M, K))
    a64, b64 = a64.T if tl else a64, b.astype(np.float64).reshape(K, N)
    rows = np.unique(np.concatenate([np.arange(0, M, 7), [M - 1]]))
    want, magnitude = a64[rows] @ b64, np.abs(a64[rows]) @ np.abs(b64)
    # fp32 products and sums, each within 2^-24 of the running magnitude
    assert np.all(np.abs(raw[:M * N].reshape(M, N)[rows] - want) <= magnitude * (K + 2) * 2.0 ** -24)
    for x in (da, db, out):
        x.free()


@pytest.mark.parametrize("M,N,K", [(1, 1, 1), (2, 1, 3), (1, 3, 2), (3, 1, 1), (1, 1, 7), (1, 1, 9), (9, 1, 1),
                                   (5, 2, 67), (1, 9, 129), (17, 3, 131), (65, 67, 1)])
@pytest.mark.parametrize("tl,tr", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_gemm_f16_operands_near_a_chunk(ipus, oracle, ctx, M, N, K, tl, tr):
    """Odd rows read at element alignment: operands of fewer elements than a 16-byte
    chunk, and ends of the operand inside one, with NaN behind them."""
    a, b, af, bf = operands(ipus, oracle, M, N, K, tl, tr, 1, True)
    pad = np.full(64, 0x7E00, np.uint16)
    da, db = (ctx.upload(np.concatenate([pad[:1], x, pad])) for x in (a, b))
    out = ctx.upload(np.full(M * N + 8, 0x7E00, np.uint16))
    ctx.launch("ipu_stack_gemm_f16", out, [da.ptr + 2, db.ptr + 2], [1, M, N, K, tl, tr, 0, 0])
    raw = out.download(np.uint16)
    assert np.all(raw[M * N:] == 0x7E00)
    assert_product(oracle.f16_to_f32(raw[:M * N]).reshape(1, M, N), af, bf, K)
    for x in (da, db, out):
        x.free()


@pytest.mark.parametrize("K", [4, 32, 36, 64])
@pytest.mark.parametrize("tl,tr", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_gemm_f32_short_sums(ipus, ctx, K, tl, tr):
    """Many tiles of a short sum run the 128 x 128 kernel, here with partial tiles."""
    M, N = 2388, 2692
    a, b = ipus.synth_f32(M * K, 78, 1, 0, 1.0), ipus.synth_f32(K * N, 78, 2, 0, 1.0)
    pad = np.full(4096, np.nan, np.float32)
    da, db = (ctx.upload(np.concatenate([x, pad])) for x in (a, b))
    out = ctx.upload(np.full(M * N + 8, 9.0, np.float32))
    ctx.launch("ipu_stack_gemm_f32", out, [da, db], [1, M, N, K, tl, tr, 0, 0])
    raw = out.download(np.float32)
    assert np.all(raw[M * N:] == 9.0)
    a64 = a.astype(np.float64).reshape((K, M) if tl else (M, K))
    b64 = b.astype(np.float64).reshape((N, K) if tr else (K, N))
    a64, b64 = a64.T if tl else a64, b64.T if tr else b64
    want, magnitude = a64 @ b64, np.abs(a64) @ np.abs(b64)
    # fp32 products and sums, each within 2^-24 of the running magnitude
    assert np.all(np.abs(raw[:M * N].reshape(M, N) - want) <= magnitude * (K + 2) * 2.0 ** -24)
    for x in (da, db, out):
        x.free()
