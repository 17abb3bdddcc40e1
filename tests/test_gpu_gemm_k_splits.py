"""fp16 GEMMs of few 32 x 32 tiles and a long K, which split K over workgroups and
merge in the same launch, against float64: partial tiles, a last split that is
partial or one K step, every layout, operands of dword alignment, batches and
epilogues; back to back, as each launch leaves the shared counters at 0."""
from __future__ import annotations

import numpy as np
import pytest

from test_gpu_gemm_tiles import assert_product, operands

pytestmark = pytest.mark.gpu

SHAPES = [  # 2 splits of the most tiles; 4 with a partial tile along N; 8 with
          # partial steps; a single tile; one row; dword-aligned pitches
          (8, 4096, 4096), (16, 2040, 4104), (24, 520, 6152), (32, 32, 2048), (1, 1024, 8192),
          (64, 64, 5000), (10, 514, 3586)]


@pytest.mark.parametrize("M,N,K", SHAPES)
@pytest.mark.parametrize("tl,tr", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_gemm_f16_k_splits(ipus, oracle, ctx, M, N, K, tl, tr):
    a, b, af, bf = operands(ipus, oracle, M, N, K, tl, tr, 1, True)
    da, db = ctx.upload(a), ctx.upload(b)
    outs = [ctx.upload(np.full(M * N + 8, 0x7E00, np.uint16)) for _ in range(3)]
    for out in outs:
        ctx.launch("ipu_stack_gemm_f16", out, [da, db], [1, M, N, K, tl, tr, 0, 0])
    raw = [out.download(np.uint16) for out in outs]
    assert np.all(raw[0][M * N:] == 0x7E00)  # nothing stored past C
    assert_product(oracle.f16_to_f32(raw[0][:M * N]).reshape(1, M, N), af, bf, K)
    assert np.array_equal(raw[0], raw[1]) and np.array_equal(raw[0], raw[2])
    for x in (da, db, *outs):
        x.free()


@pytest.mark.parametrize("shared", [True, False])
@pytest.mark.parametrize("epilogue", ["gelu", "add", "add_rows", "add_odd"])
def test_gemm_f16_k_splits_epilogues(ipus, oracle, ctx, shared, epilogue):
    """The fused epilogues give the bits of the product followed by the GELU or
    Add kernel, also where the addend keeps the batches from being folded
    (add_rows: one matrix for all) or is read by element (add_odd)."""
    B, M, N, K = 3, 5, 392, 4104
    a, b, af, bf = operands(ipus, oracle, M, N, K, 0, 0, B, shared)
    da, db = ctx.upload(a), ctx.upload(b)
    n = B * M * N
    product, want, fused = (ctx.alloc(n * 2) for _ in range(3))
    scalars = [B, M, N, K, 0, 0, M * K, 0 if shared else K * N]
    ctx.launch("ipu_stack_gemm_f16", product, [da, db], scalars)
    got = oracle.f16_to_f32(product.download(np.uint16)).reshape(B, M, N)
    assert_product(got, af, bf, K)
    if epilogue == "gelu":
        ctx.launch("ipu_stack_gemm_f16_gelu", fused, [da, db], scalars)
        ctx.launch("ipus_gelu_f16", want, [product], [n])
        expected = want.download(np.uint16)
    else:
        pitch = N + 3 if epilogue == "add_odd" else N
        matrices = 1 if epilogue == "add_rows" else B
        addend = ipus.synth_f16(matrices * M * pitch, 72, 3, 0, 1.0)
        dd = ctx.upload(addend)
        ctx.launch("ipu_stack_gemm_f16_accumulate", fused, [da, db, dd],
                   scalars + [M * pitch if matrices > 1 else 0, pitch])
        rows = oracle.f16_to_f32(addend).reshape(matrices, M, pitch)[:, :, :N]
        expected = (rows + got).astype(np.float16).view(np.uint16).reshape(-1)
        dd.free()
    assert np.array_equal(fused.download(np.uint16), expected)
    for x in (da, db, product, want, fused):
        x.free()


@pytest.mark.parametrize("M,N,K", [(8, 4096, 4096), (16, 1000, 1028), (32, 32, 640), (1, 1024, 8192),
                                   (64, 64, 2049), (10, 515, 1795)])
@pytest.mark.parametrize("tl,tr", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_gemm_f32_k_splits(ipus, ctx, M, N, K, tl, tr):
    """fp32: an fp32 sum of K rounded products, each within 2^-24 of the running
    magnitude."""
    rng = np.random.default_rng(73)
    a, b = rng.uniform(-1, 1, M * K).astype(np.float32), rng.uniform(-1, 1, K * N).astype(np.float32)
    af = a.astype(np.float64).reshape((K, M) if tl else (M, K))
    bf = b.astype(np.float64).reshape((N, K) if tr else (K, N))
    af, bf = af.T if tl else af, bf.T if tr else bf
    da, db = ctx.upload(a), ctx.upload(b)
    outs = [ctx.upload(np.full(M * N + 4, 7.5, np.float32)) for _ in range(3)]
    for out in outs:
        ctx.launch("ipu_stack_gemm_f32", out, [da, db], [1, M, N, K, tl, tr, 0, 0])
    raw = [out.download(np.float32) for out in outs]
    assert np.all(raw[0][M * N:] == 7.5)  # nothing stored past C
    got = raw[0][:M * N].reshape(M, N).astype(np.float64)
    assert np.all(np.abs(got - af @ bf) <= np.abs(af) @ np.abs(bf) * (K + 8) * 2.0 ** -24)
    assert np.array_equal(raw[0], raw[1]) and np.array_equal(raw[0], raw[2])
    for x in (da, db, *outs):
        x.free()
