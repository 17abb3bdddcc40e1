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
