"""Products of more tiles than one grid dimension holds (2^32 work-items): tall
narrow ones, and contiguous batches that run as one such product."""
from __future__ import annotations

import numpy as np
import pytest

from test_gpu_gemm_tiles import assert_product

pytestmark = pytest.mark.gpu

PERIOD, N, K = 65521, 8, 8  # the left operand repeats after PERIOD (a prime) rows


@pytest.mark.parametrize("dtype,batches,rows", [
    ("f16", 1, 2 ** 29 + 37), ("f32", 1, 2 ** 29 + 37), ("f16", 32768, 16384)])
def test_gemm_tall(ipus, oracle, ctx, dtype, batches, rows):
    f16 = dtype == "f16"
    size = 2 if f16 else 4
    synth = ipus.synth_f16 if f16 else ipus.synth_f32
    wide = (lambda x: oracle.f16_to_f32(x).astype(np.float64)) if f16 else (lambda x: x.astype(np.float64))
    raw = np.uint16 if f16 else np.float32
    pattern, b = synth(PERIOD * K, 91, 1, 0, 1.0), synth(K * N, 91, 2, 0, 1.0)
    total, row = batches * rows, K * size
    left, right = ctx.alloc(total * row), ctx.upload(b)
    first = ctx.upload(pattern)
    ctx.launch("ipu_stack_copy", left, [first], [PERIOD * row])
    filled = PERIOD
    while filled < total:  # whole periods, so the copied rows go on where the filled ones end
        n = min(filled, total - filled, 2 ** 31 // row // PERIOD * PERIOD)
        ctx.launch("ipu_stack_copy", left.ptr + filled * row, [left], [n * row])
        filled += n
    guard = np.full(8, 9.0, np.float16 if f16 else np.float32).view(raw)
    out = ctx.alloc(total * N * size + guard.nbytes)
    past = ctx.upload(guard)
    ctx.launch("ipu_stack_copy", out.ptr + total * N * size, [past], [guard.nbytes])
    ctx.launch(f"ipu_stack_gemm_{dtype}", out, [left, right],
               [batches, rows, N, K, 0, 0, rows * K if batches > 1 else 0, 0])
    window = ctx.alloc(1024 * N * size)
    # Both ends, the tiles around multiples of 2^22 tiles of 32 and 64 rows, and some between.
    starts = [0, total - 1024] + [(i << 27) - 512 for i in range(1, 4)]
    starts += np.random.default_rng(1).integers(0, total - 1024, 20).tolist()
    for at in starts:
        ctx.launch("ipu_stack_copy", window, [out.ptr + at * N * size], [window.nbytes])
        got = wide(window.download(raw)).reshape(1, 1024, N)
        rows64 = wide(pattern).reshape(PERIOD, K)[(at + np.arange(1024)) % PERIOD]
        if f16:
            assert_product(got, rows64[None], wide(b).reshape(1, K, N), K)
        else:
            want, magnitude = rows64 @ wide(b).reshape(K, N), np.abs(rows64) @ np.abs(wide(b).reshape(K, N))
            # fp32 products and sums, each within 2^-24 of the running magnitude
            assert np.all(np.abs(got[0] - want) <= magnitude * (K + 2) * 2.0 ** -24), at
    ctx.launch("ipu_stack_copy", past, [out.ptr + total * N * size], [guard.nbytes])
    assert np.array_equal(past.download(raw), guard)  # nothing stored past C
    for x in (left, right, first, out, past, window):
        x.free()
