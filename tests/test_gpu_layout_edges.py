"""Transposes and padded rearranges at sizes and addresses off the vector grid,
bit-exact against the oracle's index maps, with guard elements around the
destination and NaN patterns around the source."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

GUARD = 0x7E5A


def guarded(ctx, x, shift):
    """x at an element offset, between guard elements."""
    g = np.full(64, GUARD, np.uint16)
    return ctx.upload(np.concatenate([g[:8 + shift], x.reshape(-1), g]))


def read_guarded(buf, count, shift):
    raw = buf.download(np.uint16)
    assert np.all(raw[:8 + shift] == GUARD) and np.all(raw[8 + shift + count:] == GUARD)
    return raw[8 + shift:8 + shift + count]


@pytest.mark.parametrize("matrices,rows,cols", [
    (1, 1, 1), (1, 7, 9), (1, 8, 8), (3, 63, 65), (2, 64, 64), (1, 513, 40), (1, 729, 1152),
    (2, 1152, 729), (1, 2049, 4097), (1, 4096, 4096), (70000, 3, 5)])
@pytest.mark.parametrize("shift", [0, 1, 4])
def test_transpose_any_size_and_alignment(ipus, oracle, ctx, matrices, rows, cols, shift):
    n = matrices * rows * cols
    x = ipus.synth_f16(n, 83, 1)
    src = guarded(ctx, x, shift)
    dst = guarded(ctx, np.zeros(n, np.uint16), shift)
    ctx.launch("ipu_stack_transpose_f16", dst.ptr + 2 * (8 + shift), [src.ptr + 2 * (8 + shift)],
               [matrices, rows, cols])
    got = read_guarded(dst, n, shift)
    assert np.array_equal(got, oracle.transpose_u16(x, matrices, rows, cols).reshape(-1))
    src.free()
    dst.free()


@pytest.mark.parametrize("order,rb,cb", [(0, 0, 0), (1, 0, 0), (2, 64, 64), (2, 64, 16), (2, 16, 8),
                                         (2, 16, 20)])
@pytest.mark.parametrize("matrices,lr,pr,lc,pc", [
    (1, 1, 64, 1, 320), (1, 729, 768, 1147, 1280), (3, 17, 64, 33, 80), (2, 64, 64, 80, 80),
    (1, 33, 192, 640, 640), (1, 128, 128, 8, 160)])
@pytest.mark.parametrize("shift", [0, 3])
def test_padded_rearrange(ipus, oracle, ctx, order, rb, cb, matrices, lr, pr, lc, pc, shift):
    """Padding rows and columns are zero; the source may start at any
    element (the destination is aligned, or at any element too with shift)."""
    if cb and (pc % cb or pr % rb):
        pytest.skip("the blocks do not divide these extents")
    x = ipus.synth_f16(matrices * lr * lc, 84, 1)
    n = matrices * pr * pc
    want = oracle.rearrange_row_major_f16(x, order, matrices, lr, pr, lc, pc, rb, cb).reshape(-1)
    src = guarded(ctx, x, shift)
    for dshift in {0, shift}:
        dst = guarded(ctx, np.full(n, GUARD, np.uint16), dshift)
        ctx.launch("ipu_stack_rearrange_row_major_f16", dst.ptr + 2 * (8 + dshift),
                   [src.ptr + 2 * (8 + shift)], [lr, pr, order, lc, pc, rb, cb, matrices])
        assert np.array_equal(read_guarded(dst, n, dshift), want)
        dst.free()
    src.free()


@pytest.mark.parametrize("matrices,rows,cols,shift", [
    (12, 301, 299, 0), (12, 304, 296, 1),       # 64 x 64 tiles with partial blocks
    (70, 1001, 255, 0),                         # tall tiles, partial blocks
    (9, 301, 299, 3), (700, 65, 100, 0),        # by element: a small total, empty tiles
    (70001, 5, 13, 0), (66000, 8, 24, 0),
    (65600, 40, 40, 0)])                        # 64 x 64 tiles in two launches
def test_transpose_routes(ipus, oracle, ctx, matrices, rows, cols, shift):
    test_transpose_any_size_and_alignment(ipus, oracle, ctx, matrices, rows, cols, shift)


@pytest.mark.parametrize("rows,cols", [(1, 600_000_007), (600_000_007, 1)])
def test_transpose_of_a_long_row(ctx, rows, cols):
    """More 64-column tiles than a grid dimension holds of 512 threads."""
    n = rows * cols
    src, dst = ctx.alloc(2 * n), ctx.alloc(2 * n + 16)
    ends = np.random.default_rng(7).integers(0, 1 << 16, (3, 4096)).astype(np.uint16)
    window = ctx.alloc(ends[0].nbytes)
    starts = [0, n // 3, n - 4096]
    for x, at in zip(ends, starts):
        ctx.write(window, x)
        ctx.launch("ipu_stack_copy", src.ptr + 2 * at, [window], [window.nbytes])
    ctx.memset(dst, 0x5A)
    ctx.launch("ipu_stack_transpose_f16", dst, [src], [1, rows, cols])
    for x, at in zip(ends, starts):
        ctx.launch("ipu_stack_copy", window, [dst.ptr + 2 * at], [window.nbytes])
        assert np.array_equal(window.download(np.uint16), x), at
    ctx.launch("ipu_stack_copy", window, [dst.ptr + 2 * n], [16])
    assert np.all(window.download(np.uint16)[:8] == 0x5A5A)
    for b in (src, dst, window):
        b.free()


@pytest.mark.parametrize("matrices,rows,cols", [(70000, 3, 5), (4096, 17, 33), (1, 1, 1000000), (69967, 2, 8)])
def test_transpose_of_small_extents_keeps_the_chip_busy(ctx, matrices, rows, cols):
    """One tile per small matrix, one workgroup per CU, took 10 to 170 times as long as
    a transpose of the same elements in one matrix; a launch takes about as long."""
    n = matrices * rows * cols
    src, dst = ctx.alloc(2 * n), ctx.alloc(2 * n)

    def us(scalars):
        best = 1e9
        for _ in range(5):
            events = ctx.event_series(2)
            events.record(0)
            for _ in range(20):
                ctx.launch("ipu_stack_transpose_f16", dst, [src], scalars)
            events.record(1)
            best = min(best, float(events.durations()[0]) * 1000 / 20)
        return best

    side = int(n ** 0.5)
    assert us([matrices, rows, cols]) < 3.0 * us([1, side, side]) + 5.0
    src.free()
    dst.free()


@pytest.mark.parametrize("order", [0, 1])
@pytest.mark.parametrize("matrices,lr,pr,lc,pc", [
    (1, 24989, 24992, 3, 16), (1, 25008, 25008, 9, 16),    # either side of 400,000 elements
    (3, 2085, 2096, 50, 64), (40, 200, 208, 20, 64), (1, 1, 16, 25001, 25008)])
def test_padded_rearrange_routes(ipus, oracle, ctx, order, matrices, lr, pr, lc, pc):
    test_padded_rearrange(ipus, oracle, ctx, order, 0, 0, matrices, lr, pr, lc, pc, 3)


def test_padded_rearrange_of_one_long_row(ctx):
    """AMP-Left tiles of 32 rows for a single one: more of them than a grid dimension
    holds of 256 threads."""
    n, pc = 1_100_000_007, 1_100_000_016
    src, dst = ctx.alloc(2 * n), ctx.alloc(2 * pc)
    window = ctx.alloc(32)
    ctx.memset(src, 0x11)
    ctx.launch("ipu_stack_rearrange_row_major_f16", dst, [src], [1, 1, 0, n, pc, 0, 0, 1])
    for at in (0, n // 2 // 16 * 16, pc - 32):
        ctx.launch("ipu_stack_copy", window, [dst.ptr + 2 * at], [32])
        assert np.all(window.download(np.uint16) == 0x1111), at
    ctx.launch("ipu_stack_copy", window, [dst.ptr + 2 * (pc - 16)], [32])
    assert window.download(np.uint16).tolist() == [0x1111] * 7 + [0] * 9
    for b in (src, dst, window):
        b.free()
