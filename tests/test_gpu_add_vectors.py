"""Broadcast adds in 16-byte vectors: every shape the vector kernel takes, and
its neighbours that it does not, give the bits of numpy's elementwise sum."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SHAPES = [  # left, right, (broadcast to their common shape)
    ((64, 256), (256,)), ((64, 256), (64, 1)), ((5, 1, 24), (1, 7, 24)), ((3, 4, 8), (3, 4, 8)),
    ((2, 3, 4, 8), (3, 1, 8)), ((1,), (40,)), ((8, 1, 16, 1), (1, 6, 1, 32)),
    ((2, 1, 3, 1, 16), (1, 5, 1, 7, 16)), ((3, 20), (20,)), ((7, 33), (33,)), ((2, 5, 12), (5, 1)),
    ((1025, 1032), (1032,))]


@pytest.mark.parametrize("left,right", SHAPES)
@pytest.mark.parametrize("dtype", ["f16", "f32"])
@pytest.mark.parametrize("swap", [False, True])
def test_broadcast_add(ipus, ctx, left, right, dtype, swap):
    t = np.float16 if dtype == "f16" else np.float32
    rng = np.random.default_rng(5)
    ops = [rng.standard_normal(s).astype(t) for s in ((right, left) if swap else (left, right))]
    shape = np.broadcast_shapes(left, right)
    want = (ops[0].astype(np.float32) + ops[1].astype(np.float32)).astype(t)
    scalars = [len(shape)] + list(shape) + [1] * (6 - len(shape))
    for x in ops:
        v = np.broadcast_to(x, shape)
        scalars += [0 if n == 1 else s // x.itemsize for n, s in zip(v.shape, v.strides)]
        scalars += [0] * (6 - len(shape))
    bufs = [ctx.upload(x) for x in ops]
    out = ctx.upload(np.full(want.size + 8, 9.0, t))
    ctx.launch(f"ipu_stack_add_broadcast_{dtype}", out, bufs, scalars)
    raw = out.download(t)
    assert np.array_equal(raw[:want.size].reshape(shape), want) and np.all(raw[want.size:] == 9.0)
    # Unaligned operands give the same sums
    shifted = [ctx.upload(np.concatenate([np.zeros(1, t), x.reshape(-1)])) for x in ops]
    ctx.launch(f"ipu_stack_add_broadcast_{dtype}", out,
               [b.ptr + x.itemsize for b, x in zip(shifted, ops)], scalars)
    assert np.array_equal(out.download(t)[:want.size].reshape(shape), want)
    for b in bufs + shifted + [out]:
        b.free()


@pytest.mark.parametrize("dtype", ["f16", "f32"])
def test_broadcast_add_past_32_bit_columns(ctx, dtype):
    """A contiguous operand plus one value collapses to a single axis, here of
    2^32 + 65536 elements: columns past 2^32 read their own elements, not those
    32 bits of the column away."""
    t = np.float16 if dtype == "f16" else np.float32
    rows, columns = 65537, 65536
    size = np.dtype(t).itemsize
    left, out = ctx.alloc(rows * columns * size), ctx.alloc(rows * columns * size)
    first, last = (np.random.default_rng(i).standard_normal(columns).astype(t) for i in (1, 2))
    ends, value = [ctx.upload(first), ctx.upload(last)], ctx.upload(np.array([0.5], t))
    offsets = [0, (rows - 1) * columns * size]
    for end, at in zip(ends, offsets):
        ctx.launch("ipu_stack_copy", left.ptr + at, [end], [columns * size])
    scalars = [2, rows, columns, 1, 1, 1, 1, columns, 1, 0, 0, 0, 0] + [0] * 6
    ctx.launch(f"ipu_stack_add_broadcast_{dtype}", out, [left, value], scalars)
    for x, end, at in zip((first, last), ends, offsets):
        ctx.launch("ipu_stack_copy", end, [out.ptr + at], [columns * size])
        assert np.array_equal(end.download(t), (x.astype(np.float32) + 0.5).astype(t)), at
    for b in [left, out, value] + ends:
        b.free()
