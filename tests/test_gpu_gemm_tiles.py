"""The fp16 GEMM's 128 x 128, 64 x 64 and 32 x 32 tile kernels against float64, at
the edges of their tiles and K steps, in every layout, batch form and epilogue
(the launch picks the tile from the shape; each shape below names the tile it
was chosen for)."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def operands(ipus, oracle, M, N, K, tl, tr, batches, shared):
    a = ipus.synth_f16(batches * M * K, 71, 1, 0, 1.0)
    b = ipus.synth_f16((1 if shared else batches) * K * N, 71, 2, 0, 1.0)
    af = oracle.f16_to_f32(a).astype(np.float64).reshape((batches, K, M) if tl else (batches, M, K))
    bf = oracle.f16_to_f32(b).astype(np.float64).reshape((-1, N, K) if tr else (-1, K, N))
    af = af.transpose(0, 2, 1) if tl else af
    bf = bf.transpose(0, 2, 1) if tr else bf
    return a, b, af, bf


def assert_product(got, af, bf, K):
    """One fp16 rounding (2^-11 of the value, 2^-25 below the normal range)
    of an fp32 sum of K exact products, each addition within 2^-24 of the
    running magnitude."""
    want, magnitude = np.matmul(af, bf), np.matmul(np.abs(af), np.abs(bf))
    bound = (np.abs(want) * 2.0 ** -11 + 2.0 ** -25) * 1.001 + magnitude * (K + 2) * 2.0 ** -24
    assert np.all(np.abs(got - want) <= bound)


SHAPES = [  # tile 128: a partial tile along M and N, a partial last K step
          (1800, 2056, 584), (1792, 2048, 640),
          # tile 64: fewer than four K steps left over, partial tiles
          (520, 1160, 1160), (512, 1024, 1152),
          # tile 32: one K step and part of one, single tiles, one row of tiles
          (256, 256, 256), (8, 8, 8), (40, 72, 264), (32, 32, 128), (8, 4096, 1032)]


@pytest.mark.parametrize("M,N,K", SHAPES)
@pytest.mark.parametrize("tl,tr", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_gemm_f16_tiles(ipus, oracle, ctx, M, N, K, tl, tr):
    a, b, af, bf = operands(ipus, oracle, M, N, K, tl, tr, 1, True)
    da, db = ctx.upload(a), ctx.upload(b)
    out = ctx.upload(np.full(M * N + 8, 0x7E00, np.uint16))
    ctx.launch("ipu_stack_gemm_f16", out, [da, db], [1, M, N, K, tl, tr, 0, 0])
    raw = out.download(np.uint16)
    assert np.all(raw[M * N:] == 0x7E00)  # nothing stored past C
    assert_product(oracle.f16_to_f32(raw[:M * N]).reshape(1, M, N), af, bf, K)
    for x in (da, db, out):
        x.free()


@pytest.mark.parametrize("M,N,K", [(601, 1032, 584), (264, 392, 1160), (33, 72, 200)])
@pytest.mark.parametrize("shared", [True, False])
@pytest.mark.parametrize("epilogue", ["none", "gelu", "add"])
def test_gemm_f16_tiles_batches_and_epilogues(ipus, oracle, ctx, M, N, K, shared, epilogue):
    """Batched, the right operand shared or not; the fused epilogues give the
    bits of the product followed by the GELU or Add kernel."""
    B = 5
    a, b, af, bf = operands(ipus, oracle, M, N, K, 0, 1, B, shared)
    n = B * M * N
    da, db, out = ctx.upload(a), ctx.upload(b), ctx.alloc(n * 2)
    sc = [B, M, N, K, 0, 1, M * K, 0 if shared else K * N]
    ctx.launch("ipu_stack_gemm_f16", out, [da, db], sc)
    if epilogue == "none":
        got = oracle.f16_to_f32(out.download(np.uint16)).reshape(B, M, N)
        assert_product(got, af, bf, K)
    elif epilogue == "gelu":
        want, fused = ctx.alloc(n * 2), ctx.alloc(n * 2)
        ctx.launch("ipus_gelu_f16", want, [out], [n])
        ctx.launch("ipu_stack_gemm_f16_gelu", fused, [da, db], sc)
        assert np.array_equal(fused.download(np.uint16), want.download(np.uint16))
    else:
        d = ctx.upload(ipus.synth_f16(n, 71, 3, 0, 1.0))
        want = ctx.alloc(n * 2)
        ctx.launch("ipu_stack_add_f16", want, [out, d], [n, n, n])
        ctx.launch("ipu_stack_gemm_f16_accumulate", d, [da, db, d], sc + [M * N, N])  # in place
        assert np.array_equal(d.download(np.uint16), want.download(np.uint16))


@pytest.mark.parametrize("B,M,N,K", [(5, 141, 1032, 584), (2, 700, 1280, 1160), (7, 9, 73, 66)])
@pytest.mark.parametrize("addend", ["none", "full", "matrix", "rows"])
def test_gemm_f16_batches_as_rows(ipus, oracle, ctx, B, M, N, K, addend):
    """Contiguous batches that share the right operand run as one product of
    B M rows; an addend per matrix (which cannot) gives the same sums."""
    a, b, af, bf = operands(ipus, oracle, M, N, K, 0, 0, B, True)
    n = B * M * N
    da, db, out = ctx.upload(a), ctx.upload(b), ctx.upload(np.full(n + 8, 0x7E00, np.uint16))
    sc = [B, M, N, K, 0, 0, M * K, 0]
    ctx.launch("ipu_stack_gemm_f16", out, [da, db], sc)
    raw = out.download(np.uint16)
    assert np.all(raw[n:] == 0x7E00)
    if addend == "none":
        assert_product(oracle.f16_to_f32(raw[:n]).reshape(B, M, N), af, bf, K)
        # the same bits as each batch's rows of one 2-D product
        one = ctx.alloc(n * 2)
        ctx.launch("ipu_stack_gemm_f16", one, [da, db], [1, B * M, N, K, 0, 0, 0, 0])
        assert np.array_equal(one.download(np.uint16), raw[:n])
    else:
        count, strides = {"full": (n, [M * N, N]), "matrix": (M * N, [0, N]), "rows": (N, [0, 0])}[addend]
        d = ctx.upload(ipus.synth_f16(count, 71, 3, 0, 1.0))
        want, got = ctx.alloc(n * 2), ctx.alloc(n * 2)
        ctx.launch("ipu_stack_add_f16", want, [out, d], [n, n, count])
        ctx.launch("ipu_stack_gemm_f16_accumulate", got, [da, db, d], sc + strides)
        assert np.array_equal(got.download(np.uint16), want.download(np.uint16))


@pytest.mark.parametrize("M,N,K", [
    # 64 x 64 tiles: partial tiles, a partial last step, one step
    (1000, 1004, 1000), (520, 1160, 72), (1024, 1024, 32),
    # 32 x 32 tiles
    (8, 4, 4), (36, 68, 100), (32, 32, 64), (1, 4096, 260),
    # pitches that are no multiple of 4
    (1001, 1003, 999), (521, 1158, 65), (1, 1, 1), (33, 31, 127), (3, 4097, 130)])
@pytest.mark.parametrize("tl,tr", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_gemm_f32_tiles(ipus, ctx, M, N, K, tl, tr):
    """Every element within K + 2 fp32 roundings of the running magnitude."""
    a = ipus.synth_f32(M * K, 77, 1, 0, 1.0)
    b = ipus.synth_f32(K * N, 77, 2, 0, 1.0)
    pad = np.full(64 * max(M, N, K), np.nan, np.float32)  # read past an operand: NaN
    da, db = ctx.upload(np.concatenate([a, pad])), ctx.upload(np.concatenate([b, pad]))
    out = ctx.upload(np.full(M * N + 4, 7.0, np.float32))
    ctx.launch("ipu_stack_gemm_f32", out, [da, db], [1, M, N, K, tl, tr, 0, 0])
    raw = out.download(np.float32)
    assert np.all(raw[M * N:] == 7.0)
    af = a.astype(np.float64).reshape((K, M) if tl else (M, K))
    bf = b.astype(np.float64).reshape((N, K) if tr else (K, N))
    af, bf = af.T if tl else af, bf.T if tr else bf
    bound = np.abs(af) @ np.abs(bf) * (K + 2) * 2.0 ** -24 + 1e-30
    assert np.all(np.abs(raw[:M * N].reshape(M, N) - af @ bf) <= bound)
    for x in (da, db, out):
        x.free()


def test_gemm_f32_tiles_batched(ipus, ctx):
    B, M, N, K = 3, 100, 132, 200
    a, b = ipus.synth_f32(B * M * K, 78, 1, 0, 1.0), ipus.synth_f32(K * N, 78, 2, 0, 1.0)
    da, db, out = ctx.upload(a), ctx.upload(b), ctx.alloc(B * M * N * 4)
    ctx.launch("ipu_stack_gemm_f32", out, [da, db], [B, M, N, K, 0, 0, M * K, 0])
    got = out.download(np.float32).reshape(B, M, N)
    af, bf = a.astype(np.float64).reshape(B, M, K), b.astype(np.float64).reshape(K, N)
    bound = np.abs(af) @ np.abs(bf) * (K + 2) * 2.0 ** -24
    assert np.all(np.abs(got - af @ bf) <= bound)
    for x in (da, db, out):
        x.free()


@pytest.mark.parametrize("M,N,K", [
    (3074, 3082, 1030),   # tile 256: last step 6 k, a chunk past every edge
    (3080, 3074, 1088),   # tile 256: whole K steps, odd chunks along N only
    (1802, 2058, 590),    # tile 128
    (522, 1162, 1154),    # tile 64
    (42, 74, 266), (2, 2, 2), (34, 4098, 62),   # tile 32: K below one step
    (258, 262, 130)])
@pytest.mark.parametrize("tl,tr", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_gemm_f16_dword_aligned_pitches(ipus, oracle, ctx, M, N, K, tl, tr):
    """Row pitches that are even but no multiple of 8, at 4-byte-aligned
    addresses."""
    check_unaligned(ipus, oracle, ctx, M, N, K, tl, tr, 2)


@pytest.mark.parametrize("M,N,K", [
    (1801, 2057, 585),    # tile 128
    (521, 1161, 1155),    # tile 64
    (41, 73, 265), (1, 1, 1), (33, 4097, 61), (257, 263, 129), (64, 64, 192)])  # tile 32
@pytest.mark.parametrize("tl,tr", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_gemm_f16_odd_pitches(ipus, oracle, ctx, M, N, K, tl, tr):
    """Odd row pitches, or any at 2-byte-aligned addresses."""
    check_unaligned(ipus, oracle, ctx, M, N, K, tl, tr, 1)


@pytest.mark.parametrize("M,N,K", [(16, 5001, 768), (1030, 777, 1090), (130, 67, 64)])
def test_gemm_f16_odd_output_rows(ipus, oracle, ctx, M, N, K):
    """Dword-aligned operands (the right one transposed), C with odd rows."""
    check_unaligned(ipus, oracle, ctx, M, N, K, 0, 1, 2)


def check_unaligned(ipus, oracle, ctx, M, N, K, tl, tr, shift_elements):
    """Operands and output `shift_elements` into their allocations; NaN after both operands, so that an element read from past
    them (rather than masked or cleared) shows.  Rows at both ends and
    sampled between are checked, and nothing is stored past C."""
    a = ipus.synth_f16(M * K, 79, 1, 0, 1.0)
    b = ipus.synth_f16(K * N, 79, 2, 0, 1.0)
    at = shift_elements
    shift = np.zeros(at, np.uint16)
    pad = np.full(64 * max(M, N, K), 0x7E00, np.uint16)
    da, db = (ctx.upload(np.concatenate([shift, x, pad])) for x in (a, b))
    out = ctx.upload(np.full(M * N + 16, 0x7E00, np.uint16))
    sc = [1, M, N, K, tl, tr, 0, 0]
    ctx.launch("ipu_stack_gemm_f16", out.ptr + 2 * at, [da.ptr + 2 * at, db.ptr + 2 * at], sc)
    raw = out.download(np.uint16)
    assert np.all(raw[:at] == 0x7E00) and np.all(raw[at + M * N:] == 0x7E00)
    rows = np.unique(np.concatenate([np.arange(min(M, 20)), np.arange(max(0, M - 20), M),
                                     np.random.default_rng(3).integers(0, M, 40)]))
    af = oracle.f16_to_f32(a).astype(np.float64).reshape((K, M) if tl else (M, K))
    bf = oracle.f16_to_f32(b).astype(np.float64).reshape((N, K) if tr else (K, N))
    af, bf = (af.T if tl else af)[rows], bf.T if tr else bf
    got = oracle.f16_to_f32(raw[at:at + M * N]).reshape(M, N)
    assert_product(got[rows], af, bf, K)
    # The add epilogue, its addend (any alignment) read by element
    d = ctx.upload(np.concatenate([np.zeros(1, np.uint16), ipus.synth_f16(M * N, 79, 3, 0, 1.0)]))
    want = ctx.alloc(M * N * 2)
    fused = ctx.alloc(M * N * 2)
    ctx.launch("ipu_stack_add_f16", want, [out.ptr + 2 * at, d.ptr + 2], [M * N, M * N, M * N])
    ctx.launch("ipu_stack_gemm_f16_accumulate", fused, [da.ptr + 2 * at, db.ptr + 2 * at, d.ptr + 2],
               sc + [0, N])
    assert np.array_equal(fused.download(np.uint16), want.download(np.uint16))
    for x in (da, db, d, out, want, fused):
        x.free()
