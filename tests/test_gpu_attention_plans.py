"""The fast attention kernel's launch plans (query tiles per wave, query blocks
per workgroup) against float64, with partial query and key blocks.  The launch
picks the plan from the shape; each shape names the plan it was chosen for."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def attention64(q, k, v, causal):
    """Exact output, and a bound on the kernel's error per element."""
    d, keys = q.shape[1], k.shape[0]
    scale = 1.0 / np.sqrt(d)
    s = (q @ k.T) * scale
    # fp32 sums of d exact products, the scale and exp2 in fp32 (about 2^-22
    # of the exponent each)
    ds = (np.abs(q) @ np.abs(k).T) * scale * (d + 4) * 2.0 ** -24 + np.abs(s) * 2.0 ** -21
    if causal:
        allowed = np.arange(keys)[None, :] <= np.arange(len(q))[:, None]
        s, ds = np.where(allowed, s, -np.inf), np.where(allowed, ds, 0.0)
    p = np.exp(s - s.max(axis=1, keepdims=True))
    p /= p.sum(axis=1, keepdims=True)
    delta = 2.0 * ds.max(axis=1, keepdims=True)
    # Probabilities rounded to fp16 (2^-11), their sum with two fp16
    # additions (2^-10), fp32 accumulation.
    bound = (2.0 ** -11 + 2.0 ** -10 + delta + keys * 2.0 ** -23) * (p @ np.abs(v)) + 2.0 ** -20
    return p @ v, bound


@pytest.mark.parametrize("streams,heads,rows,keys,d,causal", [
    (64, 16, 400, 330, 72, 0),    # two tiles, single blocks
    (64, 1, 1000, 70, 32, 0),     # two tiles, pairs (one block left over: 8 blocks of 128)
    (3, 1, 129, 65, 128, 0),      # one tile, single blocks
    (2, 2, 1, 200, 64, 0),        # one query row
    (512, 8, 65, 64, 96, 0),      # one tile, pairs
    (64, 1, 1000, 1000, 64, 1),   # causal, two tiles, pairs
    (48, 12, 700, 700, 64, 1),    # causal, one tile, pairs
    (4, 1, 300, 257, 128, 1),     # causal, one tile, single blocks, fewer keys than rows
    (2, 1, 190, 190, 192, 1),     # 256-wide tiles, single blocks
])
@pytest.mark.parametrize("f16", [0, 1])
def test_attention_plans(ipus, oracle, ctx, streams, heads, rows, keys, d, causal, f16):
    q, k, v = (ipus.synth_f16(streams * n * d, 73, i, ipus.NORMAL, 1.0)
               for i, n in ((1, rows), (2, keys), (3, keys)))
    bufs = [ctx.upload(x) for x in (q, k, v)]
    count = streams * rows * d
    out = ctx.upload(np.full(count * (1 if f16 else 2) + 8, 0x7E00, np.uint16))
    ctx.launch("ipu_stack_flash_attention_heads_f16", out, bufs,
               [streams, rows, keys, d, d, 0, causal, f16, heads, heads, heads])
    raw = out.download(np.uint16)
    got = (oracle.f16_to_f32(raw[:count]) if f16 else raw[:2 * count].view(np.float32))
    got = got.reshape(streams, rows, d)
    assert np.all(raw[-8:] == 0x7E00)  # nothing stored past the output

    def stream(x, n, s):
        x = oracle.f16_to_f32(x).astype(np.float64).reshape(streams // heads, n, heads, d)
        return x[s // heads, :, s % heads, :]

    for s in sorted({0, streams // 2, streams - 1}):
        want, bound = attention64(stream(q, rows, s), stream(k, keys, s), stream(v, keys, s), causal)
        if f16:
            bound = bound + np.abs(want) * 2.0 ** -11 + 2.0 ** -24
        assert np.all(np.abs(got[s] - want) <= bound), s
    for x in bufs + [out]:
        x.free()


SPLIT_SHAPES = [  # few queries, many keys: the keys are split over workgroups
                (3, 1, 1, 1025, 128),     # a last split with a partial block
                (16, 16, 5, 2048, 72), (2, 1, 64, 4000, 64),
                (5, 1, 65, 3000, 96),     # a second query block of one row
                (2, 2, 16, 1500, 256),    # 32-key blocks
                (128, 16, 1, 1600, 32)]


@pytest.mark.parametrize("streams,heads,rows,keys,d", SPLIT_SHAPES)
@pytest.mark.parametrize("f16", [0, 1])
def test_attention_key_splits(ipus, oracle, ctx, streams, heads, rows, keys, d, f16):
    """Split launches against float64, and three in a row alike (the merge
    leaves its counters as it found them)."""
    q, k, v = (ipus.synth_f16(streams * n * d, 75, i, ipus.NORMAL, 1.0)
               for i, n in ((1, rows), (2, keys), (3, keys)))
    bufs = [ctx.upload(x) for x in (q, k, v)]
    count = streams * rows * d
    out = ctx.alloc(count * (2 if f16 else 4))
    results = []
    for _ in range(3):
        ctx.memset(out, 0xFF)
        ctx.launch("ipu_stack_flash_attention_heads_f16", out, bufs,
                   [streams, rows, keys, d, d, 0, 0, f16, heads, heads, heads])
        results.append(out.download(np.uint16))
    assert np.array_equal(results[0], results[1]) and np.array_equal(results[0], results[2])
    got = (oracle.f16_to_f32(results[0]) if f16 else results[0].view(np.float32))
    got = got.reshape(streams, rows, d)

    def stream(x, n, s):
        x = oracle.f16_to_f32(x).astype(np.float64).reshape(streams // heads, n, heads, d)
        return x[s // heads, :, s % heads, :]

    for s in sorted({0, streams // 2, streams - 1}):
        want, bound = attention64(stream(q, rows, s), stream(k, keys, s), stream(v, keys, s), 0)
        if f16:
            bound = bound + np.abs(want) * 2.0 ** -11 + 2.0 ** -24
        assert np.all(np.abs(got[s] - want) <= bound), s
    for x in bufs + [out]:
        x.free()


@pytest.mark.parametrize("dead", [64, 512, 1000])
def test_attention_key_splits_with_minus_infinity_scores(ipus, oracle, ctx, dead):
    """Keys whose scores are all -inf carry no weight, also where they fill a
    split or its first blocks; a NaN key makes every output NaN."""
    streams, rows, keys, d = 2, 3, 2048, 128
    q, k, v = (ipus.synth_f16(streams * n * d, 76, i, ipus.NORMAL, 1.0).reshape(streams, n, d)
               for i, n in ((1, rows), (2, keys), (3, keys)))
    q[:, :, 0] = 0x3C00          # 1
    k[:, :dead, 0] = 0xFC00      # -inf
    args = [streams, rows, keys, d, d, 0, 0, 0]
    bufs = [ctx.upload(x) for x in (q, k, v)]
    out = ctx.alloc(streams * rows * d * 4)
    ctx.launch("ipu_stack_flash_attention_online_f16", out, bufs, args)
    got = out.download(np.float32).reshape(streams, rows, d)
    qf, kf, vf = (oracle.f16_to_f32(x).astype(np.float64).reshape(x.shape) for x in (q, k, v))
    for s in range(streams):
        want, bound = attention64(qf[s], kf[s, dead:], vf[s, dead:], 0)
        assert np.all(np.abs(got[s] - want) <= bound)
    k[0, keys - 1, 5] = 0x7E00
    ctx.write(bufs[1], k)
    ctx.launch("ipu_stack_flash_attention_online_f16", out, bufs, args)
    got = out.download(np.float32).reshape(streams, rows, d)
    assert np.all(np.isnan(got[0])) and not np.any(np.isnan(got[1]))
    for x in bufs + [out]:
        x.free()


def test_attention_key_splits_in_a_captured_session(ipus, ctx):
    """A session's captured graph replays a split launch with the eager
    result, with other launches on the stream in between."""
    g = ipus.ComputeGraph()
    q, k, v = (g.host_input(n, [4, r, 64]) for n, r in (("q", 2), ("k", 3000), ("v", 3000)))
    g.set_outputs([g.flash_attention(q, k, v)])
    pkg = ipus.build_package(g)
    eager, replay = pkg.session(ctx), pkg.session(ctx)
    replay.capture()
    for seed in range(4):
        for i, (name, r) in enumerate((("q", 2), ("k", 3000), ("v", 3000))):
            x = ipus.synth_f16(4 * r * 64, 80 + seed, i, ipus.NORMAL, 1.0).reshape(4, r, 64)
            eager.write(name, x)
            replay.write(name, x)
        replay.run()
        eager.run()
        replay.run()
        assert np.array_equal(replay.read("output.0"), eager.read("output.0"))
    eager.close()
    replay.close()
