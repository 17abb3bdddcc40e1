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
