"""A caller records the context's stream into a graph of its own, which it may
replay on any stream beside the context's launches: nothing recorded may use
the context's workspace, whose counters and partial sums those launches use."""
from __future__ import annotations

import ctypes

import numpy as np
import pytest

from test_gpu_attention_plans import attention64
from test_gpu_gemm_tiles import assert_product, operands

pytestmark = pytest.mark.gpu


class Recording:
    """Records the context's stream (through the HIP runtime that the library
    itself is linked to) and replays the graph on a stream of its own."""

    def __init__(self, ipus, ctx):
        self.hip = ipus.load_library()
        self.ctx, self.graph, self.exec = ctx, ctypes.c_void_p(), ctypes.c_void_p()
        self.stream = ctypes.c_void_p()

    def call(self, name, *args):
        assert getattr(self.hip, name)(*args) == 0, name

    def __enter__(self):
        self.call("hipStreamBeginCapture", ctypes.c_void_p(self.ctx.stream()), 1)  # thread-local
        return self

    def __exit__(self, *exc):
        self.call("hipStreamEndCapture", ctypes.c_void_p(self.ctx.stream()), ctypes.byref(self.graph))
        self.call("hipGraphInstantiate", ctypes.byref(self.exec), self.graph, None, None,
                  ctypes.c_size_t(0))
        self.call("hipStreamCreate", ctypes.byref(self.stream))

    def replay(self):
        self.call("hipGraphLaunch", self.exec, self.stream)

    def sync(self):
        self.call("hipStreamSynchronize", self.stream)

    def close(self):
        self.call("hipGraphExecDestroy", self.exec)
        self.call("hipGraphDestroy", self.graph)
        self.call("hipStreamDestroy", self.stream)


def test_recorded_launches_run_beside_the_context(ipus, oracle, ctx):
    """Launches that split their reduction when the context runs them."""
    M, N, K = 8, 1024, 4096
    a, b, af, bf = operands(ipus, oracle, M, N, K, 0, 0, 1, True)
    streams, rows, keys, d = 4, 1, 2048, 64
    qkv = [ipus.synth_f16(streams * n * d, 75, i, ipus.NORMAL, 1.0)
           for i, n in ((1, rows), (2, keys), (3, keys))]
    ins, att = [ctx.upload(a), ctx.upload(b)], [ctx.upload(x) for x in qkv]
    outs = [(ctx.alloc(M * N * 2), ctx.alloc(streams * rows * d * 4)) for _ in range(2)]

    def launch(to):
        ctx.launch("ipu_stack_gemm_f16", to[0], ins, [1, M, N, K, 0, 0, 0, 0])
        ctx.launch("ipu_stack_flash_attention_online_f16", to[1], att,
                   [streams, rows, keys, d, d, 0, 0, 0])

    def check(to):
        assert_product(oracle.f16_to_f32(to[0].download(np.uint16)).reshape(1, M, N), af, bf, K)
        got = to[1].download(np.float32).reshape(streams, rows, d)
        q, k, v = (oracle.f16_to_f32(x).astype(np.float64).reshape(streams, -1, d) for x in qkv)
        for s in range(streams):
            want, bound = attention64(q[s], k[s], v[s], 0)
            assert np.all(np.abs(got[s] - want) <= bound), s

    recording = Recording(ipus, ctx)
    with recording:
        launch(outs[0])
    for _ in range(4):
        for buf in outs[0] + outs[1]:
            ctx.memset(buf, 0xFF)
        ctx.sync()
        for _ in range(8):
            recording.replay()
            launch(outs[1])
        recording.sync()
        ctx.sync()
        check(outs[0])
        check(outs[1])
    recording.close()
    for buf in ins + att + [x for o in outs for x in o]:
        buf.free()


def test_recorded_run_of_a_captured_session(ipus, ctx):
    """ipus_session_run of a captured session, recorded by a caller, records the
    session's steps without the workspace: the bits of the unsplit product."""
    M, N, K = 8, 256, 4096
    x, w = ipus.synth_f32(M * K, 76, 1, 0, 1.0), ipus.synth_f32(K * N, 76, 2, 0, 1.0)
    g = ipus.ComputeGraph()
    g.set_outputs([g.gemm(g.host_input("x", [M, K]), g.parameter("w", [K, N]))])
    package = ipus.build_package(g, ipus.PackageConfig(compute_precision="f32"))
    assert [s[0] for s in package.steps] == ["ipu_stack_gemm_f32"]
    session = package.session(ctx)
    session.write("x", x.reshape(M, K))
    session.write("w", w.reshape(K, N))
    session.run_sync()
    split = session.read(package.outputs[0].name).reshape(-1).copy()
    ins, plain = [ctx.upload(x), ctx.upload(w)], ctx.alloc(M * N * 4)
    direct, run = Recording(ipus, ctx), Recording(ipus, ctx)
    with direct:
        ctx.launch("ipu_stack_gemm_f32", plain, ins, [1, M, N, K, 0, 0, 0, 0])
    session.capture()
    with run:
        session.run()
    direct.replay()
    direct.sync()
    unsplit = plain.download(np.float32)
    assert not np.array_equal(unsplit, split)  # the two sums can be told apart
    for _ in range(3):
        session.run_sync()
        assert np.array_equal(session.read(package.outputs[0].name).reshape(-1), split)
        run.replay()
        run.sync()
        assert np.array_equal(session.read(package.outputs[0].name).reshape(-1), unsplit)
    direct.close()
    run.close()
    session.close()
    for buf in ins + [plain]:
        buf.free()
