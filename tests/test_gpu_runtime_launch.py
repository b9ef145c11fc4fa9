"""How the runtime enqueues a forward: short ones kernel by kernel, long ones as a graph from the
second run on the same buffers; every way gives the same bits, and a bad Gather index is reported
once whichever way it ran."""

from __future__ import annotations

import numpy as np
import pytest

from capi import Hip
from ml_graph_compiler import builders
from ml_graph_compiler.codegen import compile_graph, runtime_lib
from ml_graph_compiler.codegen.hip import generate_hip
from ml_graph_compiler.errors import CodegenError, GraphError
from ml_graph_compiler.passes import optimize
from ml_graph_compiler.schedule import schedule

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("layers", [1, 4])  # about 9 and 27 launches: both sides of the runtime's limit
def test_every_way_gives_the_same(layers, hip_cache):
    graph = builders.transformer(layers=layers)
    feeds = builders.random_feeds(graph, 3)
    other = builders.random_feeds(graph, 4)
    optimize(graph, "O3")
    schedule(graph)
    model = compile_graph(graph, cache_dir=hip_cache, name=f"ways{layers}")
    hip = Hip()
    try:
        first = model.run(feeds)["logits"]
        for _ in range(3):  # the staged graph's capture and replays
            np.testing.assert_array_equal(model.run(feeds)["logits"], first)
        second = model.run(other)["logits"]
        assert not np.array_equal(first, second)
        ids = [hip.upload(f["input_ids"]) for f in (feeds, other)]
        outs = [hip.empty(first.nbytes) for _ in range(2)]
        # two sets of buffers in turn, then each several times in a row, then inputs changed in place
        for i in (0, 1, 0, 1, 1, 1, 0, 0, 0):
            model.run_device([ids[i]], [outs[i]])
            np.testing.assert_array_equal(hip.download(outs[i], first.shape), (first, second)[i])
        hip.put(ids[0], other["input_ids"])
        model.run_device([ids[0]], [outs[0]])
        np.testing.assert_array_equal(hip.download(outs[0], first.shape), second)
        bad = other["input_ids"].copy()
        bad[0, 0] = 128  # the vocabulary
        hip.put(ids[0], bad)
        with pytest.raises(GraphError, match="out-of-range Gather"):
            model.run_device([ids[0]], [outs[0]])
        hip.put(ids[0], feeds["input_ids"])
        model.run_device([ids[0]], [outs[0]])
        np.testing.assert_array_equal(hip.download(outs[0], first.shape), first)
        model.upload(feeds)
        model.launch(3)
        np.testing.assert_array_equal(model.download()["logits"], first)
    finally:
        model.release()
        hip.free()


def test_an_error_pending_on_the_thread_is_the_callers(hip_cache):
    """Launching kernel by kernel neither reports nor clears an error that the calling thread left from
    its other work (a failed hipSetDevice)."""
    graph = builders.mlp()
    feeds = builders.random_feeds(graph, 3)
    optimize(graph, "O3")
    schedule(graph)
    model = compile_graph(graph, cache_dir=hip_cache, name="pending")
    hip = Hip()
    try:
        first = model.run(feeds)
        for _ in range(3):
            code = hip.lib.hipSetDevice(1 << 20)
            assert code != 0 and hip.lib.hipPeekAtLastError() == code
            again = model.run(feeds)
            for name, value in first.items():
                np.testing.assert_array_equal(again[name], value)
            assert hip.lib.hipGetLastError() == code
    finally:
        model.release()


def test_nothing_is_in_flight_after_a_failed_forward(hip_cache, monkeypatch):
    """A forward whose last launch is refused returns once the ones before it are done with the
    caller's buffers."""
    n = 4096
    b = builders.GraphBuilder("half", 1)
    x = b.input("x", "float32", (n, n))
    y = b.op1("MatMul", [x, x])
    graph = b.finish([("out", b.op1("MatMul", [y, x]))])
    optimize(graph, "O3")
    schedule(graph)

    def refused(*args, **kwargs):  # the same forward, then a GEMM of an unknown kernel family
        gen = generate_hip(*args, **kwargs)
        end = gen.source.rindex("mgc_hip_gemm(x, &g);")
        call = "mgc_hip_gemm(x, &g); g.kernel = 99; mgc_hip_gemm(x, &g);"
        gen.source = gen.source[:end] + call + gen.source[end + len("mgc_hip_gemm(x, &g);"):]
        return gen

    model = compile_graph(graph, cache_dir=hip_cache, name="whole")
    monkeypatch.setattr(runtime_lib, "generate_hip", refused)
    failing = compile_graph(graph, cache_dir=hip_cache, name="half")
    hip = Hip()
    try:
        pin = hip.upload(np.random.default_rng(1).standard_normal((n, n), dtype=np.float32))
        want, out = hip.empty(4 * n * n), hip.empty(4 * n * n)
        model.run_device([pin], [want])
        for _ in range(3):
            with pytest.raises(CodegenError):
                failing.run_device([pin], [out])
            got = np.empty((n,), np.float32)  # the last row, without waiting for other streams
            hip.check(hip.lib.hipMemcpy(got.ctypes.data, out + 4 * n * (n - 1), got.nbytes, 2), "hipMemcpy D2H")
            np.testing.assert_array_equal(got, hip.download(want, (n, n))[-1])
            hip.put(out, np.full((n, n), np.nan, np.float32))
    finally:
        model.release()
        failing.release()
        hip.free()
