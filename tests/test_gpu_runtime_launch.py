"""How the runtime enqueues a forward: short ones kernel by kernel, long ones as a graph from the
second run on the same buffers; every way gives the same bits, and a bad Gather index is reported
once whichever way it ran."""

from __future__ import annotations

import numpy as np
import pytest

from capi import Hip
from ml_graph_compiler import builders
from ml_graph_compiler.codegen import compile_graph
from ml_graph_compiler.errors import GraphError
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
