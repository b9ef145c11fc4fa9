"""Constant right-hand sides laid out as bf16 planes: which GEMMs get them and where they lie."""

from __future__ import annotations

import re

import numpy as np

from ml_graph_compiler import builders
from ml_graph_compiler.codegen import build as native
from ml_graph_compiler.codegen.hip import generate_hip
from ml_graph_compiler.passes import optimize
from ml_graph_compiler.schedule import schedule


def _generate(graph, planes=True):
    optimize(graph, "O3")
    schedule(graph)
    return generate_hip(graph, gemm_workspace=native.gemm_workspace_floats,
                        gemm_ln_workspace=native.gemm_layer_norm_workspace_floats,
                        gemm_planes=native.gemm_planes_bytes if planes else None)


def test_large_gemms_read_planes_past_the_plan(hip_cache):
    make = lambda: builders.transformer(batch=16, seq=128, d_model=256, heads=4, layers=2, vocab=4096, gelu="erf", causal=False)  # noqa: E731
    plain, gen = _generate(make(), planes=False), _generate(make())
    assert "planes" not in plain.source and gen.plan.arena_bytes == plain.plan.arena_bytes
    assert gen.weights.digest() == plain.weights.digest()  # the blob stays as it is
    rows = [tuple(map(int, r)) for r in re.findall(r"\{(\d+)UL, (\d+)UL, (\d+), (\d+)\}", gen.source)]
    assert rows and len({r[0] for r in rows}) == len(rows)
    used = {int(o) for o in re.findall(r"mgc_hip_gemm_planes(?:_layer_norm)?\(x, &g, \(A \+ (\d+)\)", gen.source)}
    assert used == {at for _, at, _, _ in rows}
    end = plain.arena_bytes  # the plan and the scratch area
    for off, at, n, k in sorted(rows, key=lambda r: r[1]):
        assert at % 256 == 0 and at >= end and off + 4 * n * k <= gen.weights.nbytes
        end = at + native.gemm_planes_bytes(2048, n, k)
        assert end - at >= n * k * 6
    assert end <= gen.arena_bytes
    native.build_model_library(gen.source, cache_dir=hip_cache, name="planes")


def test_small_gemms_keep_the_fp32_kernels():
    assert "planes" not in _generate(builders.mlp()).source
    for m, n, k in ((1, 768, 768), (128, 768, 768), (32, 1000, 2048), (2048, 768, 32), (0, 1, 1)):
        assert native.gemm_planes_bytes(m, n, k) == 0
    assert native.gemm_planes_bytes(2048, 3072, 768) >= 3072 * 768 * 6


def test_planes_only_for_the_call_that_reads_them():
    """1024 x 768 x 768 reads planes with a LayerNorm tail (a K split of two) but not alone."""
    def graph(norm):
        b = builders.GraphBuilder("dense", 1)
        x = b.op1("MatMul", [b.input("x", "float32", (1024, 768)), b.const(np.ones((768, 768), np.float32))])
        if norm:
            x = b.op1("LayerNormalization", [x, b.const(np.ones(768, np.float32)), b.const(np.zeros(768, np.float32))], axis=-1)
        return b.finish([("out", x)])

    assert native.gemm_planes_bytes(1024, 768, 768) > 0
    plain, tail = _generate(graph(False)), _generate(graph(True))
    assert "planes" not in plain.source and plain.arena_bytes == _generate(graph(False), planes=False).arena_bytes
    assert "mgc_hip_gemm_planes_layer_norm" in tail.source


def test_tiles_of_few_rows_read_planes_where_weights_stay_cached():
    """32-row tiles read planes in models whose weights stay near: alone (784 x 512 x 384), up to 8 MB
    (392 x 768 x 768), in an encoder of 113 MB of weights (128 x 2304 x 768) but not in one of 198 MB.
    128-row tiles and the forms that replace the element-by-element kernel read them in every model."""
    mb = 1000000
    wants = lambda m, n, k, w: native.gemm_planes_bytes(m, n, k, False, w) > 0  # noqa: E731
    assert [wants(784, 512, 384, w * mb) for w in (1, 2, 3, 102)] == [True, True, False, False]
    assert [wants(392, 768, 768, w * mb) for w in (2, 8, 9, 102)] == [True, True, False, False]
    assert [wants(128, 2304, 768, w * mb) for w in (7, 113, 160, 170, 340)] == [True, True, True, False, False]
    assert all(wants(m, n, k, 500 * mb) for m, n, k in ((2048, 3072, 768), (1, 50257, 768), (1003, 1021, 515), (7, 2999, 77)))
    seen = set()

    def record(m, n, k, layer_norm, weight_bytes):
        seen.add(weight_bytes)
        return 0

    graph = builders.resnet50(1)
    optimize(graph, "O3")
    schedule(graph)
    generate_hip(graph, gemm_workspace=native.gemm_workspace_floats, gemm_planes=record)
    assert len(seen) == 1 and 100 * mb < seen.pop() < 103 * mb  # 25.5 million weights
