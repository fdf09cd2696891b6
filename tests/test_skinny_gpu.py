"""The skinny GEMM (at most 128 rows): row blocks, split K, short K, grouped
launches, against the oracle's linear."""
import ctypes as C

import numpy as np
import pytest

import h3hip
import oracle
from conftest import assert_close, rand_bf16

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,k,n,bias", [
    (65, 64, 128, True), (96, 128, 132, False),   # 3 row blocks, 1-2 K steps
    (97, 320, 100, True), (128, 448, 4, True),    # 4 row blocks, K steps 5, 7
    (129, 512, 260, True),                        # one past: the tile kernel
    (128, 64, 32772, True), (97, 512, 33000, False),  # tiles, short K and wide
    (1, 64, 4, True), (1, 192, 4, False),         # a partial turn of the ring
    (33, 128, 300, True), (128, 192, 260, False),
    (40, 384, 260, True), (64, 1088, 65540, False),  # 6 steps; 17, one ahead
    (1, 1024, 4, True), (7, 2112, 36, False),     # split K, a short last piece
    (33, 4096, 300, True), (120, 5120, 1284, True),
    (128, 14336, 128, False),                     # 28 pieces of one tile
    (64, 512, 65540, True),                       # rounds of workgroups
])
def test_linear_skinny(gpu, m, k, n, bias):
    rng = np.random.default_rng(m + k + n)
    x, w = rand_bf16(rng, m * k), rand_bf16(rng, n * k, 0.05)
    b = rand_bf16(rng, n, 0.1) if bias else None
    out = gpu.new_bf16(m * n)
    args = (out, gpu.bf16(x), gpu.bf16(w), gpu.bf16(b) if bias else None, m,
            k, n)
    gpu.run("h3_gpu_linear_bf16", *args)
    got = gpu.read_bf16(out)
    assert_close(got, oracle.linear(x, w, b, m, k, n), what="skinny")
    gpu.run("h3_hip_linear_bf16_noalloc", *args)
    assert np.array_equal(gpu.read_bf16(out), got)


@pytest.mark.parametrize("m,k,n", [
    (1, 64, 4), (65, 512, 132), (97, 1088, 260),
    (8, 5376, 512), (128, 14336, 128),  # K in pieces
    (40, 128, 16384), (40, 128, 16388),  # the last size in one launch, and two
])
def test_linear_pair_skinny(gpu, m, k, n):
    """Each of a pair is what a linear gives (its sums in other pieces where K
    is cut)."""
    rng = np.random.default_rng(m + k + n)
    x = rand_bf16(rng, m * k)
    ws = [rand_bf16(rng, n * k, 0.05) for _ in range(2)]
    bs = [rand_bf16(rng, n, 0.1), None]
    outs = [gpu.new_bf16(m * n) for _ in range(2)]
    gpu.run("h3_hip_linear_pair_bf16", *outs, gpu.bf16(x), gpu.bf16(ws[0]),
            gpu.bf16(bs[0]), gpu.bf16(ws[1]), None, m, k, n)
    for out, w, b in zip(outs, ws, bs):
        assert_close(gpu.read_bf16(out), oracle.linear(x, w, b, m, k, n),
                     what="skinny pair")


@pytest.mark.parametrize("m,k,n,count,first", [
    (1, 64, 64, 3, 0), (40, 320, 132, 4, 1), (64, 512, 640, 5, 2),
    (65, 128, 128, 2, 0), (120, 512, 260, 3, 1),
])
def test_linear_group_skinny(gpu, m, k, n, count, first):
    """Grouped launches of few rows: each problem of the range against the
    oracle, the others untouched."""
    rng = np.random.default_rng(m + n)
    total = first + count
    x = rand_bf16(rng, m * k)
    ws = [rand_bf16(rng, n * k, 0.05) for _ in range(total)]
    bs = [rand_bf16(rng, n, 0.1) if p % 2 else None for p in range(total)]
    outs = [gpu.bf16(np.full(m * n, 5, np.uint16)) for _ in range(total)]
    arr = C.c_void_p * total
    table = gpu.L.h3_hip_linear_group_table(
        gpu.h, arr(*outs), arr(*[gpu.bf16(w) for w in ws]),
        arr(*[gpu.bf16(b) if b is not None else None for b in bs]), total, m,
        k, n)
    assert table, gpu.error()
    try:
        gpu.run("h3_hip_linear_group_bf16", table, first, count, gpu.bf16(x),
                m, k, n)
        for p in range(total):
            got = gpu.read_bf16(outs[p])
            if p < first:
                assert (got == 5).all()
            else:
                assert_close(got, oracle.linear(x, ws[p], bs[p], m, k, n),
                             what=f"group[{p}]")
    finally:
        gpu.L.h3_gpu_tensor_free(table)


@pytest.mark.parametrize("m", [8, 64, 128])
def test_noalloc_calls_of_two_contexts_overlap(m):
    """Two contexts enqueue allocation-free calls in turn and submit only
    then: each result is the one that the context gives alone."""
    k, n, calls = 14336, 1280, 8
    rng = np.random.default_rng(m)
    w = rand_bf16(rng, n * k, 0.05)
    xs = [rand_bf16(rng, m * k) for _ in range(2)]
    gpus = [h3hip.Gpu() for _ in xs]
    try:
        tw = [g.bf16(w) for g in gpus]
        tx = [g.bf16(x) for g, x in zip(gpus, xs)]
        outs = [[g.new_bf16(m * n) for _ in range(calls)] for g in gpus]
        alone = []
        for g, x, t, o in zip(gpus, tx, tw, outs):
            g.run("h3_gpu_linear_bf16", o[0], x, t, None, m, k, n)
            alone.append(g.read_bf16(o[0]))
            assert_close(alone[-1], oracle.linear(xs[len(alone) - 1], w, None,
                                                  m, k, n), what="alone")
        for g in gpus:
            g.begin()
        for c in range(calls):
            for g, x, t, o in zip(gpus, tx, tw, outs):
                g.check(g.L.h3_hip_linear_bf16_noalloc(
                    g.h, o[c], x, t, None, m, k, n), "noalloc")
        for g in gpus:
            g.submit()
        for g, o, want in zip(gpus, outs, alone):
            for t in o:
                assert np.array_equal(g.read_bf16(t), want)
    finally:
        for g in gpus:
            g.close()


def test_skinny_weight_over_two_gib(gpu):
    """The first and the last columns of a weight past 2 GiB, each block
    copied out and multiplied by the oracle."""
    m, k, n, block = 40, 2688, 420004, 68
    rng = np.random.default_rng(12)
    x = rand_bf16(rng, m * k)
    w, out, part = (gpu.new_bf16(s) for s in (n * k, m * n, block * k))
    gpu.run("h3_gpu_fill_normal_bf16", w, 0, n * k, 3, C.c_float(0.0),
            C.c_float(0.05))
    gpu.run("h3_gpu_linear_bf16", out, gpu.bf16(x), w, None, m, k, n)
    got = gpu.read_bf16(out).reshape(m, n)
    for first in (0, (1 << 30) // k - 30, n - block):
        gpu.run("h3_gpu_copy_bf16", part, 0, w, first * k, block * k)
        want = oracle.linear(x, gpu.read_bf16(part), None, m, k, block)
        assert_close(got[:, first:first + block].ravel(), want,
                     what=f"columns from {first}")
    for t in (w, out, part):
        gpu.free(t)
