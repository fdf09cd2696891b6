"""The skinny GEMM (at most 128 rows): row blocks, split K, short K, grouped
launches, against the oracle's linear."""
import ctypes as C

import numpy as np
import pytest

import oracle
from conftest import assert_close, rand_bf16

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,k,n,bias", [
    (65, 64, 128, True), (96, 128, 132, False),   # 3 row blocks, 1-2 K steps
    (97, 320, 100, True), (128, 448, 4, True),    # 4 row blocks, K steps 5, 7
    (129, 512, 260, True),                        # one past: the tile kernel
    (1, 64, 4, True), (1, 192, 4, False),         # dead steps pass both ends
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
