"""The MFMA GEMM's lower tiles (128 to 224 rows), with every epilogue: sizes at
which the tile-height estimate takes each of them, in plain rounds, with a
split tail and with every tile split."""
import numpy as np
import pytest

import oracle
from conftest import assert_close, rand_bf16

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,k,n", [
    (262, 512, 33220),   # 128 rows
    (129, 512, 33220),   # 160
    (129, 448, 196),     # 192
    (199, 448, 6084),    # 224
    (129, 2112, 1988),   # 160, every tile split
    (129, 2112, 1220),   # 192, every tile split
    (1292, 640, 22980),  # 224, a split tail
])
@pytest.mark.parametrize("gelu", [False, True])
def test_linear_low_tiles(gpu, m, k, n, gelu):
    rng = np.random.default_rng(m + k + n)
    x, w = rand_bf16(rng, m * k), rand_bf16(rng, n * k, 0.05)
    b = rand_bf16(rng, n, 0.1)
    out = gpu.new_bf16(m * n)
    gpu.run("h3_gpu_linear_gelu_bf16" if gelu else "h3_gpu_linear_bf16", out,
            gpu.bf16(x), gpu.bf16(w), gpu.bf16(b), m, k, n)
    want = oracle.linear(x, w, b, m, k, n)
    if gelu:
        want = oracle.gelu(want)
    assert_close(gpu.read_bf16(out), want, what="low tiles", chained=gelu)


@pytest.mark.parametrize("m,k,n", [
    (262, 512, 16576), (129, 512, 16576), (129, 448, 64), (199, 448, 3008),
    (129, 2112, 960), (129, 2112, 576), (1292, 640, 11456),
])
def test_mlp_low_tiles(gpu, m, k, n):
    """The same heights for the SwiGLU projection (128 columns a tile)."""
    rng = np.random.default_rng(m + k + n)
    x = rand_bf16(rng, m * k)
    w1, w2 = rand_bf16(rng, 2 * n * k, 0.05), rand_bf16(rng, k * n, 0.05)
    out = gpu.new_bf16(m * k)
    gpu.run("h3_gpu_mlp_bf16", out, gpu.bf16(x), gpu.bf16(w1), gpu.bf16(w2),
            m, k, n, k)
    assert_close(gpu.read_bf16(out), oracle.mlp(x, w1, w2, m, k, n),
                 what="low SwiGLU tiles", chained=1)
