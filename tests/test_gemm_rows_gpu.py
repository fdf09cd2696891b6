"""The MFMA GEMM's lower tiles (128 to 224 rows) with every epilogue, in plain
rounds and with every tile cut along K, and 256-row tiles with a cut tail.
test_routes.py checks that each size takes the kernel it is listed under."""
import numpy as np
import pytest

import oracle
from conftest import assert_close, rand_bf16

pytestmark = pytest.mark.gpu

# rows of a tile, form, (m, k, n) of a linear with and without GELU, and of
# the SwiGLU projection
WHOLE, CUT, TAIL = "whole", "every tile cut", "a cut tail"
LINEAR = [
    (128, WHOLE, (262, 512, 33220)), (128, WHOLE, (330, 1024, 16388)),
    (160, WHOLE, (262, 512, 16576)), (160, WHOLE, (129, 512, 33220)),
    (192, WHOLE, (129, 448, 196)), (192, WHOLE, (161, 448, 196)),
    (224, WHOLE, (199, 448, 11460)),
    (160, CUT, (129, 2112, 1988)), (160, CUT, (262, 2112, 960)),
    (192, CUT, (129, 2112, 1220)),
    (256, WHOLE, (199, 448, 6084)),
    (256, TAIL, (1292, 640, 22980)),
]
# up to 128 rows: with GELU only, the plain linear is skinny there
GELU = [
    (128, WHOLE, (128, 512, 33220)),
    (128, CUT, (64, 2112, 1988)), (128, CUT, (128, 640, 8260)),
    (192, CUT, (1, 2112, 1220)),
]
SWIGLU = [
    (128, WHOLE, (64, 512, 16576)), (128, WHOLE, (300, 512, 17408)),
    (160, WHOLE, (262, 512, 8320)), (192, WHOLE, (129, 448, 64)),
    (224, WHOLE, (199, 448, 6144)),
    (128, CUT, (64, 2112, 960)), (128, CUT, (128, 640, 4224)),
    (160, CUT, (129, 2112, 960)), (160, CUT, (262, 2112, 576)),
    (192, CUT, (129, 2112, 576)),
    (256, WHOLE, (199, 448, 3008)),
    (256, TAIL, (64, 512, 33280)),
]


@pytest.mark.parametrize("gelu,rows,form,size",
                         [(g, *s) for g in (False, True) for s in LINEAR] +
                         [(True, *s) for s in GELU])
def test_linear_low_tiles(gpu, gelu, rows, form, size):
    m, k, n = size
    rng = np.random.default_rng(m + k + n)
    x, w = rand_bf16(rng, m * k), rand_bf16(rng, n * k, 0.05)
    b = rand_bf16(rng, n, 0.1)
    out = gpu.new_bf16(m * n)
    gpu.run("h3_gpu_linear_gelu_bf16" if gelu else "h3_gpu_linear_bf16", out,
            gpu.bf16(x), gpu.bf16(w), gpu.bf16(b), m, k, n)
    want = oracle.linear(x, w, b, m, k, n)
    if gelu:
        want = oracle.gelu(want)
    assert_close(gpu.read_bf16(out), want, what=f"{rows} rows, {form}",
                 chained=gelu)


@pytest.mark.parametrize("rows,form,size", SWIGLU)
def test_mlp_low_tiles(gpu, rows, form, size):
    """The same heights for the SwiGLU projection (128 columns a tile)."""
    m, k, n = size
    rng = np.random.default_rng(m + k + n)
    x = rand_bf16(rng, m * k)
    w1, w2 = rand_bf16(rng, 2 * n * k, 0.05), rand_bf16(rng, k * n, 0.05)
    out = gpu.new_bf16(m * k)
    gpu.run("h3_gpu_mlp_bf16", out, gpu.bf16(x), gpu.bf16(w1), gpu.bf16(w2),
            m, k, n, k)
    assert_close(gpu.read_bf16(out), oracle.mlp(x, w1, w2, m, k, n),
                 what=f"{rows} rows, {form}", chained=1)
