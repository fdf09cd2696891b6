"""The small projections on the matrix cores, at the edges of their tiles."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,k,n", [
    (1, 4, 1), (3, 20, 5),          # one step, a step's tail
    (16, 256, 16), (17, 260, 33),   # a full tile, one row and column more
    (33, 128, 47), (48, 96, 64), (49, 2052, 31),
    (64, 516, 18), (65, 512, 17),   # one and two row blocks
    (39, 256, 5376), (101, 5376, 2688),
    (5, 7, 9),                      # K % 4 != 0: the general kernel
])
def test_linear_f32(gpu, m, k, n):
    """Against float64; a chain of at most ceil(K / 8) + 16 products per wave
    and 8 partial sums round by at most K + 16 half-ulps (2^-24) of the sum
    of magnitudes, the sequential chain's own bound."""
    rng = np.random.default_rng(m * 1000 + n)
    x = rng.standard_normal((m, k)).astype(np.float32)
    w = rng.standard_normal((n, k)).astype(np.float32)
    for bias in (None, rng.standard_normal(n).astype(np.float32)):
        out = gpu.new_f32(m * n)
        gpu.run("h3_gpu_linear_f32", out, gpu.f32(x), gpu.f32(w),
                None if bias is None else gpu.f32(bias), m, k, n)
        got = gpu.read_f32(out).reshape(m, n).astype(np.float64)
        add = 0.0 if bias is None else bias.astype(np.float64)
        want = x.astype(np.float64) @ w.astype(np.float64).T + add
        terms = (np.abs(x).astype(np.float64) @
                 np.abs(w).astype(np.float64).T + np.abs(add))
        assert (np.abs(got - want) <= (k + 16) * 2.0 ** -24 * terms).all()


def test_linear_f32_nonfinite(gpu):
    """An infinity or a NaN reaches the outputs of its own row and column and
    no other, tile padding included."""
    m, k, n = 19, 36, 21
    x = np.ones((m, k), np.float32)
    w = np.ones((n, k), np.float32)
    x[18, 35], w[20, 3] = np.inf, np.nan
    out = gpu.new_f32(m * n)
    gpu.run("h3_gpu_linear_f32", out, gpu.f32(x), gpu.f32(w), None, m, k, n)
    got = gpu.read_f32(out).reshape(m, n)
    want = x @ w.T
    np.testing.assert_array_equal(got, want)
