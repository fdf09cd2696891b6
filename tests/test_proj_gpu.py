"""The small projections on the matrix cores, at the edges of their tiles."""
import ctypes as C

import numpy as np
import pytest

import h3hip
import oracle
from conftest import assert_close, rand_bf16, to_f32

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,k,n", [
    (1, 4, 1), (3, 20, 5),          # one thread an output, a step's tail
    (16, 256, 16), (17, 260, 33),   # a full tile, one row and column more
    (33, 128, 47), (48, 96, 64), (49, 2052, 31),
    (64, 516, 18), (65, 512, 17), (96, 1040, 16), (97, 64, 5),
    (128, 300, 33), (129, 96, 20),  # every height, one and two row blocks
    (39, 256, 5376), (101, 5376, 2688),
    (65, 2048, 33), (96, 2052, 17),  # 96 rows a workgroup
    (1000, 128, 512), (128, 64, 5376), (70000, 4, 3),
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


@pytest.mark.parametrize("rows,k,n,mapped", [
    (1, 4, 4, False), (63, 12, 124, False), (64, 32, 128, True),
    (65, 36, 132, True), (130, 96, 5376, False), (33, 100, 260, True),
    (74, 32, 5376, False),
    (9, 6, 8, False), (9, 8, 6, False),  # K % 4, N % 4: the general kernel
])
def test_patch_linear_tiles_bit_exact(gpu, rows, k, n, mapped):
    """Bit for bit the sequential fmaf order, through every tile edge, from
    an offset input into an offset output, with values whose products
    overflow, vanish and cancel."""
    rng = np.random.default_rng(rows + k + n)
    x = rng.standard_normal((rows, k)).astype(np.float32)
    x *= np.exp2(rng.integers(-75, 66, (rows, k))).astype(np.float32)
    w = rng.standard_normal((n, k)).astype(np.float32)
    w *= np.exp2(rng.integers(-75, 66, (n, k))).astype(np.float32)
    b = rng.standard_normal(n).astype(np.float32)
    out_rows = rows + 7
    tx, tw, tb = gpu.f32(np.r_[np.zeros(4, np.float32), x.ravel()]), \
        gpu.f32(w), gpu.f32(b)
    if mapped:
        rm = rng.permutation(out_rows)[:rows].astype(np.uint32)
        out = gpu.bf16(np.full(out_rows * n, 7, np.uint16))
        gpu.run("h3_hip_patch_linear_bf16_map", out, gpu.f32(x), tw, tb,
                gpu.u32(rm), out_rows, rows, k, n)
    else:
        rm = np.arange(3, 3 + rows, dtype=np.uint32)
        out = gpu.bf16(np.full(out_rows * n, 7, np.uint16))
        gpu.run("h3_hip_patch_linear_bf16_offset", out, 3 * n, tx, 4, tw, tb,
                rows, k, n)
    got = gpu.read_bf16(out).reshape(out_rows, n)
    want = oracle.patch_linear(x.ravel(), w.ravel(), b, rows, k, n,
                               row_map=rm, out_rows=out_rows)
    want = want.reshape(out_rows, n)
    nan = np.isnan(to_f32(want))
    np.testing.assert_array_equal(np.isnan(to_f32(got[rm])), nan[rm])
    np.testing.assert_array_equal(got[rm][~nan[rm]], want[rm][~nan[rm]])
    rest = np.setdiff1d(np.arange(out_rows), rm)
    assert (got[rest] == 7).all()


@pytest.mark.parametrize("rows,width,n", [
    (1, 32, 1), (16, 256, 32), (17, 288, 33), (31, 6144, 96), (5, 5376, 95),
    (33, 5376, 32), (3, 512, 97), (2, 8192, 48),
    (1025, 64, 32), (517, 96, 33),  # 16 rows a workgroup
    (2049, 64, 96), (2100, 5376, 50),  # and 96 columns
    (1, 4096, 3), (1025, 384, 32), (517, 128, 97), (2049, 128, 96),
    (1025, 4032, 32), (1040, 4000, 96),  # just over 64 KiB of LDS
    (4, 8224, 96), (4, 264, 8),  # the general kernel, as with small weights
])
@pytest.mark.parametrize("shared", [True, False])
def test_adaln_head_tiles(gpu, rows, width, n, shared):
    """The head against the oracle through its row, width and column edges:
    one bf16 flip of a normalised value moves an output by 2^-8 of one
    product, the composite bound of assert_close."""
    rng = np.random.default_rng(rows + width + n)
    slots, mods = 3, 4
    x = rand_bf16(rng, (rows + 2) * width)
    nw = rand_bf16(rng, width, 0.1, 1.0)
    mod = rand_bf16(rng, mods * slots * width, 0.2)
    rm = rng.integers(0, mods, rows).astype(np.uint32)
    if shared:
        rm[:] = 2
    w, b = rand_bf16(rng, n * width, 0.05), rand_bf16(rng, n, 0.1)
    for bias in (b, None):
        want, inv = oracle.adaln_linear(x[2 * width:], nw, mod, rm, w, bias,
                                        rows, width, n, slots, 2, 0, 1e-5)
        out, tinv = gpu.new_bf16(rows * n), gpu.new_f32(rows)
        gpu.run("h3_gpu_adaln_linear_bf16", out, tinv, gpu.bf16(x), 2 * width,
                gpu.bf16(nw), gpu.bf16(mod), gpu.u32(rm), gpu.bf16(w),
                None if bias is None else gpu.bf16(bias), rows, width, n,
                slots, 2, 0, C.c_float(1e-5))
        np.testing.assert_allclose(gpu.read_f32(tinv), inv, rtol=1e-5)
        assert_close(gpu.read_bf16(out), want, what="head", chained=1)


def test_simple_kernels_agree(gpu, monkeypatch):
    """The three projections at the models' widths against the simple kernels
    of H3_HIP_REFERENCE=1: F32 sums within both orders' bounds (each K + 16
    half-ulps of the sum of magnitudes), the patch projection bit for bit, the
    head within the composite bound."""
    rng = np.random.default_rng(5)
    f32 = lambda *s: rng.standard_normal(s).astype(np.float32)  # noqa: E731
    m, k, n = 39, 5376, 2688
    x, w, b = f32(m, k), f32(n, k) * np.float32(0.02), f32(n)
    px, pw, pb = f32(300, 96), f32(5376, 96), f32(5376)
    hx, hw = rand_bf16(rng, 300 * 5376), rand_bf16(rng, 96 * 5376, 0.02)
    nw, mod = rand_bf16(rng, 5376, 0.1, 1.0), rand_bf16(rng, 8 * 5376, 0.1)
    hb, rm = rand_bf16(rng, 96), rng.integers(0, 4, 300).astype(np.uint32)

    def results(g):
        o, p = g.new_f32(m * n), g.new_bf16(300 * 5376)
        y, inv = g.new_bf16(300 * 96), g.new_f32(300)
        g.run("h3_gpu_linear_f32", o, g.f32(x), g.f32(w), g.f32(b), m, k, n)
        g.run("h3_gpu_patch_linear_bf16_offset", p, 0, g.f32(px), 0,
              g.f32(pw), g.f32(pb), 300, 96, 5376)
        g.run("h3_gpu_adaln_linear_bf16", y, inv, g.bf16(hx), 0, g.bf16(nw),
              g.bf16(mod), g.u32(rm), g.bf16(hw), g.bf16(hb), 300, 5376, 96,
              2, 0, 1, C.c_float(1e-5))
        return (g.read_f32(o), g.read_bf16(p), g.read_bf16(y),
                g.read_f32(inv))

    fast = results(gpu)
    monkeypatch.setenv("H3_HIP_REFERENCE", "1")
    with h3hip.Gpu() as g:
        simple = results(g)
    terms = np.abs(x).astype(np.float64) @ np.abs(w).astype(np.float64).T
    bound = 2 * (k + 16) * 2.0 ** -24 * (terms + np.abs(b))
    d = np.abs(fast[0].astype(np.float64) - simple[0])
    assert (d <= bound.ravel()).all()
    np.testing.assert_array_equal(fast[1], simple[1])
    assert_close(fast[2], simple[2], what="head", chained=1)
    np.testing.assert_allclose(fast[3], simple[3], rtol=1e-5)
