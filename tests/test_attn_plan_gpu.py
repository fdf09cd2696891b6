"""Dense attention under each launch plan (256-query items whole or with the
last round cut along the keys, 128-query items), at the real head counts: the
first, a middle and the last head against the oracle."""
import ctypes as C
import math

import numpy as np
import pytest

import oracle
from conftest import assert_close, rand_bf16, sdpa_p_rounding_bound

pytestmark = pytest.mark.gpu

HD, SCALE = 128, 1.0 / math.sqrt(128)


def _heads_close(got, q, k, v, rows, heads):
    pick = lambda x, h: np.ascontiguousarray(  # noqa: E731
        x.reshape(rows, heads, HD)[:, h])
    for h in (0, heads // 2, heads - 1):
        a = [pick(x, h).ravel() for x in (q, k, v)]
        want = oracle.sdpa(*a, rows, rows, 1, HD, SCALE)
        assert_close(pick(got, h).ravel(), want, what=f"head {h}",
                     extra_abs=sdpa_p_rounding_bound(*a, rows, rows, 1, HD,
                                                     SCALE))


# rows, heads, and the plan (test_routes.py checks it): queries an item, pieces
# of the last round's items
PLANS = [
    (65, 40, 128, 1), (300, 56, 128, 1), (512, 56, 128, 1),  # under a round
    (600, 56, 256, 1),                       # one round, whole
    (5600, 6, 256, 3), (11224, 3, 256, 5),   # one round, long: cut
    (1100, 56, 128, 1), (2100, 40, 128, 1),  # 128-query items: 504, 680
    (1200, 56, 256, 5),                      # a cut last round
    (1700, 56, 256, 1),                      # two rounds, whole
    (1280, 10, 256, 5),                      # half a round, even pieces
]


@pytest.mark.parametrize("rows,heads,queries,pieces", PLANS)
def test_sdpa_plans(gpu, rows, heads, queries, pieces):
    rng = np.random.default_rng(rows + heads)
    q, k, v = (rand_bf16(rng, rows * heads * HD) for _ in range(3))
    out = gpu.new_bf16(rows * heads * HD)
    gpu.run("h3_gpu_sdpa_bf16", out, gpu.bf16(q), gpu.bf16(k), gpu.bf16(v),
            rows, heads, HD, C.c_float(SCALE))
    _heads_close(gpu.read_bf16(out), q, k, v, rows, heads)


@pytest.mark.parametrize("rows,heads", [(300, 40), (1100, 56)])
def test_q_norm_rope_in_128_query_items(gpu, rows, heads):
    """The fused-QKV entry on 128-query items: bit for bit the result of
    normalising and rotating Q first."""
    rng = np.random.default_rng(rows)
    inner = heads * HD
    qkv = rand_bf16(rng, rows * 3 * inner)
    w = rand_bf16(rng, HD, 0.1, 1.0)
    ang = rng.uniform(-20, 20, rows * 48).astype(np.float32)
    cos, sin = gpu.bf16(np.cos(ang)), gpu.bf16(np.sin(ang))
    tw, out = gpu.bf16(w), gpu.new_bf16(rows * inner)
    fused = gpu.bf16(qkv)
    gpu.run("h3_hip_qk_norm_rope_inplace_bf16", fused, tw, tw, cos, sin, rows,
            heads, HD, 48, C.c_float(1e-6), 1)
    gpu.run("h3_hip_sdpa_qkv_norm_rope_bf16", out, fused, tw, cos, sin, rows,
            heads, HD, 48, C.c_float(1e-6), C.c_float(SCALE))
    got = gpu.read_bf16(out)
    both = gpu.bf16(qkv)
    gpu.run("h3_hip_qk_norm_rope_inplace_bf16", both, tw, tw, cos, sin, rows,
            heads, HD, 48, C.c_float(1e-6), 0)
    gpu.run("h3_hip_sdpa_qkv_bf16", out, both, rows, heads, HD,
            C.c_float(SCALE))
    assert np.array_equal(gpu.read_bf16(out), got)
    rows_of = gpu.read_bf16(both).reshape(rows, 3, inner)
    _heads_close(got, *[np.ascontiguousarray(rows_of[:, i]).ravel()
                        for i in range(3)], rows, heads)
