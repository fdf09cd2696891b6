"""Which kernels a call launches, on 256 CUs, without a GPU (launches.py)."""
import pytest

import test_attn_plan_gpu as attn_plan
import test_gemm_rows_gpu as gemm_rows
from launches import calls_made


def head(rows, width, n):
    return ["h3_gpu_adaln_linear_bf16", ["bf16", rows * n], ["f32", rows],
            ["bf16", rows * width], 0, ["bf16", width], ["bf16", 2 * width],
            ["u32", rows], ["bf16", n * width], ["bf16", n], rows, width, n,
            2, 0, 1, 1e-5]


@pytest.mark.parametrize("rows,n", [(1040, 32), (1040, 96), (2100, 96)])
@pytest.mark.parametrize("width", [3968, 4000, 4032, 4064, 5376, 8192])
def test_head_lds_limit(rows, n, width):
    """Dynamic LDS plus the kernel's static 16 + 1 floats a row stay within
    64 KiB, or the kernel's limit is raised first; a fresh process each, since
    a limit once raised stays."""
    (ok, error, (launch,)), = calls_made([head(rows, width, n)])
    assert ok, error
    assert launch.kernel.startswith("hk_adaln_head_mfma<")
    block_rows = int(launch.kernel.split(", ")[1].rstrip(">"))
    assert block_rows == 16
    assert launch.lds <= launch.lds_limit
    if launch.lds + 17 * 4 * block_rows > 64 * 1024:
        assert launch.lds_limit > 64 * 1024


@pytest.mark.parametrize("rows,width,n,kernel", [
    (74, 5376, 32, "hk_adaln_head_mfma"), (74, 128, 96, "hk_adaln_head_mfma"),
    (2048, 352, 32, "hk_adaln_head_kernel"),
    (2049, 352, 32, "hk_adaln_head_mfma"),
    (2049, 64, 64, "hk_adaln_head_mfma"),
    (2049, 64, 63, "hk_adaln_head_kernel"),
    (74, 32, 383, "hk_adaln_head_kernel"), (74, 32, 384, "hk_adaln_head_mfma"),
])
def test_head_of_a_small_weight(rows, width, n, kernel):
    (ok, error, (launch,)), = calls_made([head(rows, width, n)])
    assert ok, error
    assert launch.kernel.split("<")[0] == kernel


def linear_f32(m, k, n):
    return ["h3_gpu_linear_f32", ["f32", m * n], ["f32", m * k],
            ["f32", n * k], ["f32", n], m, k, n]


# rows, K, N, row blocks of 16 a workgroup; where K has pieces, or one round
# of CUs does not hold fewer rows a workgroup, the fewest that hold all rows
LINEAR_F32 = [(39, 256, 5376, 3), (101, 5376, 2688, 8), (39, 5376, 2688, 3),
              (16, 64, 64, 1), (39, 64, 64, 2), (128, 64, 64, 2),
              (1000, 128, 64, 2), (1000, 128, 512, 4), (128, 64, 5376, 8),
              (128, 2016, 64, 2), (128, 2048, 64, 8)]


def test_f32_linear_rows_of_a_workgroup():
    made = calls_made([linear_f32(*size[:3]) for size in LINEAR_F32])
    for (m, k, n, blocks), (ok, error, launches) in zip(LINEAR_F32, made):
        assert ok, error
        kernel = launches[0].kernel
        assert kernel.startswith(f"hk_linear_f32_mfma<{blocks}, "), (m, k, n)
        assert launches[0].lds <= max(launches[0].lds_limit, 64 * 1024)
    # few products each: one thread an output, up to 65536 outputs
    made = calls_made([linear_f32(128, 16, 512), linear_f32(129, 16, 512),
                       linear_f32(128, 20, 512)])
    assert [launches[0].kernel[:18] for _, _, launches in made] == [
        "hk_linear_f32_kern", "hk_linear_f32_mfma", "hk_linear_f32_mfma"]


def patch(rows, k, n):
    return ["h3_hip_patch_linear_bf16_offset", ["bf16", rows * n], 0,
            ["f32", rows * k], 0, ["f32", n * k], ["f32", n], rows, k, n]


@pytest.mark.parametrize("call,kernel,simple", [
    (linear_f32(39, 256, 5376), "hk_linear_f32_mfma<3, 3>",
     "hk_linear_f32_kernel"),
    (patch(1792, 96, 5376), "hk_patch_linear_mfma", "hk_patch_linear_kernel"),
    (head(74, 5376, 32), "hk_adaln_head_mfma<2, 4>", "hk_adaln_head_kernel"),
])
def test_reference_switch_takes_the_simple_kernels(call, kernel, simple):
    for flag, want in (("0", kernel), ("1", simple)):
        (ok, error, launches), = calls_made(
            [call], env={"H3_HIP_REFERENCE": flag})
        assert ok, error
        assert [l.kernel for l in launches] == [want]


MIB = 1 << 20


def linear(m, k, n, fn="h3_gpu_linear_bf16"):
    return [fn, ["bf16", m * n], ["bf16", m * k], ["bf16", n * k], None, m, k,
            n]


@pytest.mark.parametrize("call,kernels,pieces", [
    (linear(128, 14336, 128),
     ["hk_gemm_skinny<4, 3>", "hk_skinny_reduce"], 1),
    (linear_f32(101, 5376, 2688),
     ["hk_linear_f32_mfma<8, 1>", "hk_linear_f32_reduce"], 2),
])
def test_no_scratch_takes_one_piece_and_leaves_no_error(call, kernels,
                                                        pieces):
    """`pieces`: the grid's dimension that counts the pieces of K."""
    for limit in (None, MIB // 2):
        (ok, error, launches), = calls_made([call], largest_block=limit,
                                            at_start=limit)
        assert ok and not error, error
        assert (launches[0].grid[pieces] > 1) == (limit is None)
        assert [l.kernel for l in launches] == kernels[:len(launches)]
        assert len(launches) == (2 if limit is None else 1)


def attention(rows, heads):
    n = rows * heads * 128
    return ["h3_gpu_sdpa_bf16", *[["bf16", n]] * 4, rows, heads, 128, 0.088]


def attention_rope(rows, heads):
    n = rows * heads * 128
    return ["h3_hip_sdpa_rope_bf16", *[["bf16", n]] * 4,
            *[["bf16", rows * 48]] * 2, rows, heads, 128, 48, 0.088]


@pytest.mark.parametrize("call,limit,kernels,whole,grid", [
    (linear(512, 14336, 5376), 0,
     ["hk_gemm_mfma<3, false>", "hk_splitk_reduce<0>"],
     ["hk_gemm_mfma<0, false>"], 48),  # 42 tiles, in eights
    (linear(9720, 5120, 13824), 0,
     ["hk_gemm_mfma<0, false>", "hk_gemm_mfma<3, false>",
      "hk_splitk_reduce<0>"], ["hk_gemm_mfma<0, false>"],
     232),                             # 2052 tiles in nine rounds
    (attention(2378, 56), 0,
     ["hk_flash_fwd<false, false, 8>", "hk_flash_fwd<false, true, 8>",
      "hk_flash_combine<256u>"], ["hk_flash_fwd<false, false, 8>"], 560),
    # the rotated keys still need theirs, 50 of 67 MiB (blocks double)
    (attention_rope(3584, 56), 64 * MIB,
     ["hk_rope_pack", "hk_rope_keys", "hk_flash_fwd<false, false, 8>",
      "hk_flash_fwd<false, true, 8>", "hk_flash_combine<256u>"],
     ["hk_rope_pack", "hk_rope_keys", "hk_flash_fwd<false, false, 8>"],
     784),
])
def test_no_scratch_runs_whole(call, limit, kernels, whole, grid):
    """Tiles and attention items that would be cut run whole where scratch for
    the pieces cannot be had."""
    for largest, want in ((None, kernels), (limit, whole)):
        (ok, error, launches), = calls_made([call], largest_block=largest,
                                            at_start=largest)
        assert ok and not error, error
        assert [l.kernel for l in launches] == want
    assert launches[-1].grid == [grid, 1, 1]


@pytest.mark.parametrize("rows", [8, 40, 64, 128])
def test_noalloc_pieces_of_two_contexts_share_nothing(rows):
    """Few rows: each context's pieces have scratch of its own, held since its
    creation, so that calls of two contexts may overlap."""
    fn = "h3_hip_linear_bf16_noalloc"
    made = calls_made([linear(rows, 14336, 5376, fn),
                       linear(rows, 14336, 5376, fn)], contexts=2,
                      largest_block=0)
    partial = []
    for ok, error, launches in made:
        assert ok and not error, error
        assert [l.kernel for l in launches][1:] == ["hk_skinny_reduce"]
        assert launches[0].grid[1] > 1
        size = launches[0].grid[0] * launches[0].grid[1] * 65536
        partial.append((launches[0].words[7], size))
    (a, size_a), (b, size_b) = partial
    assert a and b and (a + size_a <= b or b + size_b <= a)


@pytest.mark.parametrize("rows,kernel", [(39, "hk_gemm_skinny<2, 1>"),
                                         (128, "hk_gemm_skinny<4, 3>")])
def test_few_rows_take_the_skinny_kernel_with_any_weight(rows, kernel):
    """Any weight that the GEMMs take (up to 4 GiB)."""
    for n in (5376, 420000, 780000):  # 29 MB, 2.3 GB, 4.2 GB
        (ok, error, launches), = calls_made([linear(rows, 2688, n)])
        assert ok, error
        assert launches[0].kernel in (kernel, kernel[:-2] + "3>")


def test_one_x_stage_ahead_for_rounds_of_two_row_blocks_and_long_k():
    sizes = {(40, 2688, 96768): "hk_gemm_skinny<2, 1>",
             (40, 320, 96768): "hk_gemm_skinny<2, 3>",
             (64, 1024, 32768): "hk_gemm_skinny<2, 3>",
             (8, 2688, 96768): "hk_gemm_skinny<1, 3>"}
    made = calls_made([linear(*size) for size in sizes])
    for (ok, error, launches), kernel in zip(made, sizes.values()):
        assert ok, error
        assert [l.kernel for l in launches] == [kernel]


def test_up_to_128_rows_between_one_and_two_rounds():
    """97 to 128 rows of a short K whose skinny workgroups would fill between
    one and two rounds take tiles, never cut (no scratch in a call that may
    not allocate, whose contexts may overlap)."""
    tiles = [(97, 64, 36000), (128, 512, 32772), (128, 320, 65536),
             (100, 512, 45000)]
    skinny = [(96, 512, 36000), (128, 512, 32768), (128, 512, 65540),
              (128, 576, 36000), (1, 64, 36000)]
    made = calls_made([linear(*size, "h3_hip_linear_bf16_noalloc")
                       for size in tiles + skinny], largest_block=0)
    for i, (ok, error, launches) in enumerate(made):
        assert ok and not error, error
        kernel, = [l.kernel for l in launches]
        assert kernel.startswith("hk_gemm_mfma" if i < len(tiles) else
                                 "hk_gemm_skinny"), (tiles + skinny)[i]
        assert kernel.split("<")[1][0] == "0" or i >= len(tiles)


def pair(m, k, n):
    return ["h3_hip_linear_pair_bf16", *[["bf16", m * n]] * 2,
            ["bf16", m * k], ["bf16", n * k], ["bf16", n], ["bf16", n * k],
            None, m, k, n]


@pytest.mark.parametrize("limit", [None, 0])
def test_a_pair_of_few_rows_is_one_launch(limit):
    """Both problems in one skinny launch (grid z) and one sum of the pieces,
    within the scratch that the context holds; in two past one round of CUs."""
    sizes = [(1, 64, 4), (65, 512, 132), (128, 14336, 128), (97, 5120, 5120),
             (40, 128, 16384), (40, 128, 16388)]
    made = calls_made([pair(*size) for size in sizes], largest_block=limit)
    for (m, k, n), (ok, error, launches) in zip(sizes, made):
        assert ok and not error, error
        kernel = f"hk_gemm_skinny<{(m + 31) // 32}, 3>"
        wgs = -(-n // 128)
        if 2 * wgs > 256:
            assert [l.kernel for l in launches] == [kernel, kernel]
            continue
        first, *rest = launches
        assert first.kernel == kernel and first.grid[2] == 2
        assert 2 * wgs * first.grid[1] <= 256
        cut = first.grid[1] > 1
        assert cut == (k >= 1024)
        assert [(l.kernel, l.grid[1]) for l in rest] == (
            [("hk_skinny_reduce", 2)] if cut else [])


STORE, SWIGLU_UP, GELU_UP = 0, 1, 2


def mlp(m, k, n):
    return ["h3_gpu_mlp_bf16", ["bf16", m * k], ["bf16", m * k],
            ["bf16", 2 * n * k], ["bf16", n * k], m, k, n, k]


def gemm(m, k, n, epilogue):
    if epilogue == SWIGLU_UP:
        return mlp(m, k, n)
    return linear(m, k, n, "h3_gpu_linear_gelu_bf16" if epilogue == GELU_UP
                  else "h3_gpu_linear_bf16")


def gemm_kernels(rows, form, epilogue):
    def kernel(epi):
        return (f"hk_gemm_mfma<{epi}, false>" if rows == 256 else
                f"hk_gemm_mfma_low<{epi}, false, {rows // 32}>")
    partial = 4 if epilogue == SWIGLU_UP else 3
    cut = [kernel(partial), f"hk_splitk_reduce<{epilogue}>"]
    return {gemm_rows.WHOLE: [kernel(epilogue)], gemm_rows.CUT: cut,
            gemm_rows.TAIL: [kernel(epilogue)] + cut}[form]


def test_gemm_sizes_take_the_tiles_they_are_listed_under():
    """The sizes of the GPU tests: each tile height and form is reached."""
    sizes = ([(s, e) for s in gemm_rows.LINEAR for e in (STORE, GELU_UP)] +
             [(s, GELU_UP) for s in gemm_rows.GELU] +
             [(s, SWIGLU_UP) for s in gemm_rows.SWIGLU])
    made = calls_made([gemm(*s[2], e) for s, e in sizes])
    for ((rows, form, size), e), (ok, error, launches) in zip(sizes, made):
        want = gemm_kernels(rows, form, e)
        assert ok, error
        assert [l.kernel for l in launches][:len(want)] == want, size


# (m, K, N, epilogue), rows of a tile, form
MODEL_SIZES = [
    # 6144 and 9720 rows of the Wan block keep 256-row tiles: 224 rows were
    # 0.5% better by the estimate and 1.2% slower (FFN up at 6144)
    ((6144, 5120, 13824, GELU_UP), 256, gemm_rows.TAIL),
    ((6144, 13824, 5120, STORE), 256, gemm_rows.WHOLE),
    ((6144, 5120, 15360, STORE), 256, gemm_rows.WHOLE),
    ((6144, 5120, 5120, STORE), 256, gemm_rows.WHOLE),
    ((9720, 5120, 13824, GELU_UP), 256, gemm_rows.TAIL),
    ((9720, 13824, 5120, STORE), 256, gemm_rows.WHOLE),
    ((9720, 5120, 15360, STORE), 256, gemm_rows.WHOLE),
    # a long K, several bands: 948 and 957 us of the FFN with 192 rows
    ((4600, 13824, 5120, STORE), 256, gemm_rows.TAIL),
    ((7232, 13824, 5120, STORE), 192, gemm_rows.WHOLE),
    # more rounds: 339 and 380 us with 160 rows
    ((1400, 5376, 14336, SWIGLU_UP), 256, gemm_rows.WHOLE),
    # a last band of one row tile: 238 and 254 us with 224 rows
    ((2000, 5120, 13824, GELU_UP), 256, gemm_rows.WHOLE),
    # SwiGLU of 2900-3030 rows: 192 rows gain under 1.5%
    ((2960, 5376, 14336, SWIGLU_UP), 256, gemm_rows.TAIL),
    # every tile cut, long K, 252 pieces: 79 and 82 us with 160 rows
    ((300, 14336, 5376, STORE), 256, gemm_rows.CUT),
    # gains of 5% and more
    ((778, 5376, 21504, STORE), 160, gemm_rows.WHOLE),
    ((1600, 7168, 5376, STORE), 160, gemm_rows.WHOLE),
    ((2378, 14336, 5376, STORE), 224, gemm_rows.WHOLE),
    ((1300, 5120, 15360, STORE), 192, gemm_rows.WHOLE),
    ((350, 13824, 5120, STORE), 192, gemm_rows.CUT),
    ((100, 5120, 13824, GELU_UP), 128, gemm_rows.CUT),
]


def test_gemm_tile_heights_of_the_models():
    made = calls_made([gemm(*size) for size, _, _ in MODEL_SIZES])
    for (size, rows, form), (ok, error, launches) in zip(MODEL_SIZES, made):
        want = gemm_kernels(rows, form, size[3])
        assert ok, error
        assert [l.kernel for l in launches][:len(want)] == want, size


# sizes of test_ops_gpu.py whose comments name a path: rows of a tile, form
OPS_SIZES = [
    ((300, 5376, 1024, STORE), 160, gemm_rows.CUT),
    ((512, 5120, 5120, STORE), 256, gemm_rows.CUT),
    ((260, 2048, 516, STORE), 256, gemm_rows.CUT),
    ((600, 1088, 256, STORE), 256, gemm_rows.CUT),
    ((4096, 512, 4352, STORE), 160, gemm_rows.WHOLE),
    ((1292, 512, 22980, STORE), 256, gemm_rows.TAIL),
    ((4100, 256, 4200, STORE), 256, gemm_rows.WHOLE),
    ((300, 64, 520, STORE), 256, gemm_rows.WHOLE),
    ((2378, 128, 1000, STORE), 256, gemm_rows.WHOLE),
    ((64, 256, 512, SWIGLU_UP), 256, gemm_rows.WHOLE),
    ((300, 1024, 1536, SWIGLU_UP), 160, gemm_rows.CUT),
    ((130, 5376, 512, SWIGLU_UP), 160, gemm_rows.CUT),
    ((300, 512, 4608, SWIGLU_UP), 160, gemm_rows.CUT),
    ((300, 512, 17408, SWIGLU_UP), 128, gemm_rows.WHOLE),
    ((64, 512, 33280, SWIGLU_UP), 256, gemm_rows.TAIL),
    ((1292, 640, 22980, GELU_UP), 256, gemm_rows.TAIL),
]


def test_gemm_sizes_of_the_operator_tests():
    made = calls_made([gemm(*size) for size, _, _ in OPS_SIZES])
    for (size, rows, form), (ok, error, launches) in zip(OPS_SIZES, made):
        want = gemm_kernels(rows, form, size[3])
        assert ok, error
        assert [l.kernel for l in launches][:len(want)] == want, size


# measured both ways (us, whole and cut): 33240 x 1 729 and 551, 8408 x 4 185
# and 165; 8 x 5080 116 and 117, 10 x 4056 94 and 100 stay whole
PLANS = attn_plan.PLANS + [
    (33240, 1, 256, 7), (8408, 4, 256, 3), (5080, 8, 256, 1),
    (4056, 10, 256, 1), (2378, 16, 256, 1), (2378, 56, 256, 5),
    (2378, 4, 256, 6), (1900, 8, 256, 4), (6144, 40, 256, 1),
]


def test_attention_plans():
    """How dense attention runs: queries an item, pieces of the last round."""
    made = calls_made([attention(rows, heads) for rows, heads, _, _ in PLANS])
    got = []
    for (rows, heads, _, _), (ok, error, launches) in zip(PLANS, made):
        assert ok, error
        names = [l.kernel for l in launches]
        items = -(-rows // 256) * heads
        if names == ["hk_flash_fwd<false, false, 4>"]:
            got.append((rows, heads, 128, 1))
        elif names == ["hk_flash_fwd<false, false, 8>"]:
            got.append((rows, heads, 256, 1))
        else:
            assert names[-2:] == ["hk_flash_fwd<false, true, 8>",
                                  "hk_flash_combine<256u>"]
            got.append((rows, heads, 256,
                        launches[-2].grid[0] // (items % 256)))
    assert got == PLANS
