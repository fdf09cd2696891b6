"""Which kernels a call launches, on 256 CUs, without a GPU (launches.py)."""
import pytest

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


def linear_f32(m, k, n):
    return ["h3_gpu_linear_f32", ["f32", m * n], ["f32", m * k],
            ["f32", n * k], ["f32", n], m, k, n]


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
