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
