"""Every buffer load of a skinny GEMM launch, walked on the CPU: a load is
either inside its operand or turned away by the range check.

The check lets a 16-byte load through when its lane offset is below the
buffer's bytes less the scalar offset, as unsigned numbers: a scalar offset
past the end would make that bound huge and let a dead step read far outside
the operand (one row, or four W rows of one or two k steps)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

WALK = r"""
#include <stdio.h>
#include <initializer_list>
#include "hk_skinny.h"
static int bad;
/* rows x k operand, of which the kernel asks for rows from `first` to `asked`
 * (those past the end as row `rows`), in pieces of `piece` k steps loaded up
 * to `ahead` ahead */
static void walk(uint32_t rows, uint32_t asked, uint32_t k, uint32_t piece,
                 uint32_t ahead, uint32_t first = 0) {
    const uint32_t bytes = rows * k * 2, k_steps = k / 64;
    for (uint32_t base = 0; base < k_steps; base += piece) {
        const uint32_t steps =
            piece < k_steps - base ? piece : k_steps - base;
        const uint32_t turns =
            (steps + HK_SKINNY_RING - 1) / HK_SKINNY_RING * HK_SKINNY_RING;
        for (uint32_t s = 0; s < turns + ahead; s++) {
            const uint32_t at = hk_skinny_k_bytes(base + s, k_steps);
            for (uint32_t r = first; r < asked; r++)
                for (uint32_t chunk = 0; chunk < 8; chunk++) {
                    const uint32_t row = r < rows ? r : rows;
                    const uint32_t lane =
                        hk_skinny_lane(row * k * 2 + chunk * 16, s, steps);
                    const bool passes = lane < bytes - at; /* unsigned */
                    const bool wanted = r < rows && s < steps;
                    if (at >= bytes || passes != wanted ||
                        (passes && (uint64_t)lane + at + 16 > bytes)) {
                        if (!bad++)
                            printf("rows %u k %u piece %u base %u step %u "
                                   "row %u: lane %u scalar %u of %u\n",
                                   rows, k, piece, base, s, r, lane, at,
                                   bytes);
                    }
                }
        }
    }
}
int main() {
    const uint32_t rows[] = {1, 2, 3, 4, 7, 8, 31, 32, 33};
    for (uint32_t r : rows)
        for (uint32_t k_steps = 1; k_steps <= 41; k_steps++)
            for (uint32_t piece = 4; piece < k_steps + 4; piece += 4) {
                walk(r, 64, k_steps * 64, piece, 1); /* X, one or three */
                walk(r, 64, k_steps * 64, piece, 3); /* steps ahead; W */
            }
    /* the largest W that the GEMMs take: 2 K + 4096 bytes below 2^32 */
    for (uint32_t k_steps : {1u, 2u, 3u, 42u, 84u, 224u}) {
        const uint32_t k = k_steps * 64;
        const uint32_t rows = (uint32_t)((0xffffffffull - 4096 - 2 * k) /
                                         (2 * k)) & ~3u;
        for (uint32_t piece = 4; piece < k_steps + 4; piece += 4)
            walk(rows, rows + 128, k, piece, 3, rows - 8);
    }
    if (bad) printf("%d loads\n", bad);
    return bad != 0;
}
"""


@pytest.mark.skipif(not shutil.which("g++"), reason="g++ not installed")
def test_every_load_is_inside_or_turned_away(tmp_path):
    src = tmp_path / "walk.cpp"
    src.write_text(WALK)
    exe = str(tmp_path / "walk")
    subprocess.run(["g++", "-std=c++17", "-O2", "-I",
                    os.path.join(ROOT, "h3.c_amd", "csrc"), str(src), "-o",
                    exe], check=True)
    proc = subprocess.run([exe], capture_output=True, text=True)
    assert proc.returncode == 0, proc.stdout
