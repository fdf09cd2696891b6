"""The MFMA GEMM's K loop, as compiled, moves no accumulator, touches no
scratch memory, and waits for its loads with vmcnt(2) only.

The 16x16x32 kernel holds 64 accumulator blocks in all 256 AGPRs.  Small
changes around the loop (an extra live value, a divergent branch in the
tile loop) have made the register allocator rotate those blocks through
`v_accvgpr_mov` / `v_accvgpr_write` copies inside the K loop, or spill into
scratch there, which cost the split-K instances 60-150% of their time with
correct results.  Every instance keeps two L2 prefetch loads in flight
across the stage wait; a vmcnt(0) there (which the compiler adds
for a barrier with a fence) quietly cancels the prefetch, and the cold-
weight launches of the forward lose 4-10%.  This test compiles
csrc/hk_gemm.hip as the Makefile does
(and as the phase-trace build does), takes the instructions between the
first and the last MFMA of every kernel instance, and requires none of
those.  It needs hipcc, not a GPU.
"""
import functools
import os
import re
import shutil
import subprocess
import tempfile

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = os.path.join(ROOT, "h3.c_amd", "csrc", "hk_gemm.hip")
HIPCC = "/opt/rocm/bin/hipcc"
FLAGS = ["-O3", "-std=c++17", "-fPIC", "--offload-arch=gfx950",
         "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops"]
INSTANCES = {
    "hk_gemm_mfma<0>": "_Z12hk_gemm_mfmaILi0ELb0EEv12hk_gemm_args",
    "hk_gemm_mfma<1> (SwiGLU)": "_Z12hk_gemm_mfmaILi1ELb0EEv12hk_gemm_args",
    "hk_gemm_mfma<2> (GELU)": "_Z12hk_gemm_mfmaILi2ELb0EEv12hk_gemm_args",
    "hk_gemm_mfma<0, group>": "_Z12hk_gemm_mfmaILi0ELb1EEv12hk_gemm_args",
    "hk_gemm_mfma<3> (split-K)": "_Z12hk_gemm_mfmaILi3ELb0EEv12hk_gemm_args",
    "hk_gemm_mfma<4> (split-K SwiGLU)":
        "_Z12hk_gemm_mfmaILi4ELb0EEv12hk_gemm_args",
}
# the tiles of 128 to 224 rows; nothing cuts 224-row tiles along K
INSTANCES.update({
    f"hk_gemm_mfma_low<{epi}, {'group, ' * group}{jb}>":
        f"_Z16hk_gemm_mfma_lowILi{epi}ELb{group}ELi{jb}EEv12hk_gemm_args"
    for epi, group in [(0, 0), (1, 0), (2, 0), (0, 1), (3, 0), (4, 0)]
    for jb in (4, 5, 6, 7) if jb < 7 or epi < 3})
BAD = re.compile(r"\b(v_accvgpr_mov_b32|v_accvgpr_write_b32|scratch_\w+)\b")


@functools.lru_cache(maxsize=None)
def _assembly(*extra):
    """The lines of csrc/hk_gemm.hip's device assembly."""
    work = tempfile.mkdtemp(prefix="hk_isa_")
    try:
        subprocess.run([HIPCC, *FLAGS, *extra, "--save-temps", "-c", SRC,
                        "-o", os.path.join(work, "hk_gemm.o")], cwd=work,
                       check=True, capture_output=True)
        asm = [f for f in os.listdir(work)
               if f.endswith(".s") and "amdgcn" in f]
        assert asm, "no device assembly written"
        return open(os.path.join(work, asm[0])).read().splitlines()
    finally:
        shutil.rmtree(work, ignore_errors=True)


def _body(text, sym):
    start = text.index(next(l for l in text if l.startswith(sym + ":")))
    end = next(i for i in range(start + 1, len(text))
               if text[i].startswith(".Lfunc_end"))
    return text[start:end]


def _k_loop_offenders(extra):
    text = _assembly(*extra)
    found = {}
    for name, sym in INSTANCES.items():
        body = _body(text, sym)
        mfma = [i for i, l in enumerate(body) if "v_mfma_" in l]
        jb = int((re.search(r"ELi(\d)EEv", sym) or [8, 8])[1])
        assert len(mfma) == 16 * jb, (name, len(mfma))
        loop = body[mfma[0]:mfma[-1]]
        found[name] = [l.strip() for l in loop if BAD.search(l)]
        waits = [int(m.group(1)) for l in loop
                 for m in [re.search(r"s_waitcnt\b.*vmcnt\((\d+)\)", l)]
                 if m]
        # the prefetch loads may follow the last MFMA: count them up to the
        # loop's back-edge branch
        back = next(i for i in range(mfma[-1], len(body))
                    if body[i].strip().startswith("s_cbranch"))
        pf = [l for l in body[mfma[0]:back]
              if re.search(r"buffer_load_dword\b.*\blds\b", l)]
        if waits != [2]:
            found[name].append(f"stage waits vmcnt{waits}, want [2]")
        if len(pf) != 2:
            found[name].append(f"{len(pf)} prefetch loads, want 2")
    return found


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not installed")
@pytest.mark.parametrize("extra", [[], ["-DHK_GEMM_TRACE"]],
                         ids=["product", "phase-trace"])
def test_gemm_k_loop_has_no_accumulator_copies_or_scratch(extra):
    offenders = _k_loop_offenders(extra)
    bad = {k: (len(v), v[:3]) for k, v in offenders.items() if v}
    assert not bad, bad


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not installed")
@pytest.mark.parametrize("mb,ahead", [(1, 3), (2, 1), (2, 3), (3, 3), (4, 3)])
def test_skinny_loads_leave_in_the_order_its_waits_count(mb, ahead):
    """hk_gemm_skinny<MB, XA> waits until all but the last 4 + (XA - 1)(MB + 4)
    loads have landed, which is X of the step at hand only if every step's MB
    X loads (to LDS) leave before its four W loads, and steps in order.  The
    three steps of a partial turn (none with one stage ahead) load nothing, and
    nothing is in flight at the end."""
    body = _body(_assembly(),
                 f"_Z14hk_gemm_skinnyILi{mb}ELi{ahead}EEv14hk_skinny_args")
    loads = [(i, "X" if re.search(r"\blds\b", l) else "W")
             for i, l in enumerate(body) if "buffer_load_" in l]
    step = "X" * mb + "WWWW"
    ring = "".join("X" * mb * (d < ahead) + "WWWW" for d in range(3))
    assert "".join(w for _, w in loads) == ring + 4 * step
    mfma = [i for i, l in enumerate(body) if "v_mfma_" in l]
    assert len(mfma) == (4 + 3 * (ahead > 1)) * 4 * mb
    # the turn comes first, its loads (but the first X) among its MFMAs
    first, last = mfma[0], mfma[4 * 4 * mb - 1]
    among = "".join(w for i, w in loads if first < i < last)
    assert (4 * step).endswith(among) and among.endswith(3 * step)
    assert not [l for l in body[first:last]
                if "s_cbranch" in l or "scratch_" in l]
    # the kernel's own waits, apart from the compiler's
    asm = re.findall(r"#ASMSTART\n\s*s_waitcnt vmcnt\((\d+)\)",
                     "\n".join(body))
    turn = [4 + (ahead - 1) * (mb + 4)] * 4
    tail = [4 + (2 - d) * (mb + 4) for d in range(3)] if ahead > 1 else []
    assert [int(w) for w in asm] == turn + tail + [0]
