"""What the backend launches for a call, found without a GPU: a child process
loads the built library on a HIP runtime that only keeps a list of launches
(fake_hip.cpp, a device of 256 CUs) and makes the calls.

A call is [function, argument, ...].  Tensor arguments are ["bf16", elements],
["f32", ...] or ["u32", ...]; ["=", n] is the n-th tensor made before, None is
NULL, whole numbers and floats are passed as the prototype in h3hip.py says."""
import ctypes
import functools
import json
import os
import shutil
import subprocess
import sys
import tempfile

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
LIB = os.path.join(ROOT, "h3.c_amd", "lib", "libh3_gpu_hip.so")


class Launch(dict):
    """kernel, grid, block, lds (dynamic bytes), lds_limit, words."""
    __getattr__ = dict.__getitem__


@functools.lru_cache(maxsize=None)
def _fake():
    if not shutil.which("g++") or not os.path.isdir("/opt/rocm/include/hip"):
        pytest.skip("needs g++ and the HIP headers")
    out = os.path.join(tempfile.mkdtemp(prefix="fake_hip_"), "libfake_hip.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-fPIC", "-shared",
                    "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    os.path.join(HERE, "fake_hip.cpp"), "-o", out],
                   check=True)
    return out


def calls_made(calls, env=None, largest_block=None, at_start=None,
               contexts=1):
    """One (ok, error text, [Launch]) per call.  Allocations of more than
    `largest_block` bytes fail once the contexts and the tensors are there, of
    more than `at_start` bytes while the contexts are made.  Call i is made by
    context i % contexts."""
    proc = subprocess.run(
        [sys.executable, os.path.abspath(__file__), _fake()],
        input=json.dumps([calls, largest_block, at_start, contexts]), text=True,
        capture_output=True, env={**os.environ, **(env or {})}, timeout=300)
    assert proc.returncode == 0, proc.stderr[-2000:]
    return [(ok, error, [Launch(l) for l in launches])
            for ok, error, launches in json.loads(proc.stdout)]


def _child():
    fake = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
    sys.path.insert(0, os.path.join(ROOT, "h3.c_amd"))
    import h3hip
    calls, largest_block, at_start, contexts = json.loads(sys.stdin.read())

    def limit(size):
        fake.fake_largest_block(ctypes.c_size_t(-1 if size is None else size))

    limit(at_start)
    gpus = [h3hip.Gpu() for _ in range(contexts)]
    limit(None)
    made, ready = [], []
    for i, (name, *args) in enumerate(calls):
        gpu = gpus[i % contexts]
        values = []
        for a in args:
            if isinstance(a, list) and a[0] == "=":
                a = made[a[1]]
            elif isinstance(a, list):
                if a[0] == "u32":
                    a = gpu.L.h3_gpu_tensor_from_u32(gpu.h, None, a[1])
                else:
                    a = getattr(gpu, "new_" + a[0])(a[1])
                made.append(a)
            values.append(a)
        ready.append((gpu, name, values))
    limit(largest_block)
    out = []
    for gpu, name, values in ready:
        fake.fake_clear()
        gpu.begin()
        ok = getattr(gpu.L, name)(gpu.h, *values)
        error = gpu.error()
        error = "" if error == "unknown HIP error" else error  # none left
        gpu.submit()
        launches = []
        for i in range(fake.fake_launches()):
            text = ctypes.create_string_buffer(400)
            words = (ctypes.c_uint64 * 18)()
            fake.fake_launch(ctypes.c_size_t(i), text, 400, words)
            launches.append({"kernel": text.value.decode(),
                             "grid": list(words[:3]), "block": words[3],
                             "lds": words[4], "lds_limit": words[5],
                             "words": list(words[8:])})
        out.append([bool(ok), error, launches])
    print(json.dumps(out), flush=True)
    os._exit(0)  # nothing of the fake runtime is to be torn down


if __name__ == "__main__":
    _child()
