"""What the host entry points launch, on the CPU: the library runs over a stand-in for the HIP runtime
(fake_hip.cc, preloaded into a child process), whose launches only call a hook here."""
import ctypes
import json
import os
import shutil
import subprocess
import sys

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
ROCM = os.environ.get("ROCM", "/opt/rocm")


# ---- the child process: each case returns what the test checks --------------------------------


class Launches:
    """The launches of one child: (kernel, grid, block, [argument addresses])."""

    def __init__(self):
        self.fake = ctypes.CDLL(os.environ["FAKE_HIP"])
        self.fake.fake_hip_freed.argtypes = [ctypes.c_uint64]
        kind = ctypes.CFUNCTYPE(None, ctypes.c_char_p, ctypes.c_uint32, ctypes.c_uint32, ctypes.POINTER(ctypes.c_void_p))
        self._hook = kind(lambda name, grid, block, args: self.on(name.decode(), grid, block, args))
        self.fake.fake_hip_hook(self._hook)
        sys.path.insert(0, os.path.join(ROOT, "qwen3-embedding-webgpu-prepacked_amd"))
        import qattn
        self.qattn, self.ctx = qattn, qattn.Context(0)
        self.on = lambda *a: None

    def word(self, args, index, kind=ctypes.c_uint32, offset=0):
        return kind.from_address(args[index] + offset).value


Q4_SHAPES = [(m, k, n) for k in (1024, 2048, 3072, 4096, 5120) for n in (1056, 4000)
             for m in (1, 40, 100, 200, 400, 1400, 2100, 4000, 5000, 9000)]


def weight_ranges():
    """[(m, k, n, kernel, weight range)] of projections whose caller passes more bytes than the tensor."""
    h, out = Launches(), []
    for m, k, n in Q4_SHAPES:
        def on(name, grid, block, args):
            out.append((m, k, n, name, h.word(args, 5)))  # x, ldx, M, K, w, w_bytes
        h.on = on
        need = h.qattn.lib().qattn_q4_compact_bytes(k, n)
        h.ctx.q4_matmul(1 << 20, m, k, 1 << 30, need + 5 * 640, n, 1 << 40)
        h.ctx.q4_matmul_swiglu(1 << 20, m, k, 1 << 30, h.qattn.lib().qattn_q4_compact_bytes(k, 2 * 1088) + 4, 1088, 1 << 40)
    return out


CASES = {f.__name__: f for f in (weight_ranges,)}


# ---- the tests --------------------------------------------------------------------------------


@pytest.fixture(scope="module")
def child(tmp_path_factory):
    compiler = shutil.which("g++")
    if not compiler or not os.path.isdir(os.path.join(ROCM, "include", "hip")):
        pytest.skip("no g++ or HIP headers")
    lib = str(tmp_path_factory.mktemp("fake") / "libfake_hip.so")
    subprocess.run([compiler, "-std=c++17", "-O1", "-shared", "-fPIC", "-w", "-I" + os.path.join(ROCM, "include"), "-o", lib,
                    os.path.join(HERE, "fake_hip.cc")], check=True)

    def run(case):
        preload = " ".join(v for v in (os.environ.get("LD_PRELOAD"), lib) if v)
        out = subprocess.run([sys.executable, os.path.abspath(__file__), case], check=True, capture_output=True, text=True,
                             env=dict(os.environ, LD_PRELOAD=preload, FAKE_HIP=lib), timeout=120)
        return json.loads(out.stdout)

    return run


def test_weight_ranges_end_with_the_tensor(child):
    """The kernels address weights by a per-lane offset, which the buffer's range check covers, plus a scalar
    K-block offset, which it does not: a range wider than the tensor would let the rows past a ragged
    N read up to a weight row's length past the caller's bytes."""
    launches = child("weight_ranges")
    kinds = {name.split("kernel")[0] for *_, name, _ in launches}
    assert len(launches) == 2 * len(Q4_SHAPES) and len(kinds) == 4
    for m, k, n, name, used in launches:
        rows = 2 * 1088 if "ILb1E" in name else n
        assert used == -(-rows // 32) * 32 * (k // 32) * 20, (m, k, n, name)


if __name__ == "__main__":
    print(json.dumps(CASES[sys.argv[1]]()))
