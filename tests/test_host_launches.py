"""What the host entry points launch, on the CPU: the library runs over a stand-in for the HIP runtime
(fake_hip.cc, preloaded into a child process), whose launches only call a hook here."""
import ctypes
import json
import os
import re
import shutil
import subprocess
import sys
import threading

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


def tile_heights():
    """[(m, k, n, swiglu, rows of the kernel's output tile)] of projections to wide outputs."""
    h, out = Launches(), []
    for m in (1, 33, 64, 65, 100, 128, 129, 256, 257, 300, 384, 385, 500):
        for k in (1024, 2048, 3072, 4096):
            for n in (33024, 70016, 151680):
                for swiglu in (False, True):
                    def on(name, grid, block, args):
                        kind, first = re.match(r"_ZN5qattn\d+q4_(\w+?)_kernelILb[01]EL[ib](\d+)E", name).groups()
                        rows = {"tile": 32 * int(first), "mid": 64, "small": 16 * int(first), "direct": 32}[kind]
                        out.append((m, k, n, swiglu, rows))
                    h.on = on
                    need = h.qattn.lib().qattn_q4_compact_bytes(k, n)
                    if swiglu:
                        h.ctx.q4_matmul_swiglu(1 << 20, m, k, 1 << 30, need, n // 2, 1 << 40)
                    else:
                        h.ctx.q4_matmul(1 << 20, m, k, 1 << 30, need, n, 1 << 40)
    return out


def k_blocks():
    """[(m, k, K blocks that the kernel computes)] of projections whose K is no multiple of 1,024."""
    h, out = Launches(), []
    for m in (1419, 3000, 8000, 20000):
        for k in (32, 64, 128, 256, 1056, 1280, 1536, 2080, 2560):
            def on(name, grid, block, args):
                kind, ints, fold = re.match(r"_ZN5qattn\d+q4_(\w+?)_kernelILb0E((?:Li\d+E)+)Lb([01])E", name).groups()
                groups, step = int(re.findall(r"\d+", ints)[-1]), 8 if kind == "mid" else 4
                out.append((m, k, grid, groups * 32 if groups > 1 else -(-(k // 32) // step) * step))
            h.on = on
            h.ctx.q4_matmul(1 << 20, m, k, 1 << 30, h.qattn.lib().qattn_q4_compact_bytes(k, 1024), 1024, 1 << 40)
    return out


def kernel_coverage():
    """The Q4_0 GEMM kernels of the library, and those that the bit-equality cases of test_gpu_q4.py launch
    (the whole launch and the small one it is compared with) and its strided cases:
    [[all], [[case, kernel, reference]], [strided]]."""
    import test_gpu_q4 as cases
    h, kernels, out, seen = Launches(), [], [], []
    each = ctypes.CFUNCTYPE(None, ctypes.c_char_p)(lambda name: kernels.append(name.decode()))
    h.fake.fake_hip_kernels(each)
    h.on = lambda name, *rest: seen.append(name)

    def launch(m, k, n, swiglu):
        need = h.qattn.lib().qattn_q4_compact_bytes(k, n)
        if swiglu:
            h.ctx.q4_matmul_swiglu(1 << 20, m, k, 1 << 30, need, n // 2, 1 << 40)
        else:
            h.ctx.q4_matmul(1 << 20, m, k, 1 << 30, need, n, 1 << 40, ldy=-(-n // 8) * 8)
        return seen[-1]

    for m, k, n, swiglu in cases.TILE_CASES + cases.TALL_CASES:
        out.append(((m, k, n, swiglu), launch(m, k, n, swiglu), launch(min(m, 32), k, n, swiglu)))
    for m, k, n_inter in ((40, 4096, 192),):  # test_q4_long_k_swiglu_equals_the_two_launches
        out.append(((m, k, 2 * n_inter, True), "", launch(m, k, 2 * n_inter, True)))
    strided = [launch(m, k, n, False) for m, k, n in cases.STRIDED_CASES]
    for m, k, n, swiglu in cases.WIDE_CASES:
        out.append(((m, k, n, swiglu), launch(m, k, n, swiglu), launch(m, k, 128, swiglu)))
    return [[k for k in kernels if re.search(r"q4_(tile|mid|direct|small)_kernel", k)], out, strided]


def attention_variants():
    """{lengths: {launch: [split, one entry]}}, from the kernel's template arguments."""
    h, out = Launches(), {}
    for lengths, flags in (([50], 1), ([10, 150, 64], 1), ([500] * 16, 0), ([5000], 0)):
        names = []
        h.on = lambda name, *rest: names.append(re.match(r"_ZN5qattn15attn_fwd_kernelI((?:Lb[01]E)+)E", name))
        run = h.ctx.run(h.qattn.make_desc(1 << 20, 1 << 30, 1 << 31, 1 << 32, np.cumsum([0] + lengths), flags=flags))
        seen = {}
        for launch in (run.encode, run.mask_bits, run.timeline):
            names.clear()
            launch()
            bools = [m for m in names if m][0].group(1)
            seen[launch.__name__] = [bools[2] == "1", bools[18] == "1"]
        run.destroy()
        out[",".join(map(str, lengths))] = seen
    return out


def _model(h, layers):
    compact = lambda k, n: (1 << 30, h.qattn.lib().qattn_q4_compact_bytes(k, n))  # noqa: E731
    layer = {"attn_qkv": compact(1024, 4096), "attn_output": compact(2048, 1024), "ffn_gate_up": compact(1024, 6144),
             "ffn_down": compact(3072, 1024)}
    layer.update({n: 1 << 20 for n in ("attn_norm", "attn_q_norm", "attn_k_norm", "ffn_norm")})
    return h.ctx.model((1 << 24, 840 * 1000), 1 << 20, [layer] * layers)


def fused_routes():
    """[(tokens, sequences, whether the forward takes the fused projections)]."""
    h, out, names = Launches(), [], []
    plan = _model(h, 1).plan(64, 70)
    h.on = lambda name, *rest: names.append(name)
    for tokens, nseq in ((1, 1), (32, 1), (33, 1), (32, 64), (32, 65), (31, 70)):
        cu = np.minimum(np.arange(nseq + 1), tokens).astype(np.int32)
        cu[-1] = tokens
        names.clear()
        plan.run(np.zeros(tokens, np.int32), cu, 1 << 22)
        out.append((tokens, nseq, any("q4_fused" in n for n in names)))
    return out


def rope_table_lifetime():
    """{call: [the table that a launch was passed was freed before the launch returned]} while another
    thread grows the context's table in the middle of each launch that reads it."""
    out = {}
    for call in ("fused forward", "forward", "qkv", "in place"):
        h = Launches()
        freed, threads, longest = [], [], [1100]
        main = threading.get_ident()

        def grow():
            longest[0] += 100
            h.ctx.qk_norm_rope(1 << 20, 512, 0, 4, np.array([0, longest[0]], np.int32))

        def on(name, grid, block, args):
            # FusedQkv (q, k, qkv, weight_q, weight_k, rope) or RopeArgs (in, out_q, out_k, weight_q, weight_k, rope)
            index = 7 if "q4_fused_kernelILb1" in name else 0 if "qk_norm_rope" in name else None
            if index is None or threading.get_ident() != main:
                return
            table = h.word(args, index, ctypes.c_uint64, 40)
            threads.append(threading.Thread(target=grow))
            threads[-1].start()
            threads[-1].join(0.2)  # the other thread may have to wait for this launch
            freed.append(bool(h.fake.fake_hip_freed(table)))

        h.ctx.qk_norm_rope(1 << 20, 512, 0, 4, np.array([0, 1050], np.int32))
        tokens = 20 if call == "fused forward" else 40
        cu = np.array([0, tokens], np.int32)
        plan = _model(h, 3).plan(64, 4) if "forward" in call else None
        h.on = on
        if plan:
            plan.run(np.zeros(tokens, np.int32), cu, 1 << 22)
        elif call == "qkv":
            h.ctx.qk_norm_rope_qkv(1 << 20, 1 << 21, 1 << 22, cu)
        else:
            h.ctx.qk_norm_rope(1 << 20, 512, 0, 4, cu)
        for t in threads:
            t.join()
        out[call] = freed
    return out


CASES = {f.__name__: f for f in (weight_ranges, tile_heights, k_blocks, kernel_coverage, attention_variants, fused_routes,
                                rope_table_lifetime)}


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


def test_wide_projections_of_few_rows_take_short_tiles(child):
    """However many tiles a wide weight makes, a launch of a few rows does not pay for tiles much taller
    than them."""
    launches = child("tile_heights")
    assert len(launches) == 13 * 4 * 3 * 2
    for m, k, n, swiglu, rows in launches:
        assert rows <= (64 if m <= 64 else 128 if m <= 128 or (256 < m <= 384 and k <= 1024) else 256), (m, k, n, rows)


def test_launches_that_fill_the_chip_do_not_pad_k(child):
    """Groups that each run a chunk of K, and kernels that step by eight K blocks, compute blocks past K: no
    launch of more than one workgroup per CU computes a third more than it has (or four blocks)."""
    launches = child("k_blocks")
    assert len(launches) == 4 * 9
    for m, k, grid, blocks in launches:
        assert grid <= 256 or blocks <= max(4, 4 * (k // 32) // 3), (m, k, grid, blocks)
        assert k < 1024 or blocks <= 4 * (k // 32) / 3, (m, k, grid, blocks)


def test_every_projection_kernel_is_compared_with_another(child):
    """The library holds no GEMM kernel that nothing launches, and the GPU tests compare each with another
    kernel's rows, bit for bit (or are that other kernel, which the oracle checks)."""
    kernels, cases, strided = child("kernel_coverage")
    reached = {whole for _, whole, other in cases if whole != other} | {other for *_, other in cases}
    assert len(kernels) > 20 and sorted(set(kernels) - reached) == []
    assert sorted({k for k in kernels if "ILb0E" in k} - set(strided)) == []


def test_mask_check_and_timeline_run_the_variant_that_a_launch_runs(child):
    """The executed mask and the phase stamps are those of the kernel that the run's launches take."""
    seen = child("attention_variants")
    assert {tuple(v["encode"]) for v in seen.values()} == {(False, True), (False, False), (True, False)}
    for lengths, v in seen.items():
        assert v["mask_bits"] == v["encode"] and v["timeline"] == v["encode"], (lengths, v)


def test_fused_forward_limits(child):
    for tokens, nseq, fused in child("fused_routes"):
        assert fused == (tokens <= 32 and nseq <= 64), (tokens, nseq)


def test_rope_table_outlives_the_launches_that_read_it(child):
    """One context serves several threads.  A call that needs a longer RoPE table frees the old one, which
    waits for the launches already enqueued only: no launch may be passed a table that is freed before
    the launch is enqueued, in a forward of several layers neither."""
    freed = child("rope_table_lifetime")
    assert [len(freed[c]) for c in ("fused forward", "forward", "qkv", "in place")] == [3, 3, 1, 1]
    assert not any(sum(freed.values(), [])), freed


if __name__ == "__main__":
    print(json.dumps(CASES[sys.argv[1]]()))
