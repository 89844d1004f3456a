"""The hand-counted waits of the Q4_0 GEMM kernels, followed through the gfx950 assembly on the CPU.

q4_tile_kernel and q4_mid_kernel load X tiles by LDS-DMA several steps ahead and publish them with
q4_barrier<V>: wait until at most the V newest vector-memory operations are in flight, then meet the
workgroup.  Every wavefront reads rows that others loaded, so by barrier b every load of the b-th X
tile must have landed on the strength of those explicit waits alone: the compiler's own waits, which
follow its schedule of the weight registers, do not count here.
"""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SOURCE = os.path.join(ROOT, "qwen3-embedding-webgpu-prepacked_amd", "csrc", "q4_matmul.hip")
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
PASSES = 4  # of the loop: the first ones are the prologue's, then the steady state


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    if not os.path.exists(HIPCC):
        pytest.skip("no hipcc")
    out = str(tmp_path_factory.mktemp("asm") / "q4.s")
    subprocess.run([HIPCC, "--offload-arch=gfx950", "-O3", "-std=c++17", "-Xclang", "-target-feature", "-Xclang",
                    "-packed-fp32-ops", "--cuda-device-only", "-S", "-o", out, SOURCE], check=True, capture_output=True)
    found = {}
    name = None
    for line in open(out):
        start = re.match(r"(_ZN5qattn\d+q4_(?:mid|tile)_kernel\w+):", line)
        if start:
            name = start.group(1)
            found[name] = []
        elif line.startswith(".Lfunc_end"):
            name = None
        elif name:
            found[name].append(line.split(";")[0].strip() if "#ASM" not in line else line.strip())
    return found


def tile_loads(name):
    """LDS-DMA loads of one X tile per wavefront, by the kernel's template arguments."""
    ints = [int(v) for v in re.findall(r"Li(\d+)E", name)]
    return 2 if "q4_mid" in name else ints[0] // ints[1]  # MF / NWN; mid: two K blocks


def events(lines):
    """"load", "dma" and explicit ("wait", V) events of the prologue and of the main loop: the first loop
    that issues LDS-DMA loads."""
    flat, labels, ends = [], {}, []
    asm = False
    for line in lines:
        if "#ASMSTART" in line or "#ASMEND" in line:
            asm = "#ASMSTART" in line
            continue
        label = re.match(r"(\.LBB\w+):", line)
        if label:
            labels[label.group(1)] = len(flat)
        elif re.match(r"(buffer|global|flat|scratch)_", line):
            flat.append(("dma",) if line.endswith(" lds") else ("load",))
        elif asm and "vmcnt(" in line:
            flat.append(("wait", int(re.search(r"vmcnt\((\d+)\)", line).group(1))))
        branch = re.match(r"s_c?branch\w*\s+(\.LBB\w+)", line)
        if branch and branch.group(1) in labels and ("dma",) in flat[labels[branch.group(1)]:]:
            ends.append((labels[branch.group(1)], len(flat)))
    assert ends, "no loop with LDS-DMA loads"
    first, last = ends[0]
    return flat[:first], flat[first:last]


def test_every_published_x_tile_has_landed(kernels):
    assert len([k for k in kernels if "q4_mid" in k]) >= 4 and len([k for k in kernels if "q4_tile" in k]) >= 8
    for name, lines in kernels.items():
        prologue, loop = events(lines)
        assert sum(e[0] == "wait" for e in prologue) == 1 and sum(e[0] == "wait" for e in loop) == 4, name
        group = tile_loads(name)
        issued, dma, barrier = 0, [], 0  # dma: issue numbers of the LDS-DMA loads
        for event in prologue + PASSES * loop:
            if event[0] == "wait":
                last = dma[group * (barrier + 1) - 1]
                newer = issued - 1 - last
                assert newer >= event[1], (
                    f"{name}: barrier {barrier} waits with vmcnt({event[1]}), but only {newer} operations are newer "
                    f"than the X tile it publishes")
                barrier += 1
            else:
                if event[0] == "dma":
                    dma.append(issued)
                issued += 1
