"""The order and number of the tile GEMM's vector memory loads on gfx950, pinned at build time.

matmul_tile_kernel waits for a chunk of x by the count of the loads issued after it (kLater in
gsp_matmul.hip): the direct loads of two later chunks and the weight and block-sum fetches of three.
That is sound only if every chunk issues its direct loads (to LDS) before its fetches, and if the
compiler neither drops nor merges a fetch.  This test reads the library's own gfx950 assembly.
"""
import re
import shutil
import subprocess
import sys
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent
sys.path.insert(0, str(ROOT / "glacier.serve_amd"))

# GGUF weight type -> (fetched loads per unit, units per four chunks, loads of block sums per M tile)
KERNELS = {0: (8, 4, 0), 8: (10, 2, 0), 12: (6, 1, 1), 14: (10, 1, 0)}


@pytest.fixture(scope="module")
def assembly(tmp_path_factory):
    import build

    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not Path(hipcc).exists():
        pytest.skip("hipcc is not installed")
    out = tmp_path_factory.mktemp("asm") / "matmul.s"
    cmd = [hipcc, f"--offload-arch={build.ARCH}", "-O3", "-std=c++17", "-fPIC", f"-I{ROOT / 'include'}",
           *build.DEVICE_FLAGS, "-x", "hip", "--cuda-device-only", "-S",
           str(ROOT / "glacier.serve_amd" / "csrc" / "gsp_matmul.hip"), "-o", str(out)]
    res = subprocess.run(cmd, capture_output=True, text=True)
    assert res.returncode == 0, res.stderr
    return out.read_text()


def _blocks(body: str):
    """Basic blocks, cut at barriers too."""
    cur = []
    for ln in body.splitlines():
        ln = ln.split(";")[0].strip()
        if ln.endswith(":"):
            yield cur
            cur = []
        elif ln and not ln.startswith("."):
            cur.append(ln)
            if ln.startswith(("s_cbranch", "s_branch", "s_barrier", "s_endpgm")):
                yield cur
                cur = []
    yield cur


@pytest.mark.parametrize("w_type", sorted(KERNELS))
def test_direct_loads_come_before_the_chunks_fetches(assembly, w_type):
    unit_loads, units, sums = KERNELS[w_type]
    m = re.search(rf"^(\S*18matmul_tile_kernelILi{w_type}E\S*):\s.*?s_endpgm", assembly, re.S | re.M)
    assert m, "kernel not found"
    found = {1: 0, 2: 0, 4: 0}  # direct loads of a wave and chunk: its M tiles
    for block in _blocks(m.group(0)):
        direct = [i for i, ln in enumerate(block) if re.match(r"buffer_load\S* .*\blds\b", ln)]
        fetch = [i for i, ln in enumerate(block) if re.match(r"(buffer|global|flat)_load", ln) and i not in direct]
        if len(direct) not in found or not fetch:
            continue  # the prologue stages three chunks behind a wait for everything
        assert max(direct) < min(fetch), block
        assert len(fetch) == unit_loads + sums * len(direct), (len(fetch), block)
        found[len(direct)] += 1
    assert found == {1: units, 2: units, 4: units}, found
