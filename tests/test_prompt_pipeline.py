"""The load pipeline of the MXFP4 prompt GEMM in the code the compiler makes of it (CPU
only: it compiles lb_prompt.hip to gfx950 assembly), and the prompt GEMMs' tile map.

The kernel waits for a stage by count: "all of this wave's loads but the last OPS have
arrived". That holds only if the loads of an earlier group are issued before every load of
a later one, which the scheduler does not know. The loop's order is pinned slot by slot;
the two groups loaded ahead of it must be apart too.
"""
import re
import shutil
import subprocess
from pathlib import Path

import pytest

from lowbit_amd import _build

ROOT = Path(__file__).resolve().parents[1]
KERNEL = "mxfp4_prompt_kernel"


def _hipcc():
    p = Path("/opt/rocm/bin/hipcc")
    return str(p) if p.exists() else shutil.which("hipcc")


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """The kernel's instantiations, each as its instructions (the entry block first)."""
    cc = _hipcc()
    if cc is None:
        pytest.skip("hipcc not available")
    out = tmp_path_factory.mktemp("asm") / "lb_prompt.s"
    flags = [f for f in _build.FLAGS if f != "-shared"]
    subprocess.run([cc, "--offload-arch=gfx950", *flags, f"-I{_build.INCLUDE}", "--offload-device-only", "-S",
                    str(_build.CSRC / "lb_prompt.hip"), "-o", str(out)], check=True, capture_output=True, text=True)
    found, name = {}, None
    for line in out.read_text().splitlines():
        m = re.match(r"(_Z\w+):", line)
        if m:
            name = m.group(1)
        elif line.startswith("\t.section") or line.startswith("\t.p2align"):
            name = None
        elif name and KERNEL in name:
            found.setdefault(name, []).append(line.split(";")[0].strip())
    assert len(found) == 2, list(found)
    return found


def test_groups_loaded_ahead_are_apart(kernels):
    """Before the loop: the loads to LDS of group 0, its weights', then those of group 1."""
    for name, code in kernels.items():
        kinds = []
        for ins in code[:next(i for i, s in enumerate(code) if s.startswith("s_barrier"))]:
            if ins.startswith("buffer_load"):
                kinds.append("lds" if ins.endswith("lds") else "weights")
        runs = [k for i, k in enumerate(kinds) if i == 0 or kinds[i - 1] != k]
        assert runs == ["lds", "weights", "lds", "weights"], (name, runs)
        assert kinds[:len(kinds) // 2] == kinds[len(kinds) // 2:], (name, kinds)


def test_no_step_waits_for_the_loads_it_issued(kernels):
    """In the loop, a step's loads are for two groups on; what it waits for before its own
    first load must leave the previous step's in flight (some of them at least: it issues
    8 or more after the ones that the step's first products need)."""
    for name, code in kernels.items():
        bars = [i for i, s in enumerate(code) if s.startswith("s_barrier")][:3]
        for i in bars:  # the three steps of the loop
            first = next(j for j in range(i, len(code)) if code[j].startswith("buffer_load"))
            waits = [int(n) for s in code[i - 4:first] for n in re.findall(r"vmcnt\((\d+)\)", s)]
            assert waits and min(waits) >= 8, (name, waits)


def test_tile_map_covers_every_tile_once(tmp_path):
    """Grids whose surplus workgroups fall past the last band of rows included: those must
    be turned away before the band's row count (0) divides."""
    cc = _hipcc()
    if cc is None:
        pytest.skip("hipcc not available")
    exe = tmp_path / "prompt_tiles"
    subprocess.run([cc, "--offload-host-only", "-x", "hip", "-O2", "-std=c++17", f"-I{_build.CSRC}",
                    f"-I{_build.INCLUDE}", str(ROOT / "tests" / "csrc" / "prompt_tiles.hip"), "-o", str(exe)],
                   check=True, capture_output=True, text=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout == f"tiles {820 * 2485} bad 0\n", (r.returncode, r.stdout)
