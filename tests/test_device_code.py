"""What the compiler cannot check in the device code (CPU: hipcc cross-compiles)."""

import re
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent / "pplx-garden_amd"
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"

# A 16-byte store that the compiler knows of, and a write of its data registers right behind it.
STORE_THEN_WRITE = """
#include <hip/hip_runtime.h>
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
extern "C" __global__ void known(u32x4 *p) {
    u32x4 v;
    asm volatile("; data %0" : "=v"(v));
    *p = v;
    v[0] = 0;
    asm volatile("; again %0" :: "v"(v));
}
"""


def _wait_states(text):
    return sum(int(n) + 1 for n in re.findall(r"s_nop (\d+)", text))


@pytest.mark.skipif(not Path(HIPCC).exists(), reason="needs hipcc")
def test_stores_in_inline_assembly_carry_the_wait_states_the_compiler_inserts(tmp_path):
    source = tmp_path / "known.hip"
    source.write_text(STORE_THEN_WRITE)
    assembly = subprocess.run([HIPCC, "-O3", "--offload-arch=gfx950", "-S", "--offload-device-only", str(source), "-o", "-"],
                              check=True, capture_output=True, text=True).stdout
    between = assembly[assembly.index("global_store_dwordx4"):]
    needed = _wait_states(between[:between.index("v_mov_b32")])
    assert needed > 0
    stores = [(path.name, asm) for path in sorted([*ROOT.glob("csrc/a2a_*"), *ROOT.glob("examples/*")]) for asm in
              re.findall(r'asm volatile\("([^;]*?store_dwordx[34][^:]*?)"\s*:', path.read_text())]
    assert {name for name, _ in stores} == {"a2a_device.h", "ceilings.hip"}
    for name, asm in stores:
        assert _wait_states(asm.split("store_dwordx")[1]) >= needed, (name, asm)


def test_kernels_of_short_arguments_take_no_hidden_ones():
    # blockDim and gridDim are arguments too, which the compiler adds: the launch would be a long one
    text = "\n".join((ROOT / "csrc" / name).read_text() for name in ("a2a_staged.hip", "a2a_combine.hip"))
    short = {"SendQuickArgs", "RecvRowsArgs", "CombineSendArgs", "CombineStagedArgs", "CombineSoleArgs"}
    found = set()
    for kind, body in re.findall(r"\((?:const )?(\w+)(?: &| )args[^)]*\) \{\n(.*?)^\}", text, re.M | re.S):
        if kind in short:
            found.add(kind)
            assert not re.search(r"\b(blockDim|gridDim)\b", body), kind
    assert found == short


@pytest.mark.skipif(not Path(HIPCC).exists(), reason="needs hipcc")
@pytest.mark.parametrize("limit,largest,refused", [("EXPERTS", 1984, None), ("EXPERTS", 2048, "to_first_rows"),
                                                   ("WORLD_SIZE", 64, "distances"), ("EXPERTS_PER_TOKEN", 128, "sizes")])
def test_limits_that_packed_words_do_not_hold_are_refused(tmp_path, limit, largest, refused):
    """The kernels of short arguments get sizes and distances in a few bits each: a larger limit has to end the build."""
    header = (ROOT.parent / "include" / "a2a.h").read_text()
    changed, count = re.subn(rf"(#define A2A_MAX_{limit}) \d+", rf"\1 {largest}", header)
    assert count == 1
    (tmp_path / "a2a.h").write_text(changed)
    source = tmp_path / "limits.hip"
    source.write_text('#include "a2a_staged.h"\n')
    cmd = [HIPCC, "--offload-arch=gfx950", "-std=c++17", "-fsyntax-only", "-I", str(tmp_path), "-I", str(ROOT / "csrc"), str(source)]
    result = subprocess.run(cmd, capture_output=True, text=True)
    assert (result.returncode == 0) == (refused is None), result.stderr
    assert refused is None or refused in result.stderr
