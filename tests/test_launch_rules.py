"""The launchers' rules on sizes (csrc/a2a_rules.h), compiled as plain C++ and called on the CPU."""

import ctypes
import shutil
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parent.parent / "pplx-garden_amd" / "csrc"

SOURCE = """
#include "a2a_rules.h"
extern "C" {
uint32_t layers(uint32_t tokens) { return a2a::token_layers(tokens).layers; }
uint32_t layer_rows(uint32_t tokens) { return a2a::token_layers(tokens).rows; }
}
"""


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    compiler = shutil.which("g++") or shutil.which("c++")
    if compiler is None:
        pytest.skip("needs a C++ compiler")
    folder = tmp_path_factory.mktemp("rules")
    (folder / "rules.cpp").write_text(SOURCE)
    subprocess.run([compiler, "-std=c++17", "-Wall", "-Wextra", "-Werror", "-shared", "-fPIC", "-I", str(CSRC),
                    str(folder / "rules.cpp"), "-o", str(folder / "rules.so")], check=True)
    return ctypes.CDLL(str(folder / "rules.so"))


@pytest.mark.parametrize("tokens", [1, 7, 32767, 32768, 32769, 33000, 65536, 65537, 100001, 1048577, 2147483647])
def test_the_gathers_grid_has_every_token_and_next_to_no_empty_rows(rules, tokens):
    layers, rows = rules.layers(tokens), rules.layer_rows(tokens)
    assert layers * rows >= tokens and rows <= 32768 and layers <= 65536
    assert layers * rows - tokens < layers
    assert layers == -(-tokens // 32768)
