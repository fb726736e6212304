"""CPU check of rswa_dispatch.hpp: which attention calls run query-tiled. The
cache's capacity alone must not make a short prompt one (it then runs slower than
row by row), and calls the tiled kernel has no instance for stay off it."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "unlimited-ocr.cpp_amd", "csrc")
MAIN = r"""
#include "rswa_dispatch.hpp"
#include <cstdlib>
int main(int, char** v) { return uocr_hip::rswa_call_tiled(atoll(v[1]), atoi(v[2]), atoi(v[3]), atoi(v[4])); }
"""


@pytest.fixture(scope="module")
def tiled(tmp_path_factory):
    d = tmp_path_factory.mktemp("rswa")
    (d / "m.cpp").write_text(MAIN)
    subprocess.run(["g++", "-std=c++17", "-I", CSRC, str(d / "m.cpp"), "-o", str(d / "m")], check=True)
    return lambda *a: bool(subprocess.run([d / "m", *map(str, a)]).returncode)


@pytest.mark.parametrize("rows,heads,head_dim,max_len,want", [
    (60, 10, 128, 60, False), (60, 10, 128, 1128, False), (97, 10, 128, 1128, False),  # capacity has no say
    (97, 10, 128, 0, False), (64, 10, 128, 1000, False),  # length unknown; a chunk of few rows over many keys
    (100, 10, 128, 1128, True), (100, 10, 128, 0, True), (1000, 10, 128, 1128, True), (300, 10, 128, 33, True),
    (100, 8, 64, 1128, False), (200, 8, 64, 1128, True),
    (1000, 10, 96, 1128, False), (1000, 10, 256, 1128, False), (51, 10, 128, 1128, False),
    (2**31 - 1, 64, 128, 2**31 - 1, True),
])
def test_calls(tiled, rows, heads, head_dim, max_len, want):
    assert tiled(rows, heads, head_dim, max_len) is want
