"""CPU check of rswa_dispatch.hpp: which attention calls run query-tiled. The
cache's capacity alone must not make a short prompt one (it then runs slower than
row by row), rows of one cache count the keys that they see, and calls the tiled
kernel has no instance for stay off it."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "unlimited-ocr.cpp_amd", "csrc")
MAIN = r"""
#include "rswa_dispatch.hpp"
#include <cstdlib>
int main(int n, char** v) {
    const long long rows = atoll(v[1]);
    const int heads = atoi(v[2]), hd = atoi(v[3]), len = atoi(v[4]);
    return n == 5 ? uocr_hip::rswa_call_tiled(rows, heads, hd, len)
                  : uocr_hip::rswa_one_cache_tiled(rows, heads, hd, len, atoi(v[5]), atoi(v[6]) != 0);
}
"""


@pytest.fixture(scope="module")
def tiled(tmp_path_factory):
    d = tmp_path_factory.mktemp("rswa")
    (d / "m.cpp").write_text(MAIN)
    subprocess.run(["g++", "-std=c++17", "-I", CSRC, str(d / "m.cpp"), "-o", str(d / "m")], check=True)
    return lambda *a: bool(subprocess.run([d / "m", *map(str, a)]).returncode)


@pytest.mark.parametrize("rows,heads,head_dim,max_len,want", [
    (60, 10, 128, 60, False), (60, 10, 128, 1128, False), (76, 10, 128, 1128, False),  # capacity has no say
    (60, 10, 128, 0, False), (64, 10, 128, 1000, False),  # length unknown; a few rows over many keys
    (100, 10, 128, 1128, True), (100, 10, 128, 0, True), (1000, 10, 128, 1128, True), (300, 10, 128, 33, True),
    (52, 32, 128, 1128, True), (1000, 1, 128, 1128, False),  # many heads fill the chip, one does not
    (100, 8, 64, 1128, False), (200, 8, 64, 1128, True),
    (1000, 10, 96, 1128, False), (1000, 10, 256, 1128, False), (51, 10, 128, 1128, False),
    (2**31 - 1, 64, 128, 2**31 - 1, True),
])
def test_calls(tiled, rows, heads, head_dim, max_len, want):
    assert tiled(rows, heads, head_dim, max_len) is want


@pytest.mark.parametrize("rows,heads,head_dim,kv_len,q_start,causal,want", [
    (64, 10, 128, 964, 900, 1, False), (98, 10, 128, 314, 216, 1, True), (128, 10, 128, 1028, 900, 1, True),
    (52, 32, 128, 152, 100, 1, True), (52, 32, 128, 952, 900, 1, True),  # tiled 16.8 us, rows 26; 50 / 79
    (128, 12, 64, 344, 216, 1, True), (160, 8, 64, 376, 216, 1, True), (160, 8, 64, 1060, 900, 1, False), (200, 8, 64, 1100, 900, 1, True),
    (60, 10, 128, 60, 0, 1, False), (300, 10, 128, 33, 0, 0, True), (180, 10, 128, 60, -120, 1, True),
])
def test_one_cache(tiled, rows, heads, head_dim, kv_len, q_start, causal, want):
    assert tiled(rows, heads, head_dim, kv_len, q_start, causal) is want
