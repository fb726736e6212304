"""CPU check of the block -> item order of xcd_order.hpp: the shares of the 8 XCDs
cover every item once and are even, also where there are few items (a wide
one-tile GEMM, one expert), so no call runs on a part of the chip."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "unlimited-ocr.cpp_amd", "csrc")
MAIN = r"""
#define __host__
#define __device__
#include "xcd_order.hpp"
#include <cstdio>
#include <cstdlib>
int main(int, char** v) {
    for (int x = 0; x <= uocr_hip::kXcds; ++x) printf("%d ", uocr_hip::xcd_first_item(x, atoi(v[1])));
}
"""


@pytest.fixture(scope="module")
def first_items(tmp_path_factory):
    d = tmp_path_factory.mktemp("xcd")
    (d / "m.cpp").write_text(MAIN)
    subprocess.run(["g++", "-std=c++17", "-I", CSRC, str(d / "m.cpp"), "-o", str(d / "m")], check=True)
    return lambda n: [int(s) for s in subprocess.run([d / "m", str(n)], check=True, capture_output=True,
                                                     text=True).stdout.split()]


@pytest.mark.parametrize("n", [0, 1, 7, 8, 9, 14, 28, 60, 504, 2020, 17_000_000, 2**31 - 1])
def test_shares_are_even(first_items, n):
    b = first_items(n)
    assert b[0] == 0 and b[8] == n
    assert {e - s for s, e in zip(b, b[1:])} <= {n // 8, -(-n // 8)}
