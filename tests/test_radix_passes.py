"""Passes of the hand-over's sort by element: one per 8 bits of the largest key,
nElems itself, and at most four, also for the largest element counts."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def passes(tmp_path_factory):
    d = tmp_path_factory.mktemp("radix")
    src = d / "passes.cpp"
    src.write_text("#include <cstdio>\n#include <cstdlib>\n#include \"stage_internal.h\"\n"
                   "int main(int, char **a) { std::printf(\"%d\\n\", pic::radix_passes(std::atoi(a[1]))); }\n")
    exe = d / "passes"
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-fsanitize=undefined", "-fno-sanitize-recover",
                           "-I", os.path.join(ROOT, "piclas_amd", "csrc"), "-I", os.path.join(ROOT, "include"),
                           str(src), "-o", str(exe)])
    return lambda ne: int(subprocess.run([str(exe), str(ne)], check=True, timeout=20, capture_output=True).stdout)


@pytest.mark.parametrize("ne,want", [(1, 1), (255, 1), (256, 2), (65535, 2), (65536, 3), (2**24 - 1, 3), (2**24, 4),
                                     (2**24 + 1, 4), (2**31 - 1, 4)])
def test_radix_passes(passes, ne, want):
    assert passes(ne) == want
