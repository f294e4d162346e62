"""How much memory the voxel medium's adjoint takes for its cells (no GPU: the rule alone)."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "cupbr_amd", "csrc")
GIB = 1 << 30


@pytest.fixture(scope="module")
def copies(tmp_path_factory):
    d = tmp_path_factory.mktemp("cells")
    src, exe = d / "copies.cpp", d / "copies"
    src.write_text('#include <cstdio>\n#include <cstdlib>\n#include "grid_cells.h"\n'
                   "int main(int, char** a) {\n"
                   '    std::printf("%u", cupbr::cell_copies(std::strtoull(a[1], 0, 10), std::strtoull(a[2], 0, 10),\n'
                   "                                         std::strtoull(a[3], 0, 10)));\n}\n")
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Wextra", "-Werror", f"-I{CSRC}", str(src), "-o", str(exe)], check=True)
    return lambda *args: int(subprocess.run([str(exe), *map(str, args)], check=True, capture_output=True, text=True).stdout)


def _bytes(n):
    return 32 * (n + 1) ** 3


@pytest.mark.parametrize("n,held,free,want", [
    (64, 0, 250 * GIB, 8),
    (256, 0, 250 * GIB, 8),
    (350, 0, 250 * GIB, 4),                # 8 GiB in all
    (511, 0, 250 * GIB, 2),
    (512, 0, 250 * GIB, 1),
    (700, 0, 250 * GIB, 0),
    (256, 0, 16 * GIB, 4),                 # a quarter of what is free: one copy is 0.51 GiB
    (256, 0, 2 * GIB, 0),
    (64, 0, 64 << 20, 1),
    (256, 8 * _bytes(256), 0, 8),          # held already
    (256, 2 * _bytes(256), 0, 2),
    (256, 2 * _bytes(256), 16 * GIB, 8),   # room again
])
def test_copies_fit_the_free_memory(copies, n, held, free, want):
    assert copies(_bytes(n), held, free) == want
