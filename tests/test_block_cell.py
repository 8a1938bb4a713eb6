"""The cell of a position within its block: 64-bit also where the block's cells do
not fit 32 bits (a lattice of such a block takes tens of GB on the host, so the
index is checked by itself)."""
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]
SRC = r"""
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include "hemepure_amd/csrc/lattice.h"
int main(int, char** v) {
  const int32_t x = std::atoi(v[1]), y = std::atoi(v[2]), z = std::atoi(v[3]), bs = std::atoi(v[4]);
  std::printf("%lld\n", (long long)hlb::cell_in_block(x, y, z, bs));
}
"""


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    d = tmp_path_factory.mktemp("cell")
    (d / "cell.cpp").write_text(SRC)
    subprocess.run(["g++", "-std=c++17", "-Wall", f"-I{ROOT}", str(d / "cell.cpp"), "-o", str(d / "cell")], check=True)
    return d / "cell"


@pytest.mark.parametrize("bs", [1, 6, 8, 1290, 1291, 4000])
def test_cell_in_block(exe, bs):
    for x, y, z in ((0, 0, 0), (bs - 1, bs - 1, bs - 1), (bs, 2 * bs + bs // 2, bs - 1)):
        out = subprocess.run([str(exe), *map(str, (x, y, z, bs))], capture_output=True, text=True, check=True)
        assert int(out.stdout) == ((x % bs) * bs + y % bs) * bs + z % bs
