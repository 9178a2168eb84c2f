"""The launch setting dfs_blocks and the grid it stands for (csrc/device/dfs_grid.h), compiled for the CPU."""
import os
import re
import shutil

import pytest

import util

PROGRAM = r"""
#include "dfs_grid.h"
#include <cstdio>
#include <initializer_list>
using namespace csm;
int main() {
    for (uint32_t b = 1; b <= 2 * kMaxDfsBlocks; b *= 2)
        for (uint64_t items : {1ull, 2ull, 3ull, 1000ull, 1ull << 33})
            std::printf("%u %llu %u %u\n", b, static_cast<unsigned long long>(items), dfs_grid(b, items, false), dfs_grid(b, items, true));
    std::printf("limits %u %u %u %u\n", kMinDfsBlocks, kMaxDfsBlocks, kDfsBlocks, kDfsWaves);
}
"""


@pytest.mark.skipif(not shutil.which("g++"), reason="g++ not installed")
def test_every_value_of_the_setting_is_another_grid(tmp_path):
    (tmp_path / "grid.cpp").write_text(PROGRAM)
    exe = tmp_path / "grid"
    util.run(["g++", "-O1", "-std=c++17", "-I", os.path.join(util.PKG, "csrc", "device"), str(tmp_path / "grid.cpp"), "-o", str(exe)])
    rows = [line.split() for line in util.run([str(exe)]).splitlines()]
    low, high, default, waves = map(int, rows.pop()[1:])
    for blocks, items, grid, whole in (map(int, r) for r in rows):
        most = min(blocks, high)
        assert whole == most
        assert grid == min(most, -(-items // waves))
    # what the header states, and values for the autotuner that are in range and hold the default
    m = re.search(r"dfs_blocks;.*two waves each \((\d+)\.\.(\d+), default (\d+)\)", open(util.HEADER).read())
    assert [int(x) for x in m.groups()] == [low, high, default] and waves == 2
    tuned = re.search(r"kDfsBlockValues\[\] = \{([^}]*)\}", open(os.path.join(util.PKG, "csrc", "tune.cpp")).read()).group(1)
    tuned = [int(x) for x in tuned.split(",")]
    assert default in tuned and sorted(set(tuned)) == tuned and low <= tuned[0] and tuned[-1] <= high
