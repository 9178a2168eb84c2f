"""The words of a donated range (csrc/device/range_word.h), compiled for the CPU: a wave that takes a range may
have read the frame word of any other publication of its owner, and must then not use it."""
import os
import shutil
import subprocess

import pytest

import util

PROGRAM = r"""
#include "range_word.h"
#include <cstdio>
#include <vector>
using namespace csm;

int main() {
    struct Published { unsigned long long range, frame; uint32_t group, first; };
    std::vector<Published> p = {{0, 0, 0, 0}};  // both words as the launch clears them
    uint32_t version = 0;
    for (uint32_t k = 1; k <= 70000; k++) {
        version = next_version(version);
        if (version == 0 || version > 0xFFFF) return std::printf("version %u\n", version), 1;
        // groups over all 32 bits, first items and candidate ranges over theirs
        const uint32_t group = k * 2654435761u, first = k % 64, end = kRangeMask - k % 3, cur = k % end;
        p.push_back({range_word(version, cur, end), frame_word(version, group, first), group, first});
        const Published& x = p.back();
        if (range_cur(x.range) != cur || range_end(x.range) != end) return std::printf("range %u\n", k), 1;
        if (frame_group(x.frame) != group || frame_first(x.frame) != first) return std::printf("frame %u\n", k), 1;
    }
    // a range of publication a with the frame word of publication b: taken only if they are one publication
    for (uint32_t a = 0; a < p.size(); a += a < 300 ? 1 : 997)
        for (uint32_t b = 0; b < p.size(); b++) {
            const bool versions_came_round = a && b && (a > b ? a - b : b - a) % 0xFFFF == 0;
            if (same_publication(p[a].range, p[b].frame) != (a && (a == b || versions_came_round))) return std::printf("%u %u\n", a, b), 1;
            // the owner's and the thieves' steps keep the version
            const unsigned long long left = (p[a].range & ~static_cast<unsigned long long>(kRangeMask)) | 1u;
            if (same_publication(left, p[b].frame) != same_publication(p[a].range, p[b].frame)) return std::printf("step %u\n", a), 1;
        }
    std::puts("ok");
}
"""


@pytest.mark.skipif(not shutil.which("g++"), reason="g++ not installed")
def test_a_range_is_used_with_its_own_frame_only(tmp_path):
    (tmp_path / "words.cpp").write_text(PROGRAM)
    exe = tmp_path / "words"
    util.run(["g++", "-O1", "-std=c++17", "-I", os.path.join(util.PKG, "csrc", "device"), str(tmp_path / "words.cpp"), "-o", str(exe)])
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0 and r.stdout == "ok\n", r.stdout
