"""Compiled resources of the depth-first kernels (CPU: hipcc cross-compiles gfx950 here): both are bound by the
latency of dependent loads, so the waves that are resident matter.  Their LDS stacks allow three waves
per SIMD at eight query vertices and more for smaller queries."""
import os
import shutil
import subprocess

import pytest

import util
from test_kernel_resources import HIPCC, library_hipflags, resource_report

# kernel (a fragment of its mangled name) -> minimum waves per SIMD by registers
EXPECT = {
    "k_extendILi0E": 4,
    "k_extendILi1E": 4,
    "k_direct_searchILb1E": 5,
    "k_direct_searchILb0E": 5,
}


@pytest.mark.skipif(not (os.path.exists(HIPCC) or shutil.which("hipcc")), reason="hipcc not installed")
def test_depth_first_kernels_keep_their_occupancy(tmp_path):
    cmd = [HIPCC] + [f for f in library_hipflags() if f != "-Wall"]
    cmd += ["--cuda-device-only", "-c", os.path.join(util.PKG, "csrc", "device", "enum.hip"), "-o", str(tmp_path / "enum.o"),
            "-Rpass-analysis=kernel-resource-usage"]
    r = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=600)
    assert r.returncode == 0, r.stdout[-2000:]
    report = resource_report(r.stdout)
    for frag, waves in EXPECT.items():
        hits = [x for name, x in report.items() if frag in name]
        assert len(hits) == 1, (frag, sorted(report))
        assert hits[0]["Occupancy"] >= waves, (frag, hits[0])
        assert hits[0]["ScratchSize"] == 0 and hits[0].get("VGPRs Spill", 0) == 0, (frag, hits[0])
