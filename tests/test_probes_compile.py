"""The stand-alone probes under bench/ include the library's kernels and call them with all their parameters: a parameter more or less has
them no longer compile, which nothing else would show."""
import glob
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
PROBES = sorted(os.path.relpath(p, ROOT) for p in glob.glob(os.path.join(ROOT, "bench", "**", "*.hip"), recursive=True))


@pytest.mark.skipif(shutil.which(HIPCC) is None, reason="needs hipcc")
@pytest.mark.parametrize("path", PROBES)
def test_probe_compiles(path):
    cmd = [HIPCC, "--offload-arch=gfx950", "--cuda-host-only", "-fsyntax-only", "-std=c++17", "-Illmss_amd/csrc", path]
    r = subprocess.run(cmd, cwd=ROOT, capture_output=True, text=True)
    assert r.returncode == 0, "\n".join(x for x in r.stderr.splitlines() if "error:" in x)
