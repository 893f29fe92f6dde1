"""Registers of kernels whose waves have to share a SIMD, as the compiler reports them."""
import re
import subprocess

from llmss_amd import _build


def test_attention_behind_prefixes_two_waves_a_simd(tmp_path):
    r = subprocess.run([_build.HIPCC, *_build._flags(), *_build._includes(), "--offload-device-only", "-Rpass-analysis=kernel-resource-usage", "-x", "hip",
                        "-c", _build.CSRC + "/attention_extend.hip", "-o", str(tmp_path / "o")], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    found = re.findall(r"Function Name: \S*attn_extend_kernelILi(\d+)E.*?Occupancy \[waves/SIMD\]: (\d+).*?VGPRs Spill: (\d+)", r.stderr, re.S)
    assert sorted({int(d) for d, _, _ in found}) == [64, 128, 256]
    for _, waves, spilled in found:
        assert int(waves) >= 2 and int(spilled) == 0
