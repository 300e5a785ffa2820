"""No reconstruction kernel spills registers to memory.

Every four-lane instantiation is compiled for its waves per SIMD (ReconQWaves);
the compiler's resource remarks say what each takes.
"""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_reconstruction_has_no_spills(tmp_path):
    from afar_cudaeuler2dmixo3rk3solver_amd import build as b
    if shutil.which(b.HIPCC) is None:
        pytest.skip("hipcc not available")
    cmd = [b.HIPCC] + b.COMMON + b.DEVICE + ["-I", b.CSRC, "-I", os.path.join(ROOT, "include"), "-x", "hip",
                                             "--offload-device-only", "-Rpass-analysis=kernel-resource-usage", "-c",
                                             os.path.join(b.CSRC, "kernels.hip"), "-o", str(tmp_path / "k.o")]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]
    spills, name = {}, None
    for line in r.stderr.splitlines():
        m = re.search(r"Function Name: (\S+)", line)
        if m:
            name = m.group(1)
        m = re.search(r"(?:VGPRs Spill|ScratchSize \[bytes/lane\]): (\d+)", line)
        if m and name and "k_reconstruct" in name:
            spills[name] = spills.get(name, 0) + int(m.group(1))
    assert len([n for n in spills if "k_reconstruct_q" in n]) == 36  # types, tiles, flux points or not, stencil sizes
    assert not {n: s for n, s in spills.items() if s}
