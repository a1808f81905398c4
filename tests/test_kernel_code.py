"""Properties of the compiled kernels that their sources rely on and that no
result shows, read from the gfx950 assembly of this repository's sources."""
import os
import re
import subprocess

import pytest

from vcp_amd import build as vb

pytestmark = pytest.mark.skipif(not os.path.exists(vb.HIPCC), reason="needs hipcc")


def _assembly(source, tmp_path):
    out = str(tmp_path / "k.s")
    flags = [f for f in vb.FLAGS if f != "-shared"]
    subprocess.run([vb.HIPCC, "-w", "-I", vb.CSRC] + flags + ["--cuda-device-only", "-S", source, "-o", out], check=True,
                   capture_output=True)
    with open(out) as f:
        return f.read()


def test_galerkin_stage_loads_are_global(tmp_path):
    # a FLAT load counts as an LDS operation as well, so the arithmetic that a
    # stage's loads are issued ahead of would wait for them
    s = _assembly(os.path.join(vb.CSRC, "kern_galerkin.hip"), tmp_path)
    assert "global_load_dwordx4" in s and "flat_load" not in s
    assert set(re.findall(r"; ScratchSize: (\d+)", s)) == {"0"}
