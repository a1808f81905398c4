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


def test_dpp_accumulators_share_no_factor_registers(tmp_path):
    # the DPP block writes accumulators before it has read its last factor; here
    # accumulators start with the factors' values, so that they could share
    src = tmp_path / "dpp.hip"
    src.write_text('''#include "vcphip_device.h"
#include "vcphip_dpp.h"
__global__ void k(const double* in, double* out) {
  const double x = in[threadIdx.x], y = in[64 + threadIdx.x];
  double up[8], dn[8], r1[8], r2[8];
  for (int i = 0; i < 8; ++i) {
    up[i] = x;
    dn[i] = y;
    r1[i] = r2[i] = 0.0;
  }
  vcphip_dpp_step<false, false>(x, 0.0, y, 0.0, up, dn, r1, r2);
  for (int i = 0; i < 8; ++i) {
    out[threadIdx.x + 64 * i] = up[i];
    out[512 + threadIdx.x + 64 * i] = dn[i];
  }
}
''')
    ops = re.findall(r"v_fmac_f64_dpp (v\[\d+:\d+\]), -?(v\[\d+:\d+\]), (v\[\d+:\d+\])", _assembly(str(src), tmp_path))
    assert len(ops) == 16
    assert not {o[0] for o in ops} & {f for o in ops for f in o[1:]}
