"""The link-cell passes' LDS per wave, checked by the compiler on the host."""
import os
import shutil
import subprocess

import pytest

from helpers import ROOT

HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


@pytest.mark.parametrize("kind", ["CM_KIND_EAM1", "CM_KIND_EAM3", "CM_KIND_LJ"])
def test_waves_of_a_block_start_aligned(tmp_path, kind):
    """Wave k's arrays start at k times the bytes of one wave, doubles first:
    on a multiple of 8 at least for every k, 16 for the widest LDS access."""
    if not os.path.exists(HIPCC):
        pytest.skip("no hipcc")
    src = tmp_path / "layout.hip"
    src.write_text('#include "pair_cell.h"\n' f"static_assert(wave_lds_bytes({kind}) % 16 == 0);\n")
    r = subprocess.run([HIPCC, "--offload-arch=gfx950", "--cuda-host-only", "-std=c++17", "-fsyntax-only", "-w",
                        "-I", os.path.join(ROOT, "comd_amd", "csrc"), "-I", os.path.join(ROOT, "include"), str(src)],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
