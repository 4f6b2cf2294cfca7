"""Size of the tile kernels' argument blocks: at 256 bytes instead of 240 the
smallest launches (8-point rows and columns, 32-point real rows) took 2-8%
longer."""
import os
import shutil
import subprocess

import pytest

from genfft_amd import _capi as C

HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="needs the compiler")
@pytest.mark.parametrize("struct,most", [("TileArgs", 240), ("RealRowsArgs", 280)])
def test_argument_blocks_stay_small(struct, most, tmp_path):
    src = tmp_path / "size.hip"
    src.write_text(f'#include "gfft_r2c.h"\nstatic_assert(sizeof(gfft::{struct}) <= {most}, "");\n')
    r = subprocess.run([HIPCC, "--offload-arch=gfx950", "-std=c++17", "-fsyntax-only", "-I",
                        os.path.join(os.path.dirname(C.LIB_PATH), "csrc"), str(src)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
