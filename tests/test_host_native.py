"""Host-side pieces of the native library, compiled for the host alone: no GPU needed."""
import ctypes
import os
import shutil
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "pmpic_amd", "csrc")
HIPCC = os.environ.get("HIPCC") or shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


@pytest.fixture(scope="module")
def checks(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("host") / "checks.so")
    subprocess.run([HIPCC, "-x", "hip", "--offload-host-only", "-std=c++17", "-O1", "-fPIC", "-shared",
                    "-I", CSRC, os.path.join(HERE, "host", "checks.hip"), "-o", out], check=True)
    return ctypes.CDLL(out)


@pytest.mark.parametrize("cell", [0, 1, 2**25 - 1, 2**25, 2**26 - 1])
@pytest.mark.parametrize("head", [0, 17, 63])
def test_packed_runs_hold_every_cell_of_a_slot_table(checks, cell, head):
    """The binning packs a cell and a lane in 32 bits; grids with a slot table have up to 2^26
    cells, so the packed cell reaches the top bit."""
    out = (ctypes.c_int32 * 2)()
    checks.host_run_round_trip(cell, head, out)
    assert tuple(out) == (cell, head)
