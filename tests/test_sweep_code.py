"""Code of the ILU(0) sweep kernels as compiled (AMD assembly of this source,
no GPU needed)."""
import os
import re
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "phase_amd", "csrc")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


@pytest.mark.skipif(not shutil.which(HIPCC), reason="no hipcc")
def test_sweeps_issue_their_first_loads_before_any_branch(tmp_path):
    """A sweep launch lasts about as long as its chain of memory round trips,
    whose first holds the lane records, the block record and the run's `done`
    flag together: in each kernel the vector load of the lane records comes
    before the first conditional branch (the test of `done`)."""
    make = open(os.path.join(CSRC, "Makefile")).read()
    flags = re.search(r"^HIPFLAGS := (.*?[^\\])$", make, re.M | re.S).group(1)
    flags = flags.replace("\\\n", " ").replace("$(ARCH)", "gfx950").split()
    out = tmp_path / "solver.s"
    subprocess.run([HIPCC, *flags, "--cuda-device-only", "-S", os.path.join(CSRC, "solver.hip"), "-o", str(out)],
                   check=True, stderr=subprocess.DEVNULL)
    kernels = re.findall(r"^(_ZN5phase\d+k(?:L|U|LU)SolveI\w+):.*?\n(.*?)^\.Lfunc_end", out.read_text(), re.M | re.S)
    assert len(kernels) >= 20
    late = [name for name, body in kernels if "global_load" not in body.split("s_cbranch")[0]]
    assert not late, late
