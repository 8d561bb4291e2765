"""The register-resident solvers of one system (bfm_amd/csrc/hip/resident.hip)
use no scratch memory, as the compiler reports it: a spilled register is read
back through memory in every iteration, and the solve that allocates nothing
(bfmx_system_solve_noalloc) must not need scratch that the runtime would have to
provide. The batch kernels carry more state and may spill."""

import os
import re
import shutil
import subprocess

import pytest

from bfm_amd import build as B


@pytest.mark.skipif(not shutil.which(B.HIPCC), reason="no hipcc")
def test_no_scratch(tmp_path):
    r = subprocess.run([B.HIPCC, *B.HIP_FLAGS, "--cuda-device-only", "-Rpass-analysis=kernel-resource-usage", "-c",
                        os.path.join(B.HIP_DIR, "resident.hip"), "-o", str(tmp_path / "resident.o")],
                       capture_output=True, text=True, check=True)
    used = dict(re.findall(r"Function Name: (\S+).*?ScratchSize \[bytes/lane\]: (\d+)", r.stderr, re.S))
    single = {k: int(v) for k, v in used.items() if "k_resident_pcg" in k or "k_resident_minres" in k}
    assert len(single) == 18
    assert not any(single.values()), single
