"""The register-resident kernels (bfm_amd/csrc/hip/resident.hip) that the solve
which allocates nothing (bfmx_system_solve_noalloc) launches need no scratch
memory, as the compiler reports it: for the first launch that does, the runtime
takes device memory. So do the others of one system, but for block Jacobi in
FP64 with 1024 threads, of which there is a second form for that solve."""

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
    may = [k for k in single if re.search(r"k_resident_pcgIdLi[79]ELi1ELi1024ELb0E", k)]
    assert len(single) == 20 and len(may) == 2
    assert not any(v for k, v in single.items() if k not in may), single
