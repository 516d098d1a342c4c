"""The arguments of the kernels that small products run on: a launch with more than 96 bytes of them costs the host more, and
what a kernel asks of the runtime (the size of the grid, say) comes as 256 bytes behind its own."""
import concurrent.futures as cf
import re
import shutil
import subprocess
from pathlib import Path

import pytest

from axiom_amd import build

SOURCES = ("gemm_small.hip", "gemm_f32.hip", "gemm_tile_nt.hip", "gemm_tile_nn.hip", "gemm_skinny.hip")


@pytest.mark.skipif(not (shutil.which("hipcc") or Path("/opt/rocm/bin/hipcc").exists()), reason="no hipcc")
def test_product_kernels_take_no_more_than_their_own_arguments(tmp_path):
    def metadata(name):
        out = tmp_path / (name + ".s")
        flags = [f for f in build.HIP_FLAGS if f not in ("-O3", "-fPIC", "--offload-compress")]
        subprocess.run([build._hipcc(), *flags, "-O3", "--cuda-device-only", "-S", str(build.CSRC / name), "-o", str(out)], check=True, capture_output=True)
        return name, [int(n) for n in re.findall(r"\.kernarg_segment_size: (\d+)", out.read_text())]

    with cf.ThreadPoolExecutor(len(SOURCES)) as pool:
        for name, sizes in pool.map(metadata, SOURCES):
            assert sizes and max(sizes) <= 96, (name, sorted(set(sizes)))
