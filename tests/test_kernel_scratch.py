"""The row kernels of triangle multiplication keep their registers: compiled with the
library's own flags none of them uses scratch memory (a launch that does costs about
a microsecond more, besides the traffic)."""
import os
import re
import shutil
import subprocess

import pytest

from bindcraft2_amd import build


@pytest.mark.skipif(not shutil.which(build.HIPCC), reason="no hipcc")
def test_no_scratch(tmp_path):
    src, asm = "trimul.hip", tmp_path / "device.s"
    subprocess.run([build.HIPCC, "-x", "hip", *build.FLAGS, *build.EXTRA.get(src, []), "-w", "-S",
                    "--cuda-device-only", "-I", build.CSRC, os.path.join(build.CSRC, src), "-o", str(asm)],
                   check=True)
    use = dict(re.findall(r"^\s+\.name:\s+(\S+)\s+\.private_segment_fixed_size: (\d+)", asm.read_text(), re.M))
    rows = {k: int(v) for k, v in use.items() if "gemm_" not in k}
    assert rows and not any(rows.values()), {k: v for k, v in rows.items() if v}
