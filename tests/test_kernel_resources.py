"""What the compiler says of kernels whose speed rests on their registers."""
from __future__ import annotations

import os
import re
import subprocess

import pytest

from serve_amd.csrc import build


@pytest.mark.parametrize("source", ["elementwise.hip", "gemm_split.hip"])
def test_no_register_is_spilled(source, tmp_path):
    """Every kernel of the file, every instantiation, under the build's own flags: nothing goes to scratch memory."""
    hipcc = build._hipcc()
    if hipcc is None:
        pytest.skip("no hipcc")
    flags = [f for f in build.FLAGS if f not in ("-shared", "-fPIC")]
    run = subprocess.run([hipcc, *flags, "--cuda-device-only", "-c", "-Rpass-analysis=kernel-resource-usage",
                          "-o", str(tmp_path / "x.o"), os.path.join(build.CSRC, source)], capture_output=True, text=True,
                         timeout=300)
    assert run.returncode == 0, run.stderr[-2000:]
    names = re.findall(r"Function Name: (\S+)", run.stderr)
    scratch = [int(n) for n in re.findall(r"ScratchSize \[bytes/lane\]: (\d+)", run.stderr)]
    assert len(names) == len(scratch) > 0
    assert not [(n, b) for n, b in zip(names, scratch) if b]
