"""No kernel keeps registers in scratch memory (CPU, the code as compiled here).

A spilled register costs a round trip to memory wherever it is needed again, and a
kernel with a private segment makes the runtime set scratch memory aside.
"""
from __future__ import annotations

import re
import shutil
import subprocess

import pytest

from k8v4_v030 import _build

SOURCES = sorted(p.name for p in _build.CSRC.glob("*.hip"))


@pytest.mark.skipif(shutil.which(_build.hipcc()) is None, reason="no hipcc")
@pytest.mark.parametrize("name", SOURCES)
def test_no_kernel_uses_scratch(name, tmp_path):
    asm = tmp_path / "kernels.s"
    subprocess.run([_build.hipcc(), *_build.COMMON_FLAGS, *_build.PER_FILE_FLAGS.get(name, []), "-S",
                    "--cuda-device-only", str(_build.CSRC / name), "-o", str(asm)], check=True, capture_output=True)
    use = re.findall(r"\.name:\s+(\S+)\n\s+\.private_segment_fixed_size:\s+(\d+)", asm.read_text())
    assert bool(use) == ("__global__" in (_build.CSRC / name).read_text())
    assert [kernel for kernel, size in use if int(size)] == []
