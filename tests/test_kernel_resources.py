"""The kernels that end in a row selection keep their arguments out of private memory.

select_row takes its arguments (over 200 bytes) by reference: where the compiler does not inline it, each
lane copies them to private memory before anything else, in launches that mostly find nothing to
do (the inverted lists' overflow fallback) or hold one short list per workgroup.  The compiler's
own resource remarks say how much private memory a kernel uses; no GPU is needed.
"""
from __future__ import annotations

import re
import subprocess

import pytest

from vectoraccelerate_amd import build


@pytest.mark.parametrize("source, kernels, count",
                         [("va_select", "select_kernel", 8), ("va_ivf", "fb_ivf_kernel|fb_kernel", 3)])
def test_selection_kernels_use_no_private_memory(source, kernels, count):
    cmd = [build.HIPCC, *build.CXXFLAGS, "-Rpass-analysis=kernel-resource-usage", "--cuda-device-only", "-c",
           str(build.CSRC / f"{source}.hip"), "-o", "/dev/null"]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    assert proc.returncode == 0, proc.stderr[-2000:]
    used = re.findall(r"Function Name: (\S+)(?:(?!Function Name).)*?ScratchSize \[bytes/lane\]: (\d+)", proc.stderr, re.S)
    sizes = {name: int(size) for name, size in used if re.search(kernels, name)}
    assert len(sizes) == count, sizes
    assert not any(sizes.values()), sizes
