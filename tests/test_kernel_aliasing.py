"""Kernel arguments that other arguments of the same launch point into carry no no-alias promise (read from the device
code's argument attributes as hipcc emits them)."""
import re
import shutil
import subprocess
from pathlib import Path

import pytest

from dftax_amd import build


def _arguments(source, kernel, tmp_path):
    """The argument list of a kernel in the device IR of one source file."""
    if not (Path(build.HIPCC).exists() or shutil.which(build.HIPCC)):
        pytest.skip("no hipcc")
    out = tmp_path / "device.ll"
    subprocess.run([build.HIPCC, *build.CFLAGS, "--cuda-device-only", "-S", "-emit-llvm", str(build.CSRC / source),
                    "-o", str(out)], check=True, capture_output=True, text=True)
    m = re.search(r"define [^\n]*amdgpu_kernel void @\w*" + kernel + r"\w*\(([^\n]*)\)[^\n]*\{", out.read_text())
    assert m, f"{kernel} not found in {source}"
    return m.group(1)


def test_energy_terms_are_summed_after_they_are_stored(tmp_path):
    """k_dots_final stores E[1..4] through its list and sums E[1..5] into E[0]: of its two pointers only the partial
    sums may be no-alias."""
    args = _arguments("linalg.hip", "k_dots_final", tmp_path)
    pointers = [a for a in re.split(r",\s*(?=ptr)", args) if a.startswith("ptr")]
    plain = [a for a in pointers if "byref" not in a and "byval" not in a]
    assert len(plain) == 2
    assert "noalias" in plain[0] and "noalias" not in plain[1]
