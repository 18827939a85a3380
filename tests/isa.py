"""The gfx950 assembly of one kernel source, compiled with the build's own
flags (no GPU), once per test run."""

from __future__ import annotations

import functools
import re
import shutil
import subprocess
import tempfile
from pathlib import Path

import pytest

from foldjax_amd import build as B


@functools.lru_cache(maxsize=None)
def assembly(src: str) -> tuple[str, ...]:
    hipcc = B._hipcc()
    if not shutil.which(hipcc) and not Path(hipcc).is_file():
        pytest.skip("hipcc is not available")
    with tempfile.TemporaryDirectory() as tmp:
        out = Path(tmp) / (Path(src).stem + ".s")
        cmd = [hipcc, *B.HIP_FLAGS, *B.FILE_FLAGS.get(src, []), "--cuda-device-only", "-S", str(B.CSRC / src), "-o",
               str(out)]
        proc = subprocess.run(cmd, capture_output=True, text=True)
        assert proc.returncode == 0, proc.stderr[-2000:]
        return tuple(out.read_text().splitlines())


def kernels(src: str) -> dict[str, list[str]]:
    """Each function's instructions and labels, comments stripped."""
    out: dict[str, list[str]] = {}
    name = None
    for line in assembly(src):
        text = line.split(";")[0].strip()
        m = re.match(r"\.type\s+(\S+),@function", text)
        if m:
            name = m.group(1)
            out[name] = []
        elif re.match(r"\.Lfunc_end", text):
            name = None
        elif name and text and (text.endswith(":") or not text.startswith(".")):
            out[name].append(text)
    return out
