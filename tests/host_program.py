"""Host programs over the kernels' headers (launch models and range formulas),
compiled by hipcc for the CPU alone: no GPU is needed to build or run them."""

from __future__ import annotations

import functools
import os
import subprocess
import tempfile

from mlxturbo_amd import build

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
_DIR = tempfile.TemporaryDirectory(prefix="mq_host_")


@functools.lru_cache(maxsize=None)
def _compiled(source: str) -> str:
    exe = os.path.join(_DIR.name, os.path.splitext(os.path.basename(source))[0])
    subprocess.run([build.hipcc(), "-x", "hip", "--offload-host-only", "-std=c++17", "-O1",
                    "-I", build.CSRC, "-I", os.path.join(ROOT, "include"), "-o", exe,
                    os.path.join(ROOT, "tests", source)], check=True, capture_output=True,
                   text=True, timeout=300)
    return exe


def run(source: str, lines) -> list[str]:
    """Output lines of tests/``source`` for the given input lines."""
    res = subprocess.run([_compiled(source)], input="\n".join(lines) + "\n", check=True,
                         capture_output=True, text=True, timeout=300)
    return res.stdout.splitlines()
