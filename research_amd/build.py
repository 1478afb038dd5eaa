"""Compile the HIP sources in ``research_amd/csrc`` into ``libpaged_attn.so``, and the calls from Python into the module ``_host``.

``python -m research_amd.build`` runs ``make`` with hipcc for gfx950; the
libraries land next to the package's ``_lib.py``.  hipcc cross-compiles, so
this works on a machine without a GPU.
"""

from __future__ import annotations

import importlib.util
import os
import subprocess
import sys

CSRC = os.path.join(os.path.dirname(os.path.abspath(__file__)), "csrc")


def build(force: bool = False, jobs: int = 8) -> str:
    if force:
        subprocess.run(["make", "-C", CSRC, "clean"], check=True, stdout=subprocess.DEVNULL)
    proc = subprocess.run(["make", "-C", CSRC, f"-j{jobs}", f"PYTHON={sys.executable}", "all"], stdout=subprocess.PIPE,
                          stderr=subprocess.STDOUT, text=True)
    if proc.returncode != 0:
        sys.stderr.write(proc.stdout)
        raise RuntimeError("building libpaged_attn.so / _host failed")
    from . import _lib

    return _lib.LIB_PATH


def built() -> bool:
    """Whether the library and this interpreter's module are there."""
    from . import _lib

    return os.path.exists(_lib.LIB_PATH) and importlib.util.find_spec(__package__ + "._host") is not None


if __name__ == "__main__":
    print(build(force="--force" in sys.argv))
