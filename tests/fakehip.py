"""Run a snippet against libculbm.so on the stand-in runtime of fake_hip.cpp.

The stand-in is loaded with global visibility before the library, in a process
of its own, so its symbols take the place of the HIP runtime's.  The snippet
sees `fake` (the stand-in's controls), `launched()` (the kernels launched since
the last fake.fake_clear(), by plain name), numpy as `np` and the package's
Lattice, LatticeConfig, cases and _lib."""
from __future__ import annotations

import functools
import subprocess
import sys
import tempfile
import textwrap
from pathlib import Path

ROOT = Path(__file__).resolve().parents[1]

PREAMBLE = """
import ctypes, re, sys
fake = ctypes.CDLL({so!r}, mode=ctypes.RTLD_GLOBAL)
fake.fake_limit.argtypes = [ctypes.c_size_t]
fake.fake_bytes.restype = ctypes.c_size_t
fake.fake_log.restype = ctypes.c_char_p
fake.fake_fail_new.argtypes = [ctypes.c_long]
for f in (fake.fake_copies, fake.fake_largest, fake.fake_grid):
    f.restype = ctypes.c_long
fake.fake_known.argtypes = [ctypes.c_void_p, ctypes.c_size_t]
sys.path.insert(0, {root!r})
import numpy as np
from culbm_amd import Lattice, LatticeConfig, _lib, cases
assert "torch" not in sys.modules

def launched():
    return [re.search(r"\\d(k_[a-z0-9_]+)", n).group(1).split("I")[0] for n in fake.fake_log().decode().split()]
"""


@functools.lru_cache(maxsize=None)
def library() -> str:
    out = Path(tempfile.mkdtemp(prefix="fake_hip_")) / "libfake_hip.so"
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", str(ROOT / "tests" / "fake_hip.cpp"), "-o", str(out)],
                   check=True)
    return str(out)


def run(snippet: str) -> str:
    """stdout of the snippet; a non-zero exit or a signal fails the test."""
    code = PREAMBLE.format(so=library(), root=str(ROOT)) + textwrap.dedent(snippet)
    r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=120, cwd=str(ROOT))
    assert r.returncode == 0, f"exit {r.returncode}\n{r.stdout[-2000:]}\n{r.stderr[-4000:]}"
    return r.stdout
