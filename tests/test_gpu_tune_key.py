"""The autotuner's kept choices name the line blocks of a system: a choice made without them (an
older SLLG_TUNE_FILE) is not taken for a handle that has them."""
import os
import subprocess
import sys

import pytest

import sllg

pytestmark = pytest.mark.gpu

CODE = """
import sys
sys.path.insert(0, sys.argv[1])
import sllg
from sllg import workloads as W
s = W.fcc_3shell(dims=(9, 10, 11))[0]
with sllg.Context(s) as g:
    assert "-blocks11x" in g.info()["exch_encoding"]
    r = g.autotune(2)
print("from_cache", int(r["from_cache"]), "line_mode", r["line_mode"])
"""


def _tune(path):
    pkg = os.path.dirname(os.path.dirname(os.path.abspath(sllg.__file__)))
    p = subprocess.run([sys.executable, "-c", CODE, pkg], env=dict(os.environ, SLLG_TUNE_FILE=str(path)), text=True,
                       capture_output=True, timeout=90)
    assert p.returncode == 0, p.stderr
    w = p.stdout.split()
    return int(w[1]), int(w[3])


def test_choice_without_blocks_is_not_taken(gpu, tmp_path):
    f = tmp_path / "tune"
    assert _tune(f)[0] == 0
    key, *choice = f.read_text().split()
    assert _tune(f) == (1, int(choice[-1]))  # its own choice is
    old = tmp_path / "old"  # the same system's key before blocks were part of it, packed reader
    old.write_text(" ".join([key.split("|B")[0], *choice[:-1], "1"]) + "\n")
    assert _tune(old)[0] == 0
