"""What the library does when the interpreter ends (no device)."""
import os
import subprocess
import sys

from conftest import ROOT

CODE = """
import os, sys
from pypatools_amd import _lib
h = _lib.lib()
class Seen:
    def __call__(self):
        print("released in", "parent" if os.getpid() == PARENT else "child", flush=True)
PARENT = os.getpid()
_lib._release_at_exit.__globals__["_release"] = Seen()
pid = os.fork()
if pid == 0:
    sys.exit(0)             # a normal exit of the child runs its exit handlers
os.waitpid(pid, 0)
"""


def test_a_forked_child_leaves_the_parents_memory_alone():
    """Freeing the kept blocks and pinned buffers calls the HIP runtime, which a forked child must not touch."""
    res = subprocess.run([sys.executable, "-c", CODE], cwd=ROOT, capture_output=True, text=True, timeout=120)
    assert res.returncode == 0, res.stderr
    assert res.stdout.split("\n")[:-1] == ["released in parent"], res.stdout
