"""The whole-cycle call runs on the HIP runtime that the library was built for, and is neither
taken by default nor entered on an older one that another package loaded before it, nor under
a profiler."""
import os
import subprocess
import sys

import pytest

CODE = """
{first}
import sys
sys.path.insert(0, {path!r})
from hpmp import _lib, multigrid
_lib.load()
{then}
print(_lib.load().hpg_cycle_available(), multigrid.fused_available([]))
"""


def _run(first, then=""):
    import hpmp
    path = os.path.dirname(os.path.dirname(os.path.abspath(hpmp.__file__)))
    r = subprocess.run([sys.executable, "-c", CODE.format(first=first, path=path, then=then)], capture_output=True, text=True,
                       check=True, timeout=300)
    return r.stdout.split()


def test_cycle_on_the_runtime_of_the_build():
    assert _run("") == ["1", "True"]


def test_no_cycle_under_a_profiler():
    # set after the runtime is loaded, which would look for the tool
    assert _run("", "import os; os.environ['ROCP_TOOL_LIBRARIES'] = 'tool'") == ["0", "False"]


def test_no_cycle_on_an_older_runtime_loaded_first():
    version = subprocess.run([sys.executable, "-c", "import torch; print(torch.version.hip)"], capture_output=True,
                             text=True, timeout=300).stdout.split(".")
    own = subprocess.run(["/opt/rocm/bin/hipconfig", "--version"], capture_output=True, text=True).stdout.split(".")
    if len(version) < 2 or len(own) < 2 or tuple(map(int, version[:2])) >= tuple(map(int, own[:2])):
        pytest.skip("torch brings no older HIP runtime")
    assert _run("import torch") == ["0", "False"]
