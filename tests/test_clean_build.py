"""A tree without built files: one process builds it and calls the library, and the library serves without the extension module."""
import os
import shutil
import subprocess
import sys

import pytest

from minit_amd import build

ROOT = os.path.dirname(build.HERE)
SIZES = "1, 4096, 4096, 128, 4"

# Stands for hipcc: the device objects are empty, and the library linked from them is the one that is built already; host
# code is compiled as it is.
HIPCC = """#!{python}
import os, shutil, subprocess, sys
out = sys.argv[sys.argv.index("-o") + 1]
if any(a.endswith("binding.cpp") for a in sys.argv):
    sys.exit(subprocess.run([{hipcc!r}, *sys.argv[1:]]).returncode)
open(out, "w").close() if "-c" in sys.argv else shutil.copy({library!r}, out)
"""


@pytest.fixture
def tree(tmp_path):
    """The sources of the package and of the oracle, and the environment to run them in."""
    names = shutil.ignore_patterns("*.so", "*.tmp", "_build", "__pycache__", "csrc")
    shutil.copytree(build.HERE, tmp_path / "minit_amd", ignore=names)
    shutil.copytree(build.CSRC, tmp_path / "minit_amd" / "csrc")
    shutil.copytree(build.INCLUDE, tmp_path / "include")
    shutil.copytree(os.path.join(ROOT, "oracle"), tmp_path / "oracle", ignore=names)
    shutil.copy(os.path.join(ROOT, "__graft_entry__.py"), tmp_path)
    hipcc = tmp_path / "hipcc"
    hipcc.write_text(HIPCC.format(python=sys.executable, hipcc=build.find_hipcc(), library=build.LIB_PATH))
    hipcc.chmod(0o755)
    env = {k: v for k, v in os.environ.items() if k not in ("MINIT_HIP_LIB", "PYTHONPATH")}
    return tmp_path, {**env, "HIPCC": str(hipcc)}


def _run(tree, code):
    path, env = tree
    proc = subprocess.run([sys.executable, "-c", code], cwd=path, env=env, capture_output=True, text=True, timeout=300)
    assert proc.returncode == 0, proc.stderr


CALLS = f"""
from minit_amd import lib
import minit_amd.hip.dispatch, minit_amd.quantize.gptq
calls = {{lib.call, minit_amd.hip.dispatch.call, minit_amd.quantize.gptq.call}}
assert len(calls) == 1
assert lib._call_general("mh_gptq_workspace_bytes", {SIZES}) == lib.call("mh_gptq_workspace_bytes", {SIZES})
try:
    lib.call("mh_softmax_causal", None, 256, 256, 1, 2, 7, 3, 1.0, 0)
except lib.HipError as e:
    assert "t=7 must equal" in str(e)
else:
    raise SystemExit("not refused")
"""


def test_one_process_builds_and_calls(tree):
    """The package is imported before there is anything to load."""
    _run(tree, "import __graft_entry__\n__graft_entry__.build()\n" + CALLS +
         "lib._functions['mh_gptq_workspace_bytes'] = lambda *args: 1 / 0   # what the ctypes path would call\n"
         f"lib.call('mh_gptq_workspace_bytes', {SIZES})\n")
    # the next process has the module from the start
    _run(tree, CALLS + "assert lib.call is lib._binding.call\n")


def test_the_library_without_the_module(tree):
    _run(tree, "from minit_amd import build\nbuild.build(verbose=False)\n")
    os.remove(tree[0] / "minit_amd" / os.path.basename(build.BINDING_PATH))
    _run(tree, CALLS + "assert lib._binding is None\n")


def test_a_module_that_does_not_compile_replaces_nothing(tree):
    package = tree[0] / "minit_amd"
    built = [package / os.path.basename(p) for p in (build.LIB_PATH, build.BINDING_PATH)]
    for path in built:
        path.write_bytes(b"of the build before")
    (package / "csrc" / "binding.cpp").write_text("#error\n")
    _run(tree, "from minit_amd import build\n"
               "try:\n    build.build(verbose=False)\nexcept RuntimeError as e:\n    assert 'binding' in str(e)\n"
               "else:\n    raise SystemExit('built')\n")
    assert [p.read_bytes() for p in built] == [b"of the build before"] * 2


def test_no_headers_of_python(tree):
    """The library does not need them, and no module of an earlier build stays beside it."""
    _run(tree, "from minit_amd import build\nbuild.build(verbose=False)\n"
               "build.sysconfig.get_paths = lambda: {'include': 'none'}\nbuild.build(verbose=False)\n")
    _run(tree, CALLS + "assert lib._binding is None\n")


def test_a_module_of_another_interpreter(tree):
    """Python takes any _binding.so for a module of its own; what has no tag, or another one, is not loaded here."""
    package = tree[0] / "minit_amd"
    _run(tree, "from minit_amd import build\nbuild.build(verbose=False)\n")
    built = package / os.path.basename(build.BINDING_PATH)
    for name in ("_binding.so", "_binding.cpython-399-x86_64-linux-gnu.so"):
        built = built.rename(package / name)
        _run(tree, CALLS + "assert lib._binding is None\n")
