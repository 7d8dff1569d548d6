"""When the operators find their libraries and what they raise if they do not:
in processes of their own, over copies of the package, without a GPU (the C++
kernels check their operands and query a workspace on the host)."""
import os
import shutil
import subprocess
import sys

import pytest

from chronicals_amd import build as _build

HEAD = '''
import os, shutil, sys
import torch
from chronicals_amd import _lib, build, ops
assert build.REPO_DIR == os.getcwd(), build.REPO_DIR

def call():
    """The CUDA kernel of cce_fwd on host tensors, with a d that is no multiple of 8."""
    h, w = torch.zeros(4, 7, dtype=torch.bfloat16), torch.zeros(5, 7, dtype=torch.bfloat16)
    keys = torch._C.DispatchKeySet(torch._C.DispatchKey.CUDA)
    try:
        torch.ops.chronicals_hip.cce_fwd.default.redispatch(keys, h, w, torch.zeros(4, dtype=torch.int64), None, -100,
                                                            0.0, 0.0, 0, 1, 0)
    except Exception as e:
        return e

def works():
    e = call()
    assert type(e) is _lib.CCEError and "multiple of 8" in str(e), repr(e)
'''


@pytest.fixture
def tree(tmp_path):
    """A copy of the package with its sources and built libraries."""
    for path in (_build.LIB_PATH, _build.torch_lib_path()):
        if not os.path.exists(path):
            pytest.fail(f"{path} is not built: run __graft_entry__.build()")
    shutil.copytree(_build.PKG_DIR, tmp_path / "chronicals_amd", ignore=shutil.ignore_patterns("__pycache__"))
    shutil.copytree(os.path.dirname(_build.HEADER), tmp_path / "include")
    return tmp_path


def run(tree, code, **env):
    env = dict({k: v for k, v in os.environ.items() if k not in ("CHRONICALS_CCE_LIB", "PYTHONPATH")}, **env)
    out = subprocess.run([sys.executable, "-c", HEAD + code], capture_output=True, text=True, cwd=tree, env=env,
                         timeout=300)
    assert out.returncode == 0, out.stdout + out.stderr


def test_errors_of_the_c_library_keep_their_type(tree):
    run(tree, "works()\n")


def test_a_broken_library_raises_in_the_call(tree):
    broken = tree / "broken.so"
    broken.write_bytes(b"not a library")
    run(tree, "assert type(call()) is OSError, repr(call())\n", CHRONICALS_CCE_LIB=str(broken))


def test_a_library_built_after_the_import_is_found(tree):
    run(tree, "shutil.move(build.LIB_PATH, 'away.so')\n"
              "e = call()\n"
              "assert type(e) is ImportError and 'not found' in str(e), repr(e)\n"
              "shutil.move('away.so', build.LIB_PATH)\n"
              "works()\n")


def test_a_stale_library_is_refused_until_it_is_rebuilt(tree):
    src = tree / "chronicals_amd" / "csrc" / "cce_kernels.hip"
    text = src.read_text()
    src.write_text(text + "// edit\n")
    run(tree, "e = call()\n"
              "assert type(e) is ImportError and 'other sources' in str(e), repr(e)\n"
              f"text = open({str(src)!r}).read()\n"
              f"open({str(src)!r}, 'w').write(text[:-len('// edit\\n')])\n"
              "works()\n")


def test_the_environment_names_the_library_until_the_first_call(tree):
    run(tree, "os.environ['CHRONICALS_CCE_LIB'] = '/absent/lib.so'\n"
              "e = call()\n"
              "assert type(e) is ImportError and '/absent/lib.so' in str(e), repr(e)\n"
              "del os.environ['CHRONICALS_CCE_LIB']\n"
              "works()\n")


def test_operators_built_after_the_import_are_found(tree):
    built = tree / "chronicals_amd" / "lib" / os.path.basename(_build.torch_lib_path())
    shutil.move(built, tree / "away.so")
    run(tree, "e = call()\n"
              "assert type(e) is ImportError and 'build it' in str(e), repr(e)\n"
              "shutil.move('away.so', build.torch_lib_path())\n"
              "e = call()  # loads the kernels and goes on to the tensors' own device\n"
              "assert isinstance(e, NotImplementedError), repr(e)\n"
              "works()\n")


def test_in_place_and_functional_operators_agree(tree):
    # the Python loader and the C++ kernels hold one library
    run(tree, "works()\n"
              "maps = {l.split()[-1] for l in open('/proc/self/maps') if 'libchronicals_cce' in l}\n"
              "assert maps == {os.path.realpath(build.LIB_PATH)}, maps\n"
              "assert _lib.load()._name == build.LIB_PATH\n")


def test_a_tree_without_its_sources_works(tree):
    shutil.rmtree(tree / "include")
    run(tree, "works()\n")
    shutil.rmtree(tree / "chronicals_amd" / "csrc")
    run(tree, "works()\n")
    # a build for another torch is not loaded
    lib = tree / "chronicals_amd" / "lib"
    built = os.path.basename(_build.torch_lib_path())
    shutil.move(lib / built, lib / built.replace(".so", "x.so"))
    run(tree, "e = call()\nassert type(e) is ImportError and 'build it' in str(e), repr(e)\n")
