"""What `make` builds: both HIP libraries with hipcc alone; the native host side of small steps beside them where its headers are."""
import os
import shutil
import stat
import subprocess
import sys

import pytest

PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "vllm-splitwise_amd")
LIBS = ["libsplitwise_hip.so", "libsplitwise_mixers.so"]


def _script(path, text):
    path.write_text(text)
    path.chmod(path.stat().st_mode | stat.S_IXUSR)
    return str(path)


@pytest.fixture
def tree(tmp_path):
    """The Makefile over empty sources, with a compiler that only writes its output."""
    pkg = tmp_path / "pkg"
    for name in ("csrc/a.hip", "csrc/common.cuh", "csrc/mixers/b.hip", "csrc/host/step_ops.cpp", "splitwise_amd/__init__.py",
                 "../include/splitwise_hip.h", "../include/splitwise_mixers.h"):
        (pkg / name).parent.mkdir(parents=True, exist_ok=True)
        (pkg / name).write_text("")
    shutil.copy(os.path.join(PKG, "Makefile"), pkg)
    compiler = _script(tmp_path / "compile", "#!/bin/sh\nwhile [ \"$1\" != -o ]; do shift; done\n: > \"$2\"\n")
    broken = _script(tmp_path / "broken", "#!/bin/sh\nexit 1\n")

    def make(*args, python=sys.executable, cxx=compiler):
        env = {k: v for k, v in os.environ.items() if not k.startswith("MAKE")}
        return subprocess.run(["make", "-C", str(pkg), f"HIPCC={compiler}", f"CXX={cxx}", f"PYTHON={python}", *args],
                              capture_output=True, text=True, env=env, timeout=60)
    make.broken = broken
    make.built = lambda: sorted(p.name for p in (pkg / "splitwise_amd").glob("*.so"))
    return make


@pytest.mark.parametrize("args", [[], ["-j4"], ["-B", "-j4"]], ids=" ".join)
@pytest.mark.parametrize("lacking", ["python", "headers", "compiler"])
def test_without_the_extension_both_libraries_are_built(tree, tmp_path, lacking, args):
    """No Python, a Python without its own or torch's headers, a compiler that does not take the sources."""
    python = _script(tmp_path / "python", "#!/bin/sh\necho /nowhere\n")
    done = tree(*args, **{"python": dict(python="/bin/false"), "headers": dict(python=python), "compiler": dict(cxx=tree.broken)}[lacking])
    assert done.returncode == 0, done.stderr
    assert tree.built() == LIBS and "without _step_ops" in done.stdout + done.stderr


def test_the_extension_alone_is_asked_for_strictly(tree):
    assert tree("step-ops", cxx=tree.broken).returncode != 0 and tree.built() == []


def test_with_its_headers_everything_is_built(tree):
    done = tree("-j4")
    assert done.returncode == 0, done.stderr
    assert len(tree.built()) == 3 and any(n.startswith("_step_ops") for n in tree.built())
