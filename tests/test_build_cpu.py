"""What `make` builds: both HIP libraries with hipcc alone; the native host side of small steps beside them where its headers are."""
import importlib
import os
import shutil
import stat
import subprocess
import sys
import sysconfig
import types
import warnings

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
    make.broken, make.compiler, make.directory = broken, compiler, str(pkg)
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


def _loaded(monkeypatch, extension):
    """The module that chooses the extension, imported anew where `import _step_ops` gives `extension` -> what it took, its warnings."""
    import splitwise_amd
    kept = importlib.import_module("splitwise_amd._native")
    monkeypatch.setitem(sys.modules, "splitwise_amd._step_ops", extension)
    monkeypatch.setattr(splitwise_amd, "_native", kept)                     # (put back what the import below sets)
    monkeypatch.delitem(sys.modules, "splitwise_amd._native")
    with warnings.catch_warnings(record=True) as said:
        warnings.simplefilter("always")
        taken = importlib.import_module("splitwise_amd._native").step_ops
    return taken, [str(w.message) for w in said]


@pytest.mark.parametrize("torch_was", [None, "0.0.0 other", "same version, another commit"])
def test_an_extension_of_another_torch_is_not_used(monkeypatch, torch_was):
    import torch
    if torch_was is not None and "commit" in torch_was:
        torch_was = torch.__version__ + " 0000"
    stale = types.SimpleNamespace(__file__="stale.so", SW_ABI_VERSION=7, SWM_ABI_VERSION=7, gla=lambda *a: 0)
    if torch_was is not None:
        stale.TORCH = torch_was
    taken, said = _loaded(monkeypatch, stale)
    assert taken is not stale and taken.gla(1, 2) is None
    assert len(said) == 1 and "not used" in said[0]


def test_the_extension_that_was_built_here_is_used(monkeypatch):
    kept = importlib.import_module("splitwise_amd._native")
    try:
        ours = importlib.import_module("splitwise_amd._step_ops")
    except ImportError:
        pytest.skip("built without the extension")
    assert kept.step_ops is ours
    taken, said = _loaded(monkeypatch, ours)
    assert taken is ours and said == []


def test_an_extension_that_does_not_load_is_named(monkeypatch, tmp_path):
    """None in sys.modules makes the import fail as an undefined symbol does."""
    kept = importlib.import_module("splitwise_amd._native")
    monkeypatch.setattr(kept.glob, "glob", lambda pattern: [pattern])
    taken, said = _loaded(monkeypatch, None)
    assert taken.gla(1, 2) is None and len(said) == 1 and "does not load" in said[0]
    monkeypatch.setattr(kept.glob, "glob", lambda pattern: [])
    assert _loaded(monkeypatch, None)[1] == []                              # it is optional


@pytest.mark.parametrize("theirs,bound", [(7, True), (6, False)])
def test_an_extension_of_another_interface_is_named(monkeypatch, theirs, bound):
    import ctypes
    native = importlib.import_module("splitwise_amd._native")
    seen = []
    monkeypatch.setattr(native, "step_ops", types.SimpleNamespace(__file__="stale.so", SW_ABI_VERSION=theirs, bind=seen.append))
    with warnings.catch_warnings(record=True) as said:
        warnings.simplefilter("always")
        native.bind_library(ctypes.CDLL(None), ["malloc"], 7, "SW_ABI_VERSION")
        assert len(seen) == bound and len(said) == (not bound)
        monkeypatch.setattr(native, "step_ops", native._NotBuilt())          # none there: nothing to name
        native.bind_library(ctypes.CDLL(None), ["malloc"], 7, "SW_ABI_VERSION")
    assert len(seen) == bound and len(said) == (not bound)


def test_the_extension_follows_torch(tree, tmp_path):
    """Built again when another torch is there, not otherwise, under the name of this Python's extensions."""
    fake = tmp_path / "site" / "torch"
    (fake / "include" / "ATen").mkdir(parents=True)
    (fake / "include" / "ATen" / "ATen.h").write_text("")
    (fake / "__init__.py").write_text("")
    env = dict(os.environ, PYTHONPATH=str(tmp_path / "site"))
    for version, anew in (("1.0", True), ("1.0", False), ("2.0", True), ("2.0", False)):
        (fake / "version.py").write_text(f"__version__, git_version = {version!r}, 'abc'\n")
        done = subprocess.run(["make", "-C", tree.directory, "step-ops", f"CXX={tree.compiler}", f"PYTHON={sys.executable}"],
                              capture_output=True, text=True, env=env, timeout=60)
        assert done.returncode == 0, done.stderr
        assert (f"-DSTEP_OPS_TORCH='\"{version} abc\"'" in done.stdout) == anew
    assert tree.built() == ["_step_ops" + sysconfig.get_config_var("EXT_SUFFIX")]


def test_calls_that_the_extension_does_not_take_are_not_offered(monkeypatch):
    """Slopes, sigmoid weights and values inside the key rows are common forms that it leaves to Python, by a throw."""
    import torch
    from splitwise_amd import _C, _C_mixers
    offered = []
    spy = types.SimpleNamespace(**{name: (lambda *args, name=name: offered.append(name))
                                   for name in ("paged_attention_v1", "prefill_attention", "capped_attention")})
    monkeypatch.setattr(_C, "_native", spy)
    monkeypatch.setattr(_C_mixers, "_native", spy)
    t = torch.zeros(1)
    calls = {"paged_attention_v1": (lambda slopes: _C.ops.paged_attention_v1(t, t, t, t, 1, 1.0, t, t, 16, 1, slopes, "auto"), [None], [t]),
             "prefill_attention": (lambda slopes: _C.ops.prefill_attention(t, t, t, t, t, t, 1, 1.0, slopes), [None], [t]),
             "capped_attention": (lambda v, bias: _C_mixers.capped_attention(t, t, t, v, None, None, 1, 1, 8, 8, 1.0, score_bias=bias),
                                  [t, None], [None, None, t, t])}
    for name, (call, plain, others) in calls.items():
        for i in range(0, len(others), len(plain)):
            with pytest.raises(RuntimeError, match="need tensors on a HIP device"):
                call(*others[i:i + len(plain)])
        assert offered == []
        with pytest.raises(RuntimeError, match="need tensors on a HIP device"):
            call(*plain)
        assert offered == [name]
        offered.clear()
