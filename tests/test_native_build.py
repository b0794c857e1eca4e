"""The native entry (csrc/gdn_torch.cpp) is optional wherever the library is
built: a machine that cannot build it, or holds one built against another
torch, still gets the library, and its calls take the Python path.  CPU only:
the compilers are stand-ins that write an empty file.
"""

import os
import shutil
import subprocess
import sys
import types
import warnings

import pytest

from gdn_amd import _lib, packing

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                    "gated-delta-network_amd", "csrc")


def _tool(path, fail_on=None):
    """A compiler that creates its -o file, and fails for the source `fail_on`."""
    lines = ["#!/bin/sh", "out=", "for a in \"$@\"; do"]
    if fail_on:
        lines.append(f"  [ \"$a\" = {fail_on} ] && echo 'Python.h: No such file' >&2 && exit 1")
    lines += ["  [ \"$prev\" = -o ] && out=$a", "  prev=$a", "done", ": > \"$out\""]
    path.write_text("\n".join(lines) + "\n")
    path.chmod(0o755)
    return str(path)


@pytest.fixture
def tree(tmp_path):
    """The sources alone, as an unpacked solution holds them."""
    if shutil.which("make") is None:
        pytest.skip("needs make")
    csrc = tmp_path / "pkg" / "csrc"
    shutil.copytree(CSRC, csrc, ignore=shutil.ignore_patterns("_build", ".build.lock"))
    (tmp_path / "pkg" / "gdn_amd").mkdir()
    (tmp_path / "include").mkdir()
    shutil.copy(os.path.join(CSRC, "..", "..", "include", "gdn_amd.h"), tmp_path / "include")
    return csrc


def test_make_builds_the_library_without_torch(tree, tmp_path):
    # a python3 without torch (here: one that always fails)
    python = tmp_path / "python3"
    python.write_text("#!/bin/sh\nexit 1\n")
    python.chmod(0o755)
    tool = _tool(tmp_path / "cc")
    r = subprocess.run(["make", "-j4", "-C", str(tree), f"HIPCC={tool}", f"HOSTCXX={tool}",
                        f"PYTHON={python}"], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout + r.stderr
    assert (tree.parent / "gdn_amd" / "libgdn_amd.so").exists()
    assert not list((tree.parent / "gdn_amd").glob("_native*"))


@pytest.mark.parametrize("why", ["headers", "python"])
def test_ensure_library_without_the_native_entry(tree, tmp_path, monkeypatch, why):
    # the extension's compile fails, or the python3 of PATH has no torch: the
    # interpreter that asks is the one the extension is for
    if why == "python":
        (tmp_path / "python3").write_text("#!/bin/sh\nexit 1\n")
        (tmp_path / "python3").chmod(0o755)
        monkeypatch.setenv("PATH", f"{tmp_path}:{os.environ['PATH']}")
    monkeypatch.setenv("HIPCC", _tool(tmp_path / "hipcc"))
    monkeypatch.setenv("HOSTCXX", _tool(tmp_path / "cxx", "gdn_torch.cpp" if why == "headers" else None))
    lib = tree.parent / "gdn_amd" / "libgdn_amd.so"
    monkeypatch.setattr(packing, "PKG_DIR", tree.parent / "gdn_amd")
    monkeypatch.setattr(_lib, "LIB_PATH", str(lib))
    assert packing.ensure_library() == str(lib)
    assert lib.exists()
    assert bool(list(lib.parent.glob("_native*.so"))) == (why == "python")


def test_ensure_library_without_a_compiler(tree, tmp_path, monkeypatch):
    # no library, no entry: an error
    monkeypatch.setenv("HIPCC", "/bin/false")
    monkeypatch.setattr(packing, "PKG_DIR", tree.parent / "gdn_amd")
    monkeypatch.setattr(_lib, "LIB_PATH", str(tree.parent / "gdn_amd" / "libgdn_amd.so"))
    with pytest.raises(RuntimeError, match="building"):
        packing.ensure_library()


def _with_native(monkeypatch, module):
    import gdn_amd
    monkeypatch.setattr(_lib, "_native", None)
    monkeypatch.setattr(_lib, "_native_tried", False)
    monkeypatch.setitem(sys.modules, "gdn_amd._native", module)
    monkeypatch.setattr(gdn_amd, "_native", module, raising=False)


def test_native_of_another_torch_is_not_bound(monkeypatch):
    # it would unpack tensors by another torch's layout
    def bind(*_):
        raise AssertionError("bound")
    _with_native(monkeypatch, types.SimpleNamespace(bind=bind, torch_version="0.0"))
    with pytest.warns(RuntimeWarning, match="0.0"):
        assert _lib.native() is None
    with warnings.catch_warnings():
        warnings.simplefilter("error")
        assert _lib.native() is None  # said once


def test_native_of_this_torch_is_bound(monkeypatch):
    import torch
    seen = []
    module = types.SimpleNamespace(bind=lambda *a: seen.append(a), torch_version=torch.__version__)
    _with_native(monkeypatch, module)
    assert _lib.native() is module
    assert len(seen) == 1 and len(seen[0]) == 6 and all(seen[0])


def test_native_that_does_not_load_is_said(monkeypatch):
    # there, but not loadable (None in sys.modules: ImportError on import)
    _with_native(monkeypatch, None)
    import gdn_amd
    monkeypatch.delattr(gdn_amd, "_native")
    monkeypatch.setattr(_lib, "_native_file", lambda: "_native.so")
    with pytest.warns(RuntimeWarning, match="does not load"):
        assert _lib.native() is None


def test_built_native_names_its_torch():
    import torch
    module = _lib.native()
    if module is None:
        pytest.skip("the native entry is not built")
    assert module.torch_version == torch.__version__
