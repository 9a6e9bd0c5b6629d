"""The host extension (csrc/host_params.cpp) only spares time, so the library is built with hipcc alone too; and it is taken only
where it was compiled for this torch and Python, from its source as it is."""
import os
import sys

import pytest

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "openfold-3_amd"))

import torch  # noqa: E402

from of3pair import _block, _lib  # noqa: E402
from of3pair import build as of3_build  # noqa: E402


@pytest.mark.parametrize("lacks", ["compiler", "Python.h", "torch's headers"])
def test_library_without_the_host_extension(monkeypatch, tmp_path, lacks):
    """hipcc is a stand-in that writes its output file; the host compiler is the real one, without what it lacks."""
    hipcc = tmp_path / "hipcc"
    hipcc.write_text('#!/bin/sh\nwhile [ "$1" != -o ]; do shift; done\n: > "$2"\n')
    hipcc.chmod(0o755)
    monkeypatch.setenv("HIPCC", str(hipcc))
    for name in ("LIB_DIR", "LIB_PATH", "STAMP_PATH"):
        path = getattr(of3_build, name)
        monkeypatch.setattr(of3_build, name, str(tmp_path / "lib") if name == "LIB_DIR" else str(tmp_path / "lib" / os.path.basename(path)))
    os.makedirs(of3_build.LIB_DIR)
    open(of3_build.host_path(), "w").close()  # of an earlier build
    if lacks == "compiler":
        monkeypatch.setenv("CXX", str(tmp_path / "none"))
    elif lacks == "Python.h":
        import sysconfig

        monkeypatch.setattr(sysconfig, "get_paths", lambda: {"include": str(tmp_path)})
    else:
        from torch.utils import cpp_extension

        monkeypatch.setattr(cpp_extension, "include_paths", lambda: [str(tmp_path)])
    with pytest.warns(UserWarning, match="not built"):
        assert of3_build.build() == of3_build.LIB_PATH
    assert of3_build.is_built() and not os.path.exists(of3_build.host_path())


def _prerequisites():
    import shutil
    import sysconfig

    from torch.utils import cpp_extension

    return (shutil.which(os.environ.get("CXX", "g++")) and os.path.exists(os.path.join(sysconfig.get_paths()["include"], "Python.h"))
            and any(os.path.exists(os.path.join(d, "torch", "extension.h")) for d in cpp_extension.include_paths()))


@pytest.mark.skipif(not of3_build.is_built() or not _prerequisites(), reason="library not built, or the extension cannot be")
def test_the_extension_is_there_and_taken():
    assert os.path.exists(of3_build.host_path()) and _block._scan is not None and _lib.load_scan() is not None


@pytest.mark.skipif(_block._scan is None, reason="host extension not built")
@pytest.mark.parametrize("what", ["__version__", "version.git_version", "_C._GLIBCXX_USE_CXX11_ABI", "SOABI"])
def test_not_taken_for_another_torch_or_python(monkeypatch, what):
    if what == "SOABI":
        import sysconfig

        monkeypatch.setattr(sysconfig, "get_config_var", lambda name: "cpython-39-x86_64-linux-gnu")
    else:
        monkeypatch.setattr("torch." + what, not torch._C._GLIBCXX_USE_CXX11_ABI if what.startswith("_C") else "other")
    with pytest.warns(UserWarning, match="in Python"):
        assert _lib.load_scan() is None


@pytest.mark.skipif(_block._scan is None, reason="host extension not built")
def test_not_taken_where_its_source_has_changed(monkeypatch):
    """As the library is refused then."""
    monkeypatch.setattr(of3_build, "source_digest", lambda: "another")
    assert _lib.load_scan() is None
