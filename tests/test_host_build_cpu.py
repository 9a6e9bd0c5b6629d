"""Building with hipcc alone: the host extension (csrc/host_params.cpp) only spares time, so the library comes without it."""
import os
import sys

import pytest

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "openfold-3_amd"))

from of3pair import build as of3_build  # noqa: E402


@pytest.mark.parametrize("lacks", ["compiler", "Python.h", "torch's headers"])
def test_library_without_the_host_extension(monkeypatch, tmp_path, lacks):
    """hipcc is a stand-in that writes its output file; the host compiler is the real one, without what it lacks."""
    hipcc = tmp_path / "hipcc"
    hipcc.write_text('#!/bin/sh\nwhile [ "$1" != -o ]; do shift; done\n: > "$2"\n')
    hipcc.chmod(0o755)
    monkeypatch.setenv("HIPCC", str(hipcc))
    for name in ("LIB_DIR", "LIB_PATH", "STAMP_PATH", "HOST_PATH"):
        path = getattr(of3_build, name)
        monkeypatch.setattr(of3_build, name, str(tmp_path / "lib") if name == "LIB_DIR" else str(tmp_path / "lib" / os.path.basename(path)))
    os.makedirs(of3_build.LIB_DIR)
    open(of3_build.HOST_PATH, "w").close()  # of an earlier build
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
    assert of3_build.is_built() and not os.path.exists(of3_build.HOST_PATH)
