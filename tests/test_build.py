"""The build of the library and its native caller (aiter_amd/csrc/build.py)."""
import os
import types

import pytest

from aiter_amd.csrc import build


@pytest.mark.parametrize("step", ["_compile_binding", "_link_binding"])
def test_failed_binding_keeps_the_built_pair(step, tmp_path, monkeypatch):
    """A binding that does not compile or link leaves the library of the build
    before in place: the two are replaced together."""
    for name in ("LIB", "NATIVE"):
        path = tmp_path / os.path.basename(getattr(build, name))
        path.write_text("before")
        monkeypatch.setattr(build, name, str(path))
    monkeypatch.setattr(build, "PKG", str(tmp_path))
    monkeypatch.setattr(build, "_compile", lambda src, out_dir: (src + ".o", {}))
    monkeypatch.setattr(build, "_compile_binding", lambda out_dir: "binding.o")

    def link(cmd, **kw):
        with open(cmd[cmd.index("-o") + 1], "w") as f:
            f.write("new")
        return types.SimpleNamespace(returncode=0, stderr="")

    def fails(*a):
        raise RuntimeError("no")

    monkeypatch.setattr(build.subprocess, "run", link)
    monkeypatch.setattr(build, step, fails)
    with pytest.raises(RuntimeError):
        build.build(verbose=False)
    assert open(build.LIB).read() == open(build.NATIVE).read() == "before"
