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


def test_binding_for_a_torch_without_the_newer_types(tmp_path):
    """The element types that the Python side takes only where torch has them
    are optional in the native caller too."""
    old = types.SimpleNamespace(__version__="2.6.0")
    assert build.binding_defines(old)[1:] == ["-DAITER_AMD_TORCH_E8M0=0", "-DAITER_AMD_TORCH_FP4=0"]
    text = open(os.path.join(build.HERE, "binding.cpp")).read()
    for name, macro in (("kFloat8_e8m0fnu", "AITER_AMD_TORCH_E8M0"), ("kFloat4_e2m1fn_x2", "AITER_AMD_TORCH_FP4")):
        assert [part.split("#endif")[0].count(name) for part in text.split(f"#if {macro}\n")[1:]] == [1]
        assert text.count(name) == 1
