"""The order of the build and what makes it build the extension again (build.py); nothing is compiled."""
import importlib.util
import os

import pytest

PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "spiral-s-ml-library_amd")


@pytest.fixture
def B(monkeypatch, tmp_path):
    spec = importlib.util.spec_from_file_location("spiral_build_under_test", os.path.join(PKG, "build.py"))
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    monkeypatch.setattr(mod, "OBJ", str(tmp_path))
    monkeypatch.setattr(mod, "LIB", str(tmp_path / "lib.so"))
    monkeypatch.setattr(mod, "HOST_LIB", str(tmp_path / "host.so"))
    monkeypatch.setattr(mod, "HOST_STAMP", str(tmp_path / "host.txt"))
    monkeypatch.setattr(mod, "hipcc", lambda: "hipcc")
    mod.commands = []

    def run(cmd):
        mod.commands.append(cmd)
        if cmd[0] == "g++" and mod.commands_fail:
            raise RuntimeError("command failed: g++")
        with open(cmd[cmd.index("-o") + 1], "w"):
            return ""

    mod.commands_fail = False
    monkeypatch.setattr(mod, "_run", run)
    return mod


def test_the_library_is_linked_where_the_extension_cannot_be_built(B):
    B.commands_fail = True
    with pytest.raises(RuntimeError, match=r"g\+\+"):
        B.build(force=True)
    assert any("-shared" in c and c[c.index("-o") + 1] == B.LIB for c in B.commands)


def test_another_interpreter_or_torch_builds_the_extension_again(B, monkeypatch):
    built = lambda: sum(c[0] == "g++" for c in B.commands)
    B.build(force=False)
    assert built() == 1
    B.build(force=False)
    assert built() == 1
    monkeypatch.setattr(B, "host_stamp", lambda: "another")
    B.build(force=False)
    assert built() == 2
    B.build(force=False)
    assert built() == 2
    B.build(force=True)
    assert built() == 3
