"""CPU: the host extension and the kernels' library belong together: an extension compiled from
another version of the header is refused when it is bound, and a build that fails leaves both files
as they were."""

import subprocess
from types import SimpleNamespace

import pytest

import testt_amd
from testt_amd import _ext, build_ext


@pytest.mark.parametrize("ext", [
    SimpleNamespace(__file__="old.so", abi_version=lambda: _ext.ABI_VERSION - 1),
    SimpleNamespace(__file__="older.so")])
def test_extension_of_another_version_is_refused(monkeypatch, ext):
    handle = _ext.load_library(_ext.library_path())
    bound = []
    ext.bind = lambda name, address: bound.append(name) or True
    ext.set_status = lambda *a: None
    monkeypatch.setattr(testt_amd, "_soupk_host", ext, raising=False)
    monkeypatch.setattr(_ext, "_entry", {})
    monkeypatch.setattr(_ext, "_host", None)
    with pytest.raises(_ext.SoupkError, match="rebuild"):
        _ext._bind_host(handle)
    assert not bound and not _ext._entry and _ext._host is None


def test_built_extension_has_the_version():
    assert _ext.host().abi_version() == _ext.ABI_VERSION


def test_failed_link_replaces_neither_file(monkeypatch, tmp_path):
    lib, host = tmp_path / "libsoupk.so", tmp_path / "_soupk_host.so"
    lib.write_text("old"), host.write_text("old")
    monkeypatch.setattr(build_ext, "LIB_PATH", str(lib))
    monkeypatch.setattr(build_ext, "HOST_PATH", str(host))
    monkeypatch.setattr(build_ext, "BUILD", str(tmp_path / "_build"))
    monkeypatch.setattr(build_ext, "_compile", lambda hipcc, src, *a: src + ".o")
    monkeypatch.setattr(build_ext, "_hipcc", lambda: "hipcc")
    fails = [str(lib) + ".tmp"]

    def run(cmd, **_):
        out = cmd[cmd.index("-o") + 1]
        open(out, "w").write("new")
        return SimpleNamespace(returncode=int(out in fails), stderr="")

    monkeypatch.setattr(subprocess, "run", run)
    with pytest.raises(RuntimeError, match="link"):
        build_ext.build()
    assert (lib.read_text(), host.read_text()) == ("old", "old")
    fails[:] = [str(host) + ".tmp"]
    with pytest.raises(RuntimeError, match="_soupk_host"):
        build_ext.build()
    assert (lib.read_text(), host.read_text()) == ("old", "old")
    fails.clear()
    build_ext.build()
    assert (lib.read_text(), host.read_text()) == ("new", "new")
