"""What the package's build entry points produce, with the compilers taken out."""

import os
import runpy

import pytest


def test_the_packages_build_makes_the_library_and_the_launchers(monkeypatch):
    """Every hot call needs both: a build that leaves out the launchers makes a clean tree unusable, and in a built one
    leaves launchers compiled against an earlier header beside a new library."""
    import wdl
    import wdl.build as module

    made = []
    monkeypatch.setattr(module, "build", lambda force=False: made.append(("libwdl", force)) or module.LIB)
    monkeypatch.setattr(module, "build_host", lambda force=False: made.append(("wdl_host", force)) or module.HOST)
    build = runpy.run_path(wdl.__file__)["build"]
    assert build() == module.LIB and made == [("libwdl", False), ("wdl_host", False)]
    made.clear()
    build(force=True)
    assert made == [("libwdl", True), ("wdl_host", True)]


@pytest.mark.parametrize("newer", [None, "source", "header", "force"])
def test_launchers_are_compiled_when_older_than_what_they_are_made_of(monkeypatch, tmp_path, newer):
    import wdl.build as module

    files = {name: tmp_path / name for name in ("source", "header", "so")}
    for at, name in enumerate(files):
        files[name].write_text("")
        os.utime(files[name], (at, at))
    if newer in files:
        os.utime(files[newer], (9, 9))
    monkeypatch.setattr(module, "HOST", files["so"])
    monkeypatch.setattr(module, "HOST_SRC", files["source"])
    monkeypatch.setattr(module, "HEADER", files["header"])
    ran = []

    def run(cmd, **_):
        ran.append(cmd)
        (tmp_path / "so.so.tmp").write_text("")
        return type("Done", (), dict(returncode=0))

    monkeypatch.setattr(module.subprocess, "run", run)
    assert module.build_host(force=newer == "force") == files["so"]
    assert len(ran) == (newer is not None)
