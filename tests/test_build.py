"""The incremental build's rule for recompiling a unit (no compiler run)."""
import os

import pytest

from lible_amd import build


@pytest.fixture
def unit(tmp_path, monkeypatch):
    """A source with an object, dependency list and command line as a compilation leaves them."""
    monkeypatch.setattr(build, "hipcc", lambda: "hipcc")
    monkeypatch.setattr(build, "ROOT", str(tmp_path))
    monkeypatch.setattr(build, "CSRC", str(tmp_path))
    src, header, obj = (str(tmp_path / n) for n in ("a.hip", "a.hpp", "a.o"))
    defines = ["-DLBX_UNIT=5", "-DLBX_NPARTS=5", "-DLBX_PART=3"]

    def run(cmd, **kw):
        for p, text in ((obj, ""), (obj + ".d", f"{obj}: {src} \\\n {header}\n")):
            with open(p, "w") as f:
                f.write(text)
        return type("Result", (), {"returncode": 0})

    for p in (src, header):
        with open(p, "w") as f:
            f.write("")
        os.utime(p, (1, 1))
    monkeypatch.setattr(build.subprocess, "run", run)
    assert build._stale(src, obj, defines)
    build._compile(src, obj, defines)
    return src, header, obj, defines


def test_unchanged_unit_is_kept(unit):
    src, _, obj, defines = unit
    assert not build._stale(src, obj, defines)


@pytest.mark.parametrize("which", [0, 1])
def test_newer_source_or_header(unit, which):
    os.utime(unit[which], None)
    os.utime(unit[2], (2, 2))
    assert build._stale(unit[0], unit[2], unit[3])


def test_other_flags_or_parts(unit, monkeypatch):
    src, _, obj, defines = unit
    assert build._stale(src, obj, [d.replace("NPARTS=5", "NPARTS=4") for d in defines])
    monkeypatch.setattr(build, "FLAGS", build.FLAGS + ["-mllvm", "-x"])
    assert build._stale(src, obj, defines)
