"""The C interface and its version, CPU only: the headers without their comments (entry points, structs, constants) are
those of the version the package expects, so that a library of another interface is refused by its version (hip.load) and
not by a missing symbol or a struct read wrongly. A change of the interface takes a new version and its digest here."""

import hashlib
import re
import subprocess
from pathlib import Path

import pytest

from blochparty_amd.engines import hip

INCLUDE = Path(__file__).resolve().parent.parent / "include"
DIGESTS = {26: "60bf95f834f76b87"}


def interface() -> str:
    text = "\n".join(p.read_text() for p in sorted(INCLUDE.glob("*.h")))
    return " ".join(re.sub(r"/\*.*?\*/|//[^\n]*", " ", text, flags=re.S).split())


def test_the_interface_has_its_own_version():
    digest = hashlib.sha256(interface().encode()).hexdigest()[:16]
    assert DIGESTS[hip.ABI_VERSION] == digest


def test_the_library_has_the_version():
    assert hip.load().hb_abi_version() == hip.ABI_VERSION


def test_an_older_library_is_refused_by_its_version(tmp_path, monkeypatch):
    (tmp_path / "old.c").write_text("int hb_abi_version(void) { return 25; }\n")
    subprocess.run(["gcc", "-shared", "-fPIC", "-o", str(tmp_path / "old.so"), str(tmp_path / "old.c")], check=True)
    monkeypatch.setattr(hip, "LIB_PATH", tmp_path / "old.so")
    monkeypatch.setattr(hip, "_LIB", None)
    with pytest.raises(RuntimeError, match="has ABI 25, expected"):
        hip.load()
