"""The C boundary's version: checked when the library is loaded, raised with every change of a prototype (CPU)."""

import hashlib
import os
import re

import pytest

from tace_amd import _native

HEADER = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "include", "tace_hip.h")


def _prototypes():
    """(functions, constants but the version) as declared."""
    txt = re.sub(r"/\*.*?\*/", "", open(HEADER).read(), flags=re.S)
    consts = [re.sub(r"\s+", " ", c).strip() for c in re.findall(r"^#define (TACE_\w+ .+)$", txt, flags=re.M)]
    code = re.sub(r'^\s*#.*$|extern "C" \{', "", txt, flags=re.M)
    found = re.findall(r"([\w\s\*]+?\btace_\w+\s*\([^)]*\))\s*;", code)
    return (sorted(re.sub(r"\s+", " ", f).strip() for f in found),
            sorted(c for c in consts if "ABI_VERSION" not in c))


def test_version_names_these_prototypes():
    """A changed prototype or constant needs another version: raise TACE_HIP_ABI_VERSION
    and ``_native.ABI_VERSION``, then write both values here."""
    protos, consts = _prototypes()
    assert len(protos) == len(_native.EXPORTED)
    version = int(re.search(r"TACE_HIP_ABI_VERSION (\d+)", open(HEADER).read()).group(1))
    digest = hashlib.sha256("\n".join(protos + consts).encode()).hexdigest()[:16]
    assert (version, digest) == (34, "55ce2814a4aa3fee")
    assert _native.ABI_VERSION == version


def test_library_of_another_version_is_refused(monkeypatch):
    monkeypatch.setattr(_native, "_lib", None)
    monkeypatch.setattr(_native, "ABI_VERSION", _native.ABI_VERSION - 1)
    with pytest.raises(_native.NativeError, match="ABI version"):
        _native.lib()
    assert _native._lib is None
