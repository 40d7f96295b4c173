"""The version by which a stale compiled library is refused."""

from __future__ import annotations

import hashlib
import re
from pathlib import Path

import pytest

from mini_infer_amd.exceptions import ExtensionMissingError
from mini_infer_amd.ops import library

# version -> digest of every entry point's argument types
DIGESTS = {37: "19d70346842e0dd7", 38: "5f985cd6095e4c7f", 39: "18d3fc0198a35211", 40: "6851cd991bfce4b8", 41: "9803e53b3110fced", 42: "d01bdc89bd271a04", 43: "613ab1a77867ce37", 44: "2a63e0010ae073e1",
           45: "f6d5abd47b7311f0", 46: "bc507a4251d57fa7", 47: "eefedaa760aa714e", 48: "8e751a64dde672ba", 49: "550e0b8ef907056e",
           50: "80c3c74b33a8dc1c", 51: "60445bc43334f58b", 52: "4d1ac4af3a9083a1", 53: "2bbae5280632fa47", 54: "146144b8444c2820", 55: "21fcb354686890c1", 56: "1165b637a929ca89"}


def test_the_version_changes_with_the_arguments():
    """If this fails: raise the version in library.py and runtime.hip, and add the new digest here."""
    text = ";".join(f"{name}:{','.join(t.__name__ for t in types)}" for name, types in sorted(library._SIGNATURES.items()))
    assert DIGESTS.get(library.ABI_VERSION) == hashlib.sha256(text.encode()).hexdigest()[:16]


def test_both_sides_name_the_same_version():
    source = (Path(library.__file__).parent.parent / "csrc" / "runtime.hip").read_text()
    assert re.findall(r"int mi_abi_version\(\) \{ return (\d+); \}", source) == [str(library.ABI_VERSION)]


def test_a_library_of_another_version_is_refused_before_its_functions_are_looked_up():
    class Stale:
        def __getattr__(self, name):
            raise AttributeError(name)

        def mi_abi_version(self):
            return library.ABI_VERSION - 1

    with pytest.raises(ExtensionMissingError, match="rebuild it"):
        library._declare(Stale(), Path("stale.so"))
