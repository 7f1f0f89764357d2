"""The kernel library and its header: which library is taken, and what the others are told (no GPU)."""

import re
import subprocess

import pytest

from flyweight_amd.kernels import build, ops


def _library(tmp_path, number: int) -> str:
    """A library that knows its interface number and none of the kernels."""
    source, path = tmp_path / "old.cpp", tmp_path / "libold.so"
    source.write_text('extern "C" int fw_abi_version(void) { return %d; }\n'
                      'extern "C" const char* fw_last_error(void) { return ""; }\n' % number)
    subprocess.run(["g++", "-shared", "-fPIC", "-o", str(path), str(source)], check=True)
    return str(path)


def test_a_library_of_another_interface_is_named_as_such(tmp_path, monkeypatch):
    """``ensure_built`` hands out an older library where none can be built: it lacks entry points of the present header,
    and the message has to say that it is to be built again."""
    path = _library(tmp_path, 18)
    monkeypatch.setattr(ops, "_lib", None)
    monkeypatch.setattr(ops, "_profiled", None)
    monkeypatch.setattr(build, "ensure_built", lambda: path)
    with pytest.raises(ops.KernelError, match="rebuild it"):
        ops.library()
    assert ops._lib is None


def test_the_interface_number_follows_the_declarations():
    """A signature cannot change without the number: it is formed from the header's declarations, and from them alone."""
    with open(build.HEADER, "r", encoding="utf-8") as handle:
        header = handle.read()
    number = build.abi_version(header)
    assert number == build.abi_version() and 0 < number < 1 << 31
    assert number == build.abi_version(re.sub(r"//[^\n]*", "", header) + "\n// a remark\n")
    assert number != build.abi_version(header.replace("int slots, int spread, void* stream", "int slots, void* stream"))
    assert number != build.abi_version(header.replace("float eps", "long long eps", 1))
    assert f"-DFW_ABI_VERSION={number}" in build.compile_flags()
