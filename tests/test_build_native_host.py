"""What the build script makes with torch, without it and where its C++ part does not compile."""

import sys
from pathlib import Path

import pytest
import torch

sys.path.insert(0, str(Path(__file__).resolve().parent.parent / "primus-turbo_amd"))
import build_native  # noqa: E402


def _tool(path, body):
    path.write_text("#!/bin/sh\n" + body)
    path.chmod(0o755)
    return str(path)


# (stands for hipcc and g++: the word behind -o names the file to write, the assembly of a unit beside it)
_COMPILES = """while [ "$1" != -o ]; do shift; done; : > "$2"
case "$2" in *.o) cp "$ASM" "${2%.o}-hip-amdgcn-amd-amdhsa-gfx950.s";; esac
"""


@pytest.fixture
def tree(tmp_path, monkeypatch):
    src = tmp_path / "csrc"
    src.mkdir()
    for name in ("one.hip", "two.hip", "a.h", "torch_ops.cpp"):
        (src / name).write_text("")
    for name, path in dict(CSRC=src, BUILD=tmp_path / "build", LIBDIR=tmp_path / "lib", HEADER=src / "a.h").items():
        monkeypatch.setattr(build_native, name, path)
    (tmp_path / "asm").write_text("")
    monkeypatch.setenv("ASM", str(tmp_path / "asm"))
    monkeypatch.setenv("HIPCC", _tool(tmp_path / "hipcc", _COMPILES))
    monkeypatch.setenv("CXX", _tool(tmp_path / "cxx", _COMPILES))
    return tmp_path


def _libs(tree):
    return sorted(p.name for p in (tree / "lib").iterdir())


TORCH_LIB = f"libprimus_turbo_torch-{torch.__version__}.so"


def test_both_libraries(tree):
    from primus_turbo import _native

    assert build_native.ensure_built() == tree / "lib" / build_native.LIBNAME
    assert _libs(tree) == sorted([build_native.LIBNAME, TORCH_LIB])
    assert _native.TORCH_LIB_PATH.name == TORCH_LIB


def test_without_torch(tree, monkeypatch):
    real = build_native.importlib.util.find_spec
    monkeypatch.setattr(build_native.importlib.util, "find_spec", lambda name, *a: None if name == "torch" else real(name, *a))
    build_native.ensure_built()
    assert _libs(tree) == [build_native.LIBNAME]


def test_torch_part_does_not_compile(tree, monkeypatch):
    monkeypatch.setenv("CXX", _tool(tree / "cxx", "echo no headers >&2; exit 1\n"))
    with pytest.raises(RuntimeError, match="torch_ops.cpp failed:\nno headers"):
        build_native.build()
    assert _libs(tree) == [build_native.LIBNAME]


def test_library_of_another_torch(tree, monkeypatch):
    """Neither taken for the installed one's nor overwritten."""
    build_native.build()
    monkeypatch.setattr(torch, "__version__", "0.0")
    build_native.ensure_built()
    assert _libs(tree) == sorted([build_native.LIBNAME, TORCH_LIB, "libprimus_turbo_torch-0.0.so"])


def test_unsafe_assembly(tree):
    """A copy right behind a VALU write of its descriptor fails the build and leaves no object behind."""
    (tree / "asm").write_text("_Z1k:\n\tv_readlane_b32 s1, v2, 0\n\t;;#ASMSTART\n\ts_add_u32 m0, s4, 16\n\ts_nop 0\n"
                              "\tbuffer_load_dword v1, s[0:3], 0 offen lds\n\t;;#ASMEND\n.Lfunc_end0:\n")
    with pytest.raises(RuntimeError, match="_Z1k: 1 unsafe uses"):
        build_native.build()
    assert not list((tree / "build").iterdir()) and not (tree / "lib" / build_native.LIBNAME).exists()
