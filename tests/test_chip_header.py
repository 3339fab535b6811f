"""CPU checks of include/cup2d_chip.h: valid in C and C++, every function exported and bound."""

import ctypes
import os
import re
import subprocess

import pytest

from cup2d_amd import _lib

INCLUDE = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "include")


def test_functions_are_exported_and_bound():
    txt = re.sub(r"/\*.*?\*/", "", open(os.path.join(INCLUDE, "cup2d_chip.h")).read(), flags=re.S)
    names = set(re.findall(r"\b(cup2d_\w+)\s*\(", txt))
    lib = ctypes.CDLL(_lib.LIB_PATH)
    assert len(names) == 4 and names == set(_lib.CHIP_SIGNATURES)
    assert all(hasattr(lib, n) for n in names)


@pytest.mark.parametrize("cmd", [["gcc", "-std=c99", "-x", "c"], ["g++", "-std=c++17", "-x", "c++"]])
def test_header_compiles(cmd, tmp_path):
    src = tmp_path / "t"
    src.write_text('#include "cup2d_chip.h"\nint main(void) { return cup2d_ps_on_chip(0); }\n')
    r = subprocess.run(cmd + ["-Wall", "-Wextra", "-Werror", "-pedantic", "-fsyntax-only", "-I", INCLUDE, str(src)],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr


def test_without_a_handle():
    lib = _lib.load()
    assert lib.cup2d_ps_on_chip(None) == 0 and lib.cup2d_psb_on_chip(None) == 0
    assert lib.cup2d_ps_set_on_chip(None, 0, 0) == 1 and lib.cup2d_psb_set_on_chip(None, 0, 0) == 1  # EINVAL
