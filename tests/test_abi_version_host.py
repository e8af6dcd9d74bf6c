"""The version of the C ABI (CPU only): header, library and Python loader state the same one, and
it stands for the layout of the structs, so that a program built on another is told."""
import ctypes
import os
import re
import subprocess

import pytest

from diffrax_amd import _lib, _mlp, _sde

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "include", "diffrax_amd.h")

# sizeof of each struct by interface version; a change takes a new DFX_VERSION and a new row
SIZES = {
    200: dict(dfx_erk_problem=216, dfx_erk_io=200, dfx_erk_adjoint_io=40, dfx_sde_problem=40,
              dfx_sde_io=96, dfx_mlp_problem=200, dfx_mlp_io=144),
}
PYTHON = dict(dfx_erk_problem=_lib.ErkProblem, dfx_erk_io=_lib.ErkIO,
              dfx_erk_adjoint_io=_lib.AdjointIO, dfx_sde_problem=_sde.SdeProblem,
              dfx_sde_io=_sde.SdeIO, dfx_mlp_problem=_mlp.MlpProblem, dfx_mlp_io=_mlp.MlpIO)


def _header_version():
    return int(re.search(r"^#define DFX_VERSION (\d+)$", open(HEADER).read(), re.M).group(1))


def test_one_version():
    assert _header_version() == _lib.VERSION == _lib.load().dfx_version()


def test_a_version_has_one_layout(tmp_path):
    sizes = SIZES[_header_version()]
    src = tmp_path / "sizes.c"
    src.write_text('#include <stdio.h>\n#include "diffrax_amd.h"\nint main(void) {\n' + "".join(
        f'  printf("{n} %zu\\n", sizeof({n}));\n' for n in sizes) + "  return 0;\n}\n")
    exe = str(tmp_path / "sizes")
    subprocess.run(["gcc", "-I", os.path.dirname(HEADER), str(src), "-o", exe], check=True)
    out = subprocess.run([exe], check=True, capture_output=True, text=True).stdout
    found = {n: int(s) for n, s in (line.split() for line in out.splitlines())}
    assert found == sizes
    assert {n: ctypes.sizeof(PYTHON[n]) for n in sizes} == sizes


def test_loader_refuses_another_version(monkeypatch):
    monkeypatch.setattr(_lib, "_lib", None)
    monkeypatch.setattr(_lib, "VERSION", _lib.VERSION + 100)
    with pytest.raises(_lib.LibraryMissing, match="version"):
        _lib.load()
