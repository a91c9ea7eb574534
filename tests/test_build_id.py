"""The library's version names what it was built from, so a tuned launch choice is not taken over by a
build whose variants are other kernels."""
import os
import re
import shutil

import pytest

from lime_amd import _lib, build


def test_the_id_follows_the_sources_and_flags(tmp_path, monkeypatch):
    for name in ("CSRC", "INCLUDE"):
        shutil.copytree(getattr(build, name), tmp_path / name)
        monkeypatch.setattr(build, name, str(tmp_path / name))
    first = build.build_id()
    assert build.build_id() == first and build.build_id(("-g",)) != first
    with open(tmp_path / "CSRC" / "common.hpp", "a") as f:
        f.write("// changed\n")
    second = build.build_id()
    with open(tmp_path / "INCLUDE" / "lime_hip.h", "a") as f:
        f.write("\n")
    assert len({first, second, build.build_id()}) == 3


def test_the_loaded_library_names_its_build_and_the_tuning_keys_hold_it():
    if not os.path.exists(_lib.LIB_PATH):
        pytest.skip("liblime_hip.so is not built (python -m lime_amd.build)")
    from lime_amd import autotune
    version = _lib.load().lime_version().decode()
    assert re.fullmatch(r".*gfx950.* build [0-9a-f]{12}", version)
    assert autotune._version() == version
