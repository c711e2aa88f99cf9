"""The ahead-of-time build: what it leaves beside the target."""

from __future__ import annotations

import os
import shutil
import stat
import subprocess

import pytest

from deformops_amd import _build


@pytest.mark.parametrize("umask", [0o022, 0o027])
def test_a_built_library_is_readable_as_the_umask_says(tmp_path, umask):
    compiler = shutil.which("g++")
    if compiler is None:
        pytest.skip("no host compiler")
    source = tmp_path / "one.cpp"
    source.write_text('extern "C" int one() { return 1; }\n')
    target = tmp_path / "lib" / "libone.so"
    previous = os.umask(umask)
    try:
        for _ in range(2):  # also in the place of an older build
            assert _build._compile([compiler, "-shared", "-fPIC", str(source)], target, verbose=False) == target
    finally:
        os.umask(previous)
    assert stat.S_IMODE(target.stat().st_mode) == 0o777 & ~umask
    assert [p.name for p in target.parent.iterdir()] == ["libone.so"]


def test_a_failed_build_keeps_the_library_that_is_there(tmp_path):
    target = tmp_path / "libone.so"
    target.write_bytes(b"older")
    with pytest.raises(subprocess.CalledProcessError):
        _build._compile([shutil.which("false") or "false"], target, verbose=False)
    assert target.read_bytes() == b"older" and [p.name for p in tmp_path.iterdir()] == ["libone.so"]
