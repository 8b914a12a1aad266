"""CPU: the pool of device blocks (ornithology_amd/csrc/oh_pool.h) over a made-up
device: which blocks serve which sizes, its bounds, what is given back first,
and the second try of an allocation that fails."""
import shutil
import subprocess

import pytest

import clibs

CHECKS = ("fit", "unusable_bytes", "unusable_blocks", "bounds", "share", "asking", "owners", "threads", "retry", "other_pools")


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    if not shutil.which("g++"):
        pytest.skip("no g++")
    out = tmp_path_factory.mktemp("pool") / "pool_check"
    r = subprocess.run(["g++", "-std=c++17", "-Wall", "-Wextra", "-Werror", "-O1", f"-I{clibs.ROOT / 'ornithology_amd' / 'csrc'}",
                        str(clibs.ROOT / "tests" / "pool_check.cpp"), "-o", str(out), "-pthread"], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    return out


@pytest.mark.parametrize("check", CHECKS)
def test_pool(program, check):
    r = subprocess.run([str(program), check], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
