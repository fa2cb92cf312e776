"""What a new sampler and a new output slice leave in and take of device memory,
on the CPU: tests/c/test_workspace_create.c stands in for the HIP calls of
create."""
import subprocess
from pathlib import Path

import pytest

import fg_hip

ROOT = Path(__file__).resolve().parent.parent


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    lib = Path(fg_hip.load_library()._name)
    exe = tmp_path_factory.mktemp("workspace") / "test_workspace_create"
    subprocess.run(["gcc", "-std=c17", "-O1", "-Wall", "-Wextra", "-Werror", "-rdynamic",
                    f"-I{ROOT / 'include'}", "-o", str(exe),
                    str(ROOT / "tests" / "c" / "test_workspace_create.c"), str(lib),
                    f"-Wl,-rpath,{lib.parent}", "-Wl,--allow-shlib-undefined"], check=True)
    return exe


def test_hand_off_words_start_cleared(program):
    r = subprocess.run([program], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr


def test_slice_workspace(program):
    """A whole-head slice holds 64 tokens' logits in 64 MB at most, and takes
    fewer when memory is short."""
    r = subprocess.run([program, "slice"], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
