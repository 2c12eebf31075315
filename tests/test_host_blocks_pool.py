"""The pool of device blocks that calls on host memory keep, on the CPU over a HIP
that only counts: which calls allocate, what stays held, and that idle blocks never
stand in the way of another allocation."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
MB = 1 << 20


@pytest.fixture(scope="module")
def pool(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("pool") / "pool")
    cxx = os.environ.get("CXX") or shutil.which("g++") or shutil.which("c++")
    assert cxx, "a host C++ compiler"
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    subprocess.run([cxx, "-O1", "-std=c++17", "-pthread", "-w", "-D__HIP_PLATFORM_AMD__", "-I", os.path.join(rocm, "include"),
                    os.path.join(HERE, "host_blocks_host.cpp"), os.path.join(ROOT, "zml_amd", "csrc", "runtime.cpp"),
                    "-o", exe], check=True)

    def run(*commands):
        r = subprocess.run([exe], input="\n".join(commands) + "\n", capture_output=True, text=True, timeout=20)
        assert r.returncode == 0, r.stdout
        return [tuple(map(int, line.split())) for line in r.stdout.splitlines()]
    return run


@pytest.mark.parametrize("others", ["", f" {64 << 10}", f" {64 << 10} {200 << 10}"])
def test_growing_calls_keep_their_own_blocks(pool, others):
    """Calls of one to three blocks, one of them larger every time: the sizes in use are
    kept, however many smaller ones came before, and no more than eight blocks of 16 MiB."""
    for made in range(1, 16):
        out = pool(*(f"call {k * MB}{others}" for k in range(1, made + 1)), *[f"call {made * MB}{others}"] * 3)
        assert [o[0] for o in out[-3:]] == [0, 0, 0], made
        assert all(o[2] <= 8 * 16 * MB for o in out)


def test_many_blocks_at_once_stay_bounded(pool):
    out = pool("call " + " ".join(str(k * MB) for k in range(1, 17)), f"call {17 * MB}", f"call {9 * MB} {16 * MB}")
    assert out[0][2] <= 8 * 16 * MB
    assert out[1][:2] == (1, 1)          # above the size that is kept: made and freed
    assert out[2][0] == 0                # the largest ones were kept


def test_idle_blocks_make_room_for_a_workspace(pool):
    fill = "call " + " ".join([str(16 * MB)] * 8)
    out = pool(f"room {200 * MB}", fill, f"ws 3 {150 * MB}", f"ws 3 {150 * MB}", f"call {16 * MB}", f"ws 4 {60 * MB}")
    assert out[1][2] == 128 * MB
    assert out[2][3] == 0 and out[2][2] == 150 * MB
    assert out[3][0] == 0
    assert out[4][3] == 0
    assert out[5][3] == 1                # really no room: it fails
    out = pool(f"room {200 * MB}", fill, f"call {150 * MB}")
    assert out[2][3] == 0
