"""The engine's host code on the CPU: tests/cpp/alloc_host.cpp defines the HIP calls that
the library makes, refuses memory where the test wants it and counts launches."""
import os
import subprocess

import pytest

from tomokvas_amd import build

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
PKG = os.path.join(ROOT, "tomokvas_amd")


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("alloc") / "alloc_host")
    # -rdynamic: the library's HIP calls bind to the program's
    cmd = [build.hipcc(), "-O1", "-std=c++17", "-Wall", "-rdynamic",
           "-I", os.path.join(ROOT, "include"), os.path.join(HERE, "cpp", "alloc_host.cpp"), "-o", out, "-L", PKG,
           "-l:libtomokvas_fdk.so", "-Wl,-rpath," + PKG, "-Wl,--allow-shlib-undefined"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-4000:]
    return out


@pytest.mark.parametrize("mode", ["stack", "filtered"])
def test_storage_that_cannot_be_allocated(exe, mode):
    r = subprocess.run([exe, mode], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr[-2000:]


def test_storage_grows_on_the_context_s_device(exe):
    r = subprocess.run([exe, "device"], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr[-2000:]


def test_filter_into_overlapping_buffers(exe):
    r = subprocess.run([exe, "overlap"], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr[-2000:]


def test_angle_block_budget_is_what_the_engine_holds(exe):
    r = subprocess.run([exe, "budget"], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr[-2000:]
