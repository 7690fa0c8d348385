"""The order of one handle's calls across streams (csrc/streamorder.h), on a
simulated device: whatever streams the handle is bound to, each operation starts
after every earlier one, and freeing the handle waits for all of them."""
from __future__ import annotations

import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]


@pytest.fixture(scope="module")
def sim(tmp_path_factory):
    cxx = shutil.which("g++")
    assert cxx, "the C++ compiler of the build is missing"
    exe = tmp_path_factory.mktemp("order") / "stream_order"
    subprocess.run([cxx, "-std=c++17", "-O1", "-Wall", "-Werror", f"-I{ROOT / 'sunnynet_amd' / 'csrc'}",
                    str(ROOT / "tests" / "cpp" / "stream_order.cpp"), "-o", str(exe)], check=True)

    def run(script):
        r = subprocess.run([str(exe)], input=script.replace(";", "\n"), capture_output=True, text=True, check=True,
                           timeout=20)
        return r.stdout.split("\n")[:-1]
    return run


def _ordered(lines):
    return all(x.split()[1] == "1" and x.split()[0] != "error" for x in lines)


@pytest.mark.parametrize("script", [
    "bind A;async;bind B;async;bind A;async;free",
    # bound in between to a stream on which nothing, or nothing that marks, runs
    "bind A;async;bind B;bind C;async;free",
    "bind A;async;bind B;bind C;bind D;async;bind B;async;free",
    # freed on the third stream
    "bind A;async;bind B;bind C;free",
    "bind A;async;async;bind B;bind A;bind C;async;free",
    # one handle value, several streams: the per-thread stream
    "bind P;thread 1;async;thread 2;async;thread 1;async;free",
])
def test_every_stream_waits(sim, script):
    assert _ordered(sim(script)), script


def test_capture_keeps_the_mark(sim):
    # a call captured on B marks nothing; the work on A is still waited for
    assert _ordered(sim("bind A;async;bind B;capture B;async;endcapture B;bind C;async;free"))


def test_capture_waits_on_the_host(sim):
    # the capturing stream cannot wait for A's event; what it captures is
    # replayed later, on any stream, after the work that the handle had running
    assert _ordered(sim("bind A;async;capture B;bind B;async;endcapture B;quiet;free"))
