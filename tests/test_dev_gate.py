"""The gate that keeps two grid-synchronizing kernels off one device
(csrc/devgate.h), in threads and processes."""
from __future__ import annotations

import os
import shutil
import signal
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    cxx = shutil.which("g++")
    assert cxx, "the C++ compiler of the build is missing"
    out = tmp_path_factory.mktemp("gate") / "dev_gate"
    subprocess.run([cxx, "-std=c++17", "-O1", "-Wall", "-Werror", "-pthread",
                    f"-I{ROOT / 'sunnynet_amd' / 'csrc'}", str(ROOT / "tests" / "cpp" / "dev_gate.cpp"),
                    "-o", str(out)], check=True)
    return str(out)


def _run(*args, **kw):
    return subprocess.run([str(a) for a in args], capture_output=True, text=True, timeout=60, **kw)


@pytest.mark.parametrize("procs,threads", [(1, 4), (3, 1), (2, 2)])
def test_one_at_a_time(exe, tmp_path, procs, threads):
    counter = tmp_path / "n"
    counter.write_text("0\n")
    ps = [subprocess.Popen([exe, "excl", tmp_path / "gate", str(threads), "60", counter]) for _ in range(procs)]
    assert [p.wait(60) for p in ps] == [0] * procs
    assert int(counter.read_text()) == procs * threads * 60


def test_callers_in_loops_take_turns(exe, tmp_path):
    ps = [subprocess.Popen([exe, "loop", tmp_path / "gate", "1.5"], stdout=subprocess.PIPE, text=True)
          for _ in range(2)]
    n = [int(p.communicate(timeout=60)[0]) for p in ps]
    assert min(n) > 100 and max(n) < 2 * min(n), n


def test_a_killed_holder_lets_go(exe, tmp_path):
    p = subprocess.Popen([exe, "hold", tmp_path / "gate", "30"], stdout=subprocess.PIPE, text=True)
    assert p.stdout.readline() == "in\n"
    p.send_signal(signal.SIGKILL)
    p.wait(20)
    assert _run(exe, "try", tmp_path / "gate", 10).stdout.split()[0] == "1"


def test_a_stuck_holder_is_waited_for_once(exe, tmp_path):
    """Up to the limit, and not again until it has let go."""
    p = subprocess.Popen([exe, "hold", tmp_path / "gate", "20"], stdout=subprocess.PIPE, text=True)
    assert p.stdout.readline() == "in\n"
    q = subprocess.Popen([exe, "try", tmp_path / "gate", "0.3", "4", "0.5"], stdout=subprocess.PIPE, text=True)
    tries = [q.stdout.readline().split() for _ in range(2)]
    p.kill()
    p.wait(20)
    tries += [x.split() for x in q.communicate(timeout=20)[0].splitlines()]
    assert [x[0] for x in tries] == ["0", "0", "1", "1"]
    assert 0.25 < float(tries[0][1]) < 5 and all(float(x[1]) < 0.2 for x in tries[1:])


@pytest.mark.parametrize("what", ["no folder", "a folder", "a fifo", "a link"])
def test_unusable_files(exe, tmp_path, what):
    path = tmp_path / ("missing/gate" if what == "no folder" else "gate")
    if what == "a folder":
        path.mkdir()
    elif what == "a fifo":
        os.mkfifo(path)
    elif what == "a link":
        (tmp_path / "there").write_text("")
        path.symlink_to(tmp_path / "there")
    ok, took = _run(exe, "try", path, 10).stdout.split()
    assert ok == "0" and float(took) < 1


def test_another_users_files_will_do(exe, tmp_path):
    for f in ("gate", "gate.next"):
        (tmp_path / f).write_text("")
        (tmp_path / f).chmod(0o444)
    assert _run(exe, "try", tmp_path / "gate", 10).stdout.split()[0] == "1"
    assert _run(exe, "try", tmp_path / "new", 10, umask=0o077).stdout.split()[0] == "1"
    assert all((tmp_path / f).stat().st_mode & 0o777 == 0o444 for f in ("new", "new.next"))
