"""Steps on the caller's streams: two handles stepped from two threads on two
streams at once give what each gives alone (their persistent kernels must not
share the device), and a handle that moves between streams goes on from its state,
also while its earlier calls are still running."""
from __future__ import annotations

import ctypes
import fcntl
import subprocess
import sys
import threading
import time
from concurrent.futures import ThreadPoolExecutor
from pathlib import Path

import numpy as np
import pytest
import torch

from sunnynet_amd import _native
from sunnynet_amd.blob import pack_sunny_blob
from sunnynet_amd.config import SMALL
from sunnynet_amd.runtime.model import HipModel
from sunnynet_amd.runtime.rwkv7 import HipRwkv7
from sunnynet_amd.rwkv7 import RWKV_TINY, init_rwkv7, pack_rwkv7_blob
from sunnynet_amd.weights import init_sunnynet

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def paths(tmp_path_factory):
    d = tmp_path_factory.mktemp("streams")
    (d / "s.bin").write_bytes(pack_sunny_blob(init_sunnynet(SMALL, 0)))
    (d / "r.bin").write_bytes(pack_rwkv7_blob(init_rwkv7(RWKV_TINY, 2)))
    return d / "s.bin", d / "r.bin"


def _make(kind, paths):
    if kind.startswith("rwkv"):
        return HipRwkv7(paths[1], max_batch=int(kind[4:]))
    c = SMALL
    B = {"sunny1": 1, "sunny4": 4, "sunny20": 20}[kind]
    return HipModel(paths[0], c.vocab_size, c.dim, c.inner, c.rank, c.taps, c.layers, max_batch=B)


def _run(h, kind, n, streams):
    B, V = h.max_batch, h.vocab
    rng = np.random.default_rng(5)
    out = []
    for i in range(n):
        with torch.cuda.stream(streams[i % len(streams)]):
            t = torch.from_numpy(rng.integers(0, V, B).astype(np.int32)).cuda()
            out.append(h.step_batch(t).cpu())
    return out


@pytest.mark.parametrize("a,b", [("sunny1", "rwkv1"), ("sunny4", "sunny20"), ("sunny1", "sunny20")])
def test_two_threads_two_streams(gpu, paths, a, b):
    print("two threads, two streams:", a, b, flush=True)
    n = 24
    alone = {}
    for k in (a, b):
        h = _make(k, paths)
        alone[k] = _run(h, k, n, [torch.cuda.current_stream()])
        h.close()
    got, errs = {}, []

    def work(k):
        try:
            h = _make(k, paths)
            got[k] = _run(h, k, n, [torch.cuda.Stream()])
            h.close()
        except Exception as e:      # reported below: a thread's exception is lost
            errs.append(e)

    ts = [threading.Thread(target=work, args=(k,)) for k in (a, b)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not errs, errs
    for k in (a, b):
        assert all(torch.equal(x, y) for x, y in zip(got[k], alone[k])), k


@pytest.mark.parametrize("kind", ["sunny1", "sunny4", "rwkv1", "rwkv12"])
def test_moves_between_streams(gpu, paths, kind):
    print("steps alternating between two streams:", kind, flush=True)
    h = _make(kind, paths)
    ref = _run(h, kind, 6, [torch.cuda.current_stream()])
    h.reset()
    got = _run(h, kind, 6, [torch.cuda.Stream(), torch.cuda.current_stream(), torch.cuda.Stream()])
    assert all(torch.equal(x, y) for x, y in zip(got, ref))


def _calls(h, kind, toks, streams, between):
    """A chain of calls, each on the next of `streams`, none waited for. `between`
    binds the handle to one more stream before each call: with a read of the state
    (which only copies), or with nothing."""
    keep, i = [], 0

    def on(f):
        nonlocal i
        with torch.cuda.stream(streams[i % len(streams)]):
            keep.append(f())
        i += 1

    for t in toks:
        if between == "state":
            on(lambda: h.get_state(h.max_batch))
        elif between == "bind":
            on(h._bind_stream)
        on(lambda: h.step_batch(t))
        if kind == "sunny20":
            on(lambda: h.prefill_batch(torch.stack([t, t, t, t], 1)))
            on(lambda: h.decode_greedy(t, 3))
    on(lambda: h.get_state(h.max_batch))
    return keep


@pytest.mark.parametrize("between", ["none", "bind", "state"])
@pytest.mark.parametrize("kind", ["rwkv12", "sunny20"])
def test_running_calls_move_between_streams(gpu, paths, monkeypatch, kind, between):
    """Calls that return before they are done (captured steps, prefill, captured
    greedy decoding) over three streams, synchronized once at the end."""
    print("calls in flight over three streams:", kind, between, flush=True)
    monkeypatch.setenv("SNHIP_BATCH_PERSIST", "0")    # read at load: the captured per-kernel step
    h = _make(kind, paths)
    assert kind != "sunny20" or h.batch_grid == 0
    rng = np.random.default_rng(6)
    toks = [torch.from_numpy(rng.integers(0, h.vocab, h.max_batch).astype(np.int32)).cuda() for _ in range(6)]
    _calls(h, kind, toks, [torch.cuda.current_stream()], between)     # graphs captured, workspaces there
    torch.cuda.synchronize()
    out = []
    for streams in ([torch.cuda.current_stream()], [torch.cuda.Stream() for _ in range(3)]):
        h.reset()
        out.append(_calls(h, kind, toks, streams, between))
        torch.cuda.synchronize()
    flat = [[x for r in o if r is not None for x in (r if isinstance(r, tuple) else (r,))] for o in out]
    assert len(flat[0]) == len(flat[1])
    for x, y in zip(*flat):
        assert torch.equal(x, y), kind
    h.close()


@pytest.mark.parametrize("running", [False, True])
def test_prefill_captured_on_another_stream(gpu, paths, running):
    """A prefill captured on a stream of its own, after (or while) the handle works
    on another: every replay goes on from the state as an eager call does."""
    print("prefill captured on another stream, work running:", running, flush=True)
    h, ref = _make("sunny4", paths), _make("sunny4", paths)
    rng = np.random.default_rng(7)
    toks = torch.from_numpy(rng.integers(0, h.vocab, (4, 40)).astype(np.int32)).cuda()
    side, cap = torch.cuda.Stream(), torch.cuda.Stream()
    out = [x.prefill_batch(toks) for x in (h, ref)]      # workspaces and planes are there
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=cap):
        if running:
            with torch.cuda.stream(side):
                h.prefill_batch(toks, logits=False)
        lg = h.prefill_batch(toks)
    torch.cuda.synchronize()
    if running:
        ref.prefill_batch(toks, logits=False)
    for i in range(4):
        want = ref.prefill_batch(toks)
        state = ref.get_state(4)
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(lg, want), i
        assert all(torch.equal(a, b) for a, b in zip(h.get_state(4), state)), i
    # and an eager call afterwards
    assert torch.equal(h.prefill_batch(toks), ref.prefill_batch(toks))
    assert torch.equal(out[0], out[1])
    h.close()
    ref.close()


@pytest.mark.parametrize("kind", ["rwkv12", "sunny20"])
def test_per_thread_stream_in_two_threads(gpu, paths, monkeypatch, kind):
    """One handle bound to the per-thread stream (one handle value, another stream in
    every thread), its calls alternating between two threads, none waited for."""
    print("per-thread stream, two threads:", kind, flush=True)
    monkeypatch.setenv("SNHIP_BATCH_PERSIST", "0")
    lib = _native.lib()
    step, bind = ((lib.snhip_rk_step_batch_dev, lib.snhip_rk_set_stream) if kind == "rwkv12"
                  else (lib.snhip_step_batch_dev, lib.snhip_set_stream))
    h = _make(kind, paths)
    rng = np.random.default_rng(8)
    n, B = 12, h.max_batch
    toks = torch.from_numpy(rng.integers(0, h.vocab, (n, B)).astype(np.int32)).cuda()
    out = torch.empty(2, n, B, h.vocab, device="cuda")
    per_thread = 2          # hipStreamPerThread
    h.step_batch(toks[0])   # the graph is captured
    torch.cuda.synchronize()
    for run in range(2):
        h.reset()
        _native.check(bind(h._h, per_thread if run else 0), "set_stream")
        errs = []

        def call(i):
            rc = step(h._h, toks[i].data_ptr(), B, out[run, i].data_ptr())
            if rc:
                errs.append((i, rc))
        with ThreadPoolExecutor(1) as a, ThreadPoolExecutor(1) as b:
            for i in range(n):
                (a, b)[i % 2].submit(call, i).result()
            assert not errs, errs
            torch.cuda.synchronize()
    assert torch.equal(out[0], out[1])
    h.close()


@pytest.mark.parametrize("a,b", [("sunny1", "rwkv1"), ("sunny4", "sunny20")])
def test_two_threads_per_thread_stream(gpu, paths, a, b):
    """Two handles bound to the per-thread stream, stepped from two threads at once."""
    print("two threads, per-thread streams:", a, b, flush=True)
    n, per_thread = 24, 2
    h = {k: _make(k, paths) for k in (a, b)}
    rng = np.random.default_rng(9)
    toks = {k: torch.from_numpy(rng.integers(0, h[k].vocab, (n, h[k].max_batch)).astype(np.int32)).cuda()
            for k in (a, b)}
    want = {k: torch.stack([h[k].step_batch(t) for t in toks[k]]) for k in (a, b)}
    got = {k: torch.empty_like(want[k]) for k in (a, b)}
    lib = _native.lib()
    torch.cuda.synchronize()
    errs = []

    def work(k):
        rk = "_rk" if k.startswith("rwkv") else ""
        step, bind = getattr(lib, f"snhip{rk}_step_batch_dev"), getattr(lib, f"snhip{rk}_set_stream")
        rc = bind(h[k]._h, per_thread)
        for i in range(n):
            rc = rc or step(h[k]._h, toks[k][i].data_ptr(), h[k].max_batch, got[k][i].data_ptr())
        if rc:
            errs.append((k, rc, _native.last_error()))
    for k in (a, b):
        h[k].reset()
    torch.cuda.synchronize()
    ts = [threading.Thread(target=work, args=(k,)) for k in (a, b)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    torch.cuda.synchronize()
    assert not errs, errs
    for k in (a, b):
        assert torch.equal(got[k], want[k]), k
        h[k].close()


def test_a_call_does_not_wait_for_foreign_work(gpu, paths):
    """A call whose stream is busy with work of the caller's (here 0.6 s of it) does
    not hold up a step of another handle on another stream: that work may be waiting
    for the step's result."""
    print("a step beside a call that is behind other work", flush=True)
    ha, hb = _make("sunny1", paths), _make("rwkv1", paths)
    t = torch.zeros(1, dtype=torch.int32, device="cuda")
    ha.step_batch(t)
    hb.step_batch(t)
    n = 1_000_000
    ev = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
    torch.cuda._sleep(n)
    ev[0].record()
    torch.cuda._sleep(n)
    ev[1].record()
    torch.cuda.synchronize()
    sa, busy = torch.cuda.Stream(), torch.cuda.Event()
    with torch.cuda.stream(sa):
        torch.cuda._sleep(int(n * 600 / ev[0].elapsed_time(ev[1])))
        busy.record()
    # a stream that the runtime has not put on the busy one's hardware queue
    sb = None
    for c in [torch.cuda.Stream() for _ in range(8)]:
        with torch.cuda.stream(c):
            t.clone()
            e = torch.cuda.Event()
            e.record()
        time.sleep(0.01)
        if e.query():
            sb = c
            break
    assert sb is not None and not busy.query()

    def first():
        with torch.cuda.stream(sa):
            ha.step_batch(t)
    th = threading.Thread(target=first)
    th.start()
    time.sleep(0.1)             # the first call is waiting by now
    with torch.cuda.stream(sb):
        hb.step_batch(t)
    still = not busy.query()      # (the step returns when it is done)
    th.join()
    torch.cuda.synchronize()
    assert still, "the second handle's step waited for the first one's stream"
    ha.close()
    hb.close()


_CHILD = """
import sys
import numpy as np, torch
sys.path.insert(0, sys.argv[1])
from pathlib import Path
from tests.test_streams_gpu import _make, _tokens
h = {k: _make(k, (Path(sys.argv[2]), Path(sys.argv[3]))) for k in sys.argv[5:]}
toks = {k: _tokens(x) for k, x in h.items()}
torch.cuda.synchronize()
print("ready", flush=True)
sys.stdin.readline()
out = {}
for k, x in h.items():
    for _ in range(10):
        x.reset()
        out[k] = torch.stack([x.step_batch(t) for t in toks[k]]).cpu().numpy()
    x.reset()
    out[k + " greedy"] = x.decode_greedy(toks[k][0], 8).cpu().numpy()
np.savez(sys.argv[4], **out)
for x in h.values():
    x.close()
"""


def _tokens(h):
    rng = np.random.default_rng(5)
    return [torch.from_numpy(rng.integers(0, h.vocab, h.max_batch).astype(np.int32)).cuda() for _ in range(24)]


@pytest.mark.parametrize("n,locks", [(2, "shared"), (1, "no folder"), (1, "stuck")])
def test_processes(gpu, paths, tmp_path, monkeypatch, n, locks):
    """Two processes that step on one device at once: each gets what it gets alone.
    Without a folder for the lock files, and while another process sits on them, the
    calls take the per-kernel steps."""
    print("processes:", n, "lock files:", locks, flush=True)
    kinds = ["sunny1", "sunny4", "sunny20", "rwkv1"]
    monkeypatch.setenv("SNHIP_LOCK_DIR", str(tmp_path / "missing" if locks == "no folder" else tmp_path))
    monkeypatch.setenv("SNHIP_GATE_SECONDS", "0.2" if locks == "stuck" else "60")
    pci = ctypes.create_string_buffer(64)
    assert _native.lib().hipDeviceGetPCIBusId(pci, 64, 0) == 0
    lock = tmp_path / f"snhip-{pci.value.decode()}.lock"
    held = None
    if locks == "stuck":
        held = open(lock, "w")
        fcntl.flock(held, fcntl.LOCK_EX)
    root = str(Path(__file__).resolve().parents[1])
    ps = [subprocess.Popen([sys.executable, "-c", _CHILD, root, str(paths[0]), str(paths[1]),
                            str(tmp_path / f"o{i}.npz"), *kinds],
                           stdin=subprocess.PIPE, stdout=subprocess.PIPE, text=True) for i in range(n)]
    try:
        for p in ps:
            assert p.stdout.readline() == "ready\n"
        for p in ps:
            p.stdin.write("\n")
            p.stdin.flush()
        assert [p.wait(60) for p in ps] == [0] * n
    finally:
        for p in ps:
            p.kill()
        if held:
            held.close()
    assert lock.exists() == (locks != "no folder")
    for k in kinds:
        h = _make(k, paths)
        toks = _tokens(h)
        want = torch.stack([h.step_batch(t) for t in toks]).cpu().numpy()
        h.reset()
        greedy = h.decode_greedy(toks[0], 8).cpu().numpy()
        for i in range(n):
            o = np.load(tmp_path / f"o{i}.npz")
            if locks == "shared" or k == "rwkv1":
                assert np.array_equal(o[k], want), (i, k)
            else:                                         # another order of the sums
                assert np.abs(o[k] - want).max() < 2e-5, (i, k)
            assert np.array_equal(o[k + " greedy"], greedy), (i, k)
        h.close()
