"""The ring form of the recurrence (k_scan_ring: few channels, any width and
length) against the oracle, bit for bit: forward in both forms and backward, at
the edges of its 64-channel workgroups, its slots and its tiles and of the rules
that choose it (forward pinned to it and as chosen), from an unaligned view; and with
infinities and NaN against the other kernels."""
from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle
from sunnynet_amd import runtime

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1, 1), (3, 2, 7), (1, 33, 64), (2, 31, 65), (1, 256, 63), (5, 257, 13), (3, 333, 777),
          (2, 511, 128), (1, 513, 1000), (1, 1025, 8),
          (3, 40, 2731), (9, 65, 2047),
          (2, 23, 100), (2, 24, 100), (2, 79, 100), (2, 128, 128), (2, 129, 128), (13, 32, 1001),
          (8, 64, 2048), (9, 65, 2048), (13, 129, 2046)]


def _dev(x, off=0):
    t = torch.from_numpy(x)
    if not off:
        return t.cuda()
    buf = torch.empty(t.numel() + off, device="cuda")    # a view that starts off its allocation's alignment
    v = buf[off:].view(t.shape)
    v.copy_(t)
    return v


@pytest.mark.parametrize("B,T,N", SHAPES)
@pytest.mark.parametrize("gated", [True, False])
@pytest.mark.parametrize("pin", [None, "ring,1,32,32", "ring,1,64,32"])
def test_forward(gpu, monkeypatch, B, T, N, gated, pin):
    print("ring scan", B, T, N, gated, pin, flush=True)
    if pin:
        monkeypatch.setenv("SNHIP_SCAN_SHAPE", pin)
    rng = np.random.default_rng(T * 1000 + N)
    a = rng.random((B, T, N), dtype=np.float32)
    b = rng.standard_normal((B, T, N)).astype(np.float32)
    s0 = rng.standard_normal((B, N)).astype(np.float32)
    ro, rs = oracle.recur_scan(a, b, s0, gated)
    for off in (0, 1):
        out, send = runtime.scan(_dev(a, off), _dev(b, off), _dev(s0, off), gated=gated)
        assert np.array_equal(out.cpu().numpy(), ro) and np.array_equal(send.cpu().numpy(), rs)


@pytest.mark.parametrize("B,T,N", SHAPES)
def test_backward(gpu, B, T, N):
    print("ring scan backward", B, T, N, flush=True)
    rng = np.random.default_rng(T * 1000 + N)
    p = rng.random((B, T, N), dtype=np.float32)
    nu, dout = (rng.standard_normal((B, T, N)).astype(np.float32) for _ in range(2))
    s0 = rng.standard_normal((B, N)).astype(np.float32)
    out, _ = oracle.recur_scan(p, nu, s0, True)
    ref = oracle.scan_bwd(p, nu, s0, out, dout)
    for off in (0, 3):
        got = runtime.scan_bwd(*(_dev(x, off) for x in (p, nu, s0, out, dout)))
        for g, r in zip(got, ref):
            assert np.array_equal(g.cpu().numpy(), r)


@pytest.mark.parametrize("gated", [True, False])
def test_special_values(gpu, monkeypatch, gated):
    print("ring scan, infinities and NaN", gated, flush=True)
    rng = np.random.default_rng(1)
    a = rng.random((2, 300, 72), dtype=np.float32)
    b = rng.standard_normal((2, 300, 72)).astype(np.float32)
    for x in (a, b):
        i = rng.integers(0, x.size, 200)
        x.flat[i] = rng.choice([np.inf, -np.inf, np.nan, 0.0, -0.0, 3.4e38], 200)
    s0 = np.zeros((2, 72), np.float32)
    s0[0, :3] = [np.inf, -np.inf, np.nan]
    args = [_dev(x) for x in (a, b, s0)]
    monkeypatch.setenv("SNHIP_SCAN_SHAPE", "ring,1,32,32")
    got = runtime.scan(*args, gated=gated)
    monkeypatch.setenv("SNHIP_SCAN_SHAPE", "gen,1,8,16")
    ref = runtime.scan(*args, gated=gated)
    for g, r in zip(got, ref):
        assert torch.equal(torch.isnan(g), torch.isnan(r))
        assert torch.equal(torch.nan_to_num(g), torch.nan_to_num(r))
