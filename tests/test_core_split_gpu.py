"""The split form of the fused block core (gate kernels over the whole chip, the
chain as a ring scan) against the oracle: widths and lengths at the edges of its
lane pairs, chunks of time and ring workgroups and of the rules that choose it,
from aligned and unaligned storage, where the ddelta partials are limited by
their scratch, with saturated gates, and with outputs that overlap inputs.

Bar: the reference's own (tests/test_architecture.py:738-740, 803-805), 1e-5 on
states, u and p and 1e-4 on dq, ddelta and ds0 (relative to the largest
magnitude where that is above 1)."""
from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle
from sunnynet_amd import _native, runtime

pytestmark = pytest.mark.gpu

FWD_TOL, BWD_TOL = 1e-5, 1e-4
SHAPES = [(1, 1, 8), (2, 7, 8), (3, 9, 40), (1, 33, 136), (2, 257, 200), (1, 2049, 8), (3, 64, 128),
          (33, 31, 264), (32, 150, 2048), (2, 32, 72), (2, 49, 72), (9, 33, 1000), (3, 49, 8),
          (2, 75, 264)]


def _inputs(B, T, D, seed):
    rng = np.random.default_rng(seed)
    q = (rng.standard_normal((B, T, 2 * D)) * 0.6).astype(np.float32)
    delta = (0.01 + 0.4 * rng.random(D)).astype(np.float32)
    s0 = (rng.standard_normal((B, D)) * 0.1).astype(np.float32)
    dstate, du_in = (rng.standard_normal((B, T, D)).astype(np.float32) for _ in range(2))
    return q, delta, s0, dstate, du_in


def _dev(*xs, off=0):
    out = []
    for x in xs:
        t = torch.from_numpy(np.ascontiguousarray(x))
        v = torch.empty(t.numel() + off, device="cuda")[off:].view(t.shape)   # off floats past an aligned start
        v.copy_(t)
        out.append(v)
    return out


def _close(got, ref, names, tol, rel):
    for name, a, b in zip(names, got, ref):
        a = a.cpu().numpy()
        bar = tol * max(1.0, float(np.abs(b).max())) if rel else tol
        assert np.abs(a - b).max() < bar, name


@pytest.mark.parametrize("B,T,D", SHAPES)
@pytest.mark.parametrize("off", [0, 1])
def test_matches_oracle(gpu, B, T, D, off):
    print("core split", B, T, D, off, flush=True)
    q, delta, s0, dstate, du_in = _inputs(B, T, D, B * 1000 + T + D)
    ref = oracle.core_fwd(q, delta, s0)
    _close(runtime.core_fwd(*_dev(q, delta, s0, off=off)), ref, ("states", "u", "p"), FWD_TOL, False)
    rb = oracle.core_bwd(q, delta, s0, *ref, dstate, du_in)
    gb = runtime.core_bwd(*_dev(q, delta, s0, *ref, dstate, du_in, off=off))
    _close(gb, rb, ("dq", "ddelta", "ds0"), BWD_TOL, True)


def test_saturated_gates(gpu):
    """Gates of magnitude 50 and 100 (exp overflows or underflows): the
    reference's non-finite pattern and its finite values."""
    print("core split, saturated gates", flush=True)
    B, T, D = 2, 45, 72
    q, delta, s0, _, _ = _inputs(B, T, D, 3)
    rng = np.random.default_rng(4)
    mask = rng.random((B, T, D)) < 0.1
    q[..., D:][mask] = rng.choice([-100.0, 100.0, -50.0, 50.0], size=int(mask.sum())).astype(np.float32)
    ref = oracle.core_fwd(q, delta, s0)
    for a, b in zip(runtime.core_fwd(*_dev(q, delta, s0)), ref):
        a = a.cpu().numpy()
        assert np.array_equal(np.isnan(a), np.isnan(b)) and np.array_equal(np.isinf(a), np.isinf(b))
        fin = np.isfinite(b)
        assert np.abs(a[fin] - b[fin]).max() < FWD_TOL


@pytest.mark.parametrize("B,T,D", [(2, 37, 40), (2, 64, 128), (2, 57, 40), (2, 272, 128)])
def test_outputs_over_inputs(gpu, B, T, D):
    """dq in place of q and ds0 in place of s0 give what separate outputs give."""
    print("core split, in place", B, T, D, flush=True)
    q, delta, s0, dstate, du_in = _inputs(B, T, D, 9)
    dv = _dev(q, delta, s0)
    fwd = runtime.core_fwd(*dv)
    ds, di = _dev(dstate, du_in)
    sep = runtime.core_bwd(*dv, *fwd, ds, di)
    ddelta = torch.zeros(D, device="cuda")
    ptrs = [t.data_ptr() for t in (*dv, *fwd, ds, di, dv[0], ddelta, dv[2])]
    rc = _native.lib().snhip_abi_core_bwd_dev(*ptrs, B, T, D, _native.stream_handle(ds.device))
    _native.check(rc, "snhip_abi_core_bwd_dev")
    _close((dv[0], ddelta, dv[2]), [x.cpu().numpy() for x in sep], ("dq", "ddelta", "ds0"), BWD_TOL, True)
