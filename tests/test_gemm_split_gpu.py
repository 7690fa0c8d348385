"""Prefill products from fp16 planes (every value as h + l, three matrix products)
against the same prefill on the fp32 matrix cores (SNHIP_GEMM_SPLIT=0): at rows and
widths around the tiles and stages, split K and whole, in each weight format and
across chunks; with weights of very different magnitudes; and with infinities.

Bar: the prefill's own against the oracle (logits within 2e-5, states within 1e-5);
both forms round in fp32, so neither is the other's reference."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from sunnynet_amd.blob import pack_sunny_blob
from sunnynet_amd.config import SMALL, TINY
from sunnynet_amd.runtime.model import HipModel
from sunnynet_amd.weights import gaussian_matmuls, init_sunnynet

pytestmark = pytest.mark.gpu
TOL = 2e-5

MID = SMALL.with_(vocab_size=1000, dim=192, inner=2080, rank=96, layers=2)   # rows of K past the register form


def _both(monkeypatch, path, cfg, toks, **kw):
    out = []
    for split in (True, False):
        if split:
            monkeypatch.delenv("SNHIP_GEMM_SPLIT", raising=False)
        else:
            monkeypatch.setenv("SNHIP_GEMM_SPLIT", "0")
        hm = HipModel(path, cfg.vocab_size, cfg.dim, cfg.inner, cfg.rank, cfg.taps, cfg.layers,
                      max_batch=toks.shape[0], **kw)
        lg = hm.prefill_all(toks)
        out.append([x.cpu().numpy() for x in (lg, *hm.get_state(toks.shape[0]))])
    return out


@pytest.mark.parametrize("cfg,B,T,kw,chunk", [
    (TINY, 1, 65, {}, None), (TINY, 3, 43, {}, None), (TINY, 2, 700, {}, "129"), (MID, 1, 128, {}, None),
    (MID, 5, 77, {"weights": "fp16"}, None), (MID, 1, 257, {"weights": "int4", "block": 32}, None),
    (SMALL, 2, 130, {"weights": "int4", "block": 64}, None), (SMALL, 33, 63, {}, None),
    (SMALL.with_(vocab_size=33000, layers=1), 5, 100, {}, None)])
def test_matches_fp32_products(gpu, tmp_path, monkeypatch, cfg, B, T, kw, chunk):
    print("split products", cfg.dim, cfg.inner, cfg.rank, B, T, kw, chunk, flush=True)
    if chunk:
        monkeypatch.setenv("SNHIP_PREFILL_CHUNK", chunk)
    p = tmp_path / "m.bin"
    p.write_bytes(pack_sunny_blob(gaussian_matmuls(init_sunnynet(cfg, 0), seed=5)))
    toks = torch.from_numpy(np.random.default_rng(B + T).integers(0, cfg.vocab_size, (B, T)).astype(np.int32)).to(gpu)
    a, b = _both(monkeypatch, p, cfg, toks, **kw)
    assert np.abs(a[0] - b[0]).max() < TOL
    assert np.abs(a[1] - b[1]).max() < 1e-5 and np.abs(a[2] - b[2]).max() < 1e-5


def test_rows_of_any_magnitude(gpu, tmp_path, monkeypatch):
    """V scaled by 2^-70 and U by 2^70, with rows of zeros: the planes' powers of
    two keep every row's digits."""
    print("split products, magnitudes", flush=True)
    cfg = TINY
    w = gaussian_matmuls(init_sunnynet(cfg, 0), seed=6)
    for L in w.layers:
        L.U.mul_(2.0 ** 70)
        L.V.mul_(2.0 ** -70)
        L.U[3::7] = 0.0
    p = tmp_path / "m.bin"
    p.write_bytes(pack_sunny_blob(w))
    toks = torch.from_numpy(np.random.default_rng(1).integers(0, cfg.vocab_size, (2, 90)).astype(np.int32)).to(gpu)
    a, b = _both(monkeypatch, p, cfg, toks)
    assert np.isfinite(b[0]).all() and np.abs(a[0] - b[0]).max() < TOL


@pytest.mark.parametrize("where", ["V", "U", "W_z"])
def test_infinite_weights_and_bad_tokens(gpu, tmp_path, monkeypatch, where):
    """An infinite weight, and a token outside the vocabulary (a row of NaN): the
    same outputs are finite, infinite and NaN in both forms, signs included."""
    print("split products, infinities", where, flush=True)
    cfg = TINY.with_(layers=1)
    w = gaussian_matmuls(init_sunnynet(cfg, 0), seed=7)
    getattr(w.layers[0], where)[5, 3] = float("inf")
    p = tmp_path / "m.bin"
    p.write_bytes(pack_sunny_blob(w))
    toks = np.random.default_rng(2).integers(0, cfg.vocab_size, (3, 50)).astype(np.int32)
    toks[1, 20] = cfg.vocab_size + 7
    for x, y in zip(*_both(monkeypatch, p, cfg, torch.from_numpy(toks).to(gpu))):
        assert np.array_equal(np.isnan(x), np.isnan(y))
        assert np.array_equal(np.isinf(x), np.isinf(y)) and np.array_equal(x[np.isinf(x)], y[np.isinf(y)])
        fin = np.isfinite(y)
        assert fin.sum() == 0 or np.abs(x[fin] - y[fin]).max() < TOL
