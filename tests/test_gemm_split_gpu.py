"""Prefill products from fp16 planes (every value as h + l, three matrix products)
against the same prefill on the fp32 matrix cores (SNHIP_GEMM_SPLIT=0): at rows and
widths around the tiles and stages, split K and whole, in each weight format and
across chunks; with weights of very different magnitudes; and with infinities.

Bar: the prefill's own against the oracle (logits within 2e-5, states within 1e-5);
both forms round in fp32, so neither is the other's reference. Against 64 bits the
planes' error is to be no larger than that of the fp32 matrix cores."""
from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle
from oracle.torch_ref import TorchSunny, forward_hist_to_step
from sunnynet_amd import _native
from sunnynet_amd.blob import pack_sunny_blob
from sunnynet_amd.config import SMALL, SUNNY_100M, TINY, matmul_params
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


def _in_64_bits(w, toks, block):
    """Logits, s and hist of the prefill in 64 bits, from what the handle multiplies:
    decay and W_eff rounded to fp32 as in the blob, INT4 values dequantized."""
    ref, ref32 = TorchSunny(w, torch.float64), TorchSunny(w, torch.float32)

    def mat(m):
        m = m.float().contiguous()
        if block:
            m = torch.from_numpy(oracle.dequant_i4(*oracle.quant_i4(m.numpy(), block), m.shape[1], block))
        return m.double()
    for a, b in zip(ref.layers, ref32.layers):
        a.delta = b.delta.double()
        a.V, a.U, a.W_z, a.W_c, a.W_eff = (mat(m) for m in (b.V, b.U, b.W_z, b.W_c, b.W_eff))
    ref.head = mat(ref32.head)
    lg, (s, hist) = ref.forward(toks.long().cpu())
    return lg, s, forward_hist_to_step(hist)


@pytest.mark.parametrize("block", [0, 32])
@pytest.mark.parametrize("B,T", [(4, 200), (1, 999), (16, 64)])
def test_error_against_64_bits(gpu, tmp_path, monkeypatch, B, T, block):
    """At the 100M model's width, split K and whole: no output is further from the
    64-bit result than with the products on the fp32 matrix cores (2-norm)."""
    print("split products against 64 bits", B, T, block, flush=True)
    cfg = SUNNY_100M.with_(vocab_size=512, layers=4)
    w = gaussian_matmuls(init_sunnynet(cfg, 0), seed=8)
    p = tmp_path / "m.bin"
    p.write_bytes(pack_sunny_blob(w))
    toks = torch.from_numpy(np.random.default_rng(T).integers(0, cfg.vocab_size, (B, T)).astype(np.int32)).to(gpu)
    kw = {"weights": "int4", "block": block} if block else {}
    split, fp32 = _both(monkeypatch, p, cfg, toks, **kw)
    for x, y, e in zip(split, fp32, _in_64_bits(w, toks, block)):
        e = e.numpy()
        es, ef = (np.linalg.norm(v - e) / np.linalg.norm(e) for v in (x, y))
        print(f"  planes {es:.3e}, fp32 matrix cores {ef:.3e}", flush=True)
        assert es <= ef


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


@pytest.mark.parametrize("where", ["row of W", "row of X"])
def test_tiny_value_times_infinity(gpu, tmp_path, monkeypatch, where):
    """A value too small for the planes beside its row's largest, times an infinity,
    is that infinity and not zero times it: in the vocabulary head, an infinite
    weight on a channel of 2^-60, and an infinite channel on a weight of 2^-60 (and
    of 2^-149, fp32's smallest)."""
    print("split products, tiny times infinity:", where, flush=True)
    cfg = TINY.with_(layers=1)
    w = gaussian_matmuls(init_sunnynet(cfg, 0), seed=9)
    if where == "row of W":
        w.no_g[3], w.no_c[3] = 2.0 ** -60, 0.0
        w.embed[7, 3] = float("inf")
    else:
        w.no_c[3] = float("inf")
        w.embed[9, 3], w.embed[11, 3], w.embed[13, 3], w.embed[15, 3] = 2.0 ** -60, -2.0 ** -149, 0.0, -0.0
    p = tmp_path / "m.bin"
    p.write_bytes(pack_sunny_blob(w))
    toks = np.random.default_rng(3).integers(20, cfg.vocab_size, (3, 50)).astype(np.int32)
    a, b = _both(monkeypatch, p, cfg, torch.from_numpy(toks).to(gpu))
    assert np.isinf(b[0]).any() and np.isinf(b[0][..., 7 if where == "row of W" else 9]).all()
    assert np.array_equal(np.isnan(a[0]), np.isnan(b[0]))
    assert np.array_equal(a[0][np.isinf(b[0])], b[0][np.isinf(b[0])])
    fin = np.isfinite(b[0])
    assert np.isfinite(a[0][fin]).all()
    assert fin.sum() == 0 or np.abs(a[0][fin] - b[0][fin]).max() < TOL


def test_planes_and_memory(gpu, tmp_path, monkeypatch):
    """The weights' planes are made at load, not in the first prefill; without memory
    for them, at load or beside a prefill's workspace, the products are the fp32 ones;
    and a prefill that does not fit even so fails and leaves the handle usable."""
    print("planes and memory", flush=True)
    cfg, lib = SMALL, _native.lib()
    p = tmp_path / "m.bin"
    p.write_bytes(pack_sunny_blob(gaussian_matmuls(init_sunnynet(cfg, 0), seed=4)))
    toks = torch.from_numpy(np.random.default_rng(5).integers(0, cfg.vocab_size, (1, 200)).astype(np.int32)).to(gpu)

    def load():
        return HipModel(p, cfg.vocab_size, cfg.dim, cfg.inner, cfg.rank, cfg.taps, cfg.layers)

    def run(h):
        h.reset()
        return [x.cpu() for x in (h.prefill_batch(toks), *h.get_state(1))]

    def same(a, b):
        return all(torch.equal(x, y) for x, y in zip(a, b))
    base = lib.snhip_device_bytes()
    monkeypatch.setenv("SNHIP_GEMM_SPLIT", "0")
    h = load()
    plain_bytes = lib.snhip_device_bytes() - base
    plain = run(h)
    plain_ws = lib.snhip_device_bytes() - base - plain_bytes
    h.close()
    assert lib.snhip_device_bytes() == base
    monkeypatch.delenv("SNHIP_GEMM_SPLIT")
    h = load()
    planes_bytes = lib.snhip_device_bytes() - base - plain_bytes
    assert planes_bytes >= 4 * matmul_params(cfg)
    split = run(h)
    ws = lib.snhip_device_bytes() - base - plain_bytes - planes_bytes
    assert 0 < ws < plain_ws and not same(split, plain)       # no rows stored beside their planes
    assert same(run(h), split) and lib.snhip_device_bytes() - base == plain_bytes + planes_bytes + ws
    h.close()
    # no room for the planes at load
    monkeypatch.setenv("SNHIP_MEM_LIMIT", str(base + plain_bytes + planes_bytes // 2))
    h = load()
    assert lib.snhip_device_bytes() - base == plain_bytes
    monkeypatch.delenv("SNHIP_MEM_LIMIT")
    assert same(run(h), plain)
    h.close()
    # no room for the workspace beside them
    h = load()
    monkeypatch.setenv("SNHIP_MEM_LIMIT", str(base + plain_bytes + planes_bytes + ws // 2))
    assert same(run(h), plain)
    assert lib.snhip_device_bytes() - base == plain_bytes + plain_ws
    h.close()
    # nor without them
    h = load()
    monkeypatch.setenv("SNHIP_MEM_LIMIT", str(base + plain_bytes + plain_ws // 2))
    with pytest.raises(_native.SnHipError):
        run(h)
    monkeypatch.delenv("SNHIP_MEM_LIMIT")
    assert same(run(h), plain)
    h.close()
    assert lib.snhip_device_bytes() == base
