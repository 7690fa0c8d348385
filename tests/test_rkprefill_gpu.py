"""RWKV-7 prefill in chunks of tokens (rkprefill.hip) against the oracle's
token-by-token steps: logits, state and shift vectors bit for bit, from a
carried state, at the edges of the LayerNorm's row groups, of the recurrence's
read-ahead and of the chunk; row lengths with and without the lane-sliced sums,
stored INT4, quantized at load and fp32 weights, tiled and stored products."""
from __future__ import annotations

import numpy as np
import pytest

import oracle
from sunnynet_amd import _native
from sunnynet_amd.runtime.rwkv7 import HipRwkv7
from sunnynet_amd.rwkv7 import RwkvConfig, init_rwkv7, pack_rwkv7_blob

pytestmark = pytest.mark.gpu

# dim 128: one lane sums a row; 768 and 1024: 12 and 16 values per lane
CFGS = {128: RwkvConfig(layers=2, dim=128, head_size=64, ff=256, vocab=512, ranks=(64, 64, 32, 64)),
        768: RwkvConfig(layers=3, dim=768, head_size=64, ff=1536, vocab=1024, ranks=(64, 64, 32, 128)),
        1024: RwkvConfig(layers=2, dim=1024, head_size=64, ff=1280, vocab=512, ranks=(32, 68, 12, 100))}


@pytest.mark.parametrize("dim,int4,T,env", [
    (128, False, 2, {}), (128, False, 5, {}), (128, True, 65, {}), (128, True, 513, {}),
    (128, True, 30, {"SNHIP_RKQ_W4": "0"}), (128, False, 30, {"SNHIP_RKQ_W4": "0"}),
    (128, False, 31, {"SNHIP_RK_EXACT": "0"}),
    (768, False, 7, {}), (768, True, 6, {}), (768, True, 130, {}), (768, True, 1025, {}),
    (1024, False, 33, {}),
])
def test_prefill_equals_steps(gpu, tmp_path, monkeypatch, dim, int4, T, env):
    print("rwkv7 chunked prefill", dim, int4, T, env, flush=True)
    cfg = CFGS[dim]
    blob = pack_rwkv7_blob(init_rwkv7(cfg, 3), int4=int4)
    path = tmp_path / "rk.bin"
    path.write_bytes(blob)
    for k, v in env.items():
        monkeypatch.setenv(k, v)
    hm = HipRwkv7(path, max_batch=2)
    orc = oracle.RkOracle(blob)
    toks = np.random.default_rng(T).integers(0, cfg.vocab, T + 5)
    for t in toks[:3]:
        hm.step_raw(int(t))
        orc.step([t])
    S1, sh1 = (x[1:].clone() for x in hm.get_state())
    got = np.asarray(hm.prefill([int(t) for t in toks[3:3 + T]]), np.float32)
    for t in toks[3:3 + T]:
        ref = orc.step([t])[0]
    assert np.array_equal(got, ref)
    S, sh = hm.get_state()
    So, sho = orc.get_state()
    assert np.array_equal(S[:1].cpu().numpy(), So) and np.array_equal(sh[:1].cpu().numpy(), sho)
    assert (S[1:] == S1).all() and (sh[1:] == sh1).all()     # sequence 1 is untouched
    for t in toks[3 + T:]:                                   # and the steps go on from there
        assert np.array_equal(np.asarray(hm.step(int(t)), np.float32), orc.step([t])[0])


@pytest.mark.parametrize("room", [0, 400_000, 3_000_000])
def test_prefill_without_memory(gpu, tmp_path, monkeypatch, room):
    """With no memory for the workspace of 512 tokens the prompt runs in shorter
    chunks, and with none at all token by token: never an error, the same bits."""
    print("rwkv7 prefill, bytes left:", room, flush=True)
    cfg = CFGS[128]
    blob = pack_rwkv7_blob(init_rwkv7(cfg, 3))
    path = tmp_path / "rk.bin"
    path.write_bytes(blob)
    lib = _native.lib()
    hm = HipRwkv7(path)
    orc = oracle.RkOracle(blob)
    toks = [int(t) for t in np.random.default_rng(4).integers(0, cfg.vocab, 90)]
    before = lib.snhip_device_bytes()
    monkeypatch.setenv("SNHIP_MEM_LIMIT", str(before + room))
    got = np.asarray(hm.prefill(toks), np.float32)
    taken = lib.snhip_device_bytes() - before
    assert taken <= room and (taken > 0) == (room > 0)
    for t in toks:
        ref = orc.step([t])[0]
    assert np.array_equal(got, ref)
    So, sho = orc.get_state()
    S, sh = hm.get_state()
    assert np.array_equal(S.cpu().numpy(), So) and np.array_equal(sh.cpu().numpy(), sho)
    hm.close()
    assert lib.snhip_device_bytes() < before
