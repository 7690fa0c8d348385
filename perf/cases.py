"""Calls of this framework whose time is followed from change to change.

Each case is one call, or one short chain of calls, that a program makes through
the public entry points: the recurrence and the fused block core (forward, and
forward with backward under autograd), the SunnyNet handle (decode steps, prompt
prefill, every-position forward) and the RWKV-7 handle (decode steps, prompt
prefill). The sizes are those of the configurations in ``sunnynet_amd.config``
and ``sunnynet_amd.rwkv7``, of the benchmark and of the tests; ``draw`` gives
more cases of the same ranges. ``exact`` restates each path in plain torch in
64 bits.
"""
from __future__ import annotations

import functools
import math
import os

import numpy as np
import torch

from sunnynet_amd.blob import pack_sunny_blob
from sunnynet_amd.config import PRESETS, matmul_params
from sunnynet_amd.runtime import core_forward, gated_scan, scan
from sunnynet_amd.runtime.model import HipModel, HipSunnyNet
from sunnynet_amd.runtime.rwkv7 import HipRwkv7
from sunnynet_amd.rwkv7 import RWKV_CFG4, RWKV_TINY, init_rwkv7, pack_rwkv7_blob
from sunnynet_amd.weights import SunnyLayerWeights, SunnyWeights, horizon_logit

DEV = "cuda:0"
RWKV = {"12x768": RWKV_CFG4, "tiny": RWKV_TINY}
INT4_BLOCK = 32          # the INT4 group size of the measured workloads
STEPS = 4                # decode steps of one pass


def listed():
    return [
        # The measured prefill recurrence: a long batch over a wide layer.
        {"name": "scan_gated_b16", "kind": "scan", "gated": True, "B": 16, "T": 4096, "N": 2048},
        # A small odd-sized recurrence in the FMA form: launch and latency.
        {"name": "scan_fma_ragged", "kind": "scan", "gated": False, "B": 3, "T": 333, "N": 777},
        # Training through the recurrence at the 100M model's width.
        {"name": "scan_train_b4", "kind": "scan_train", "B": 4, "T": 2048, "N": 1024},
        # Training through the fused block core at the 100M model's width.
        {"name": "core_train_b8", "kind": "core_train", "B": 8, "T": 2048, "D": 1024},
        # The same on a short batch of prompts that no tile divides.
        {"name": "core_train_ragged", "kind": "core_train", "B": 3, "T": 777, "D": 200},
        # One user's decode: SunnyNet-100M at full precision.
        {"name": "sunny_step_fp32_b1", "kind": "sunny_step", "model": "100m", "weights": "fp32", "B": 1,
         "prompt": 16},
        # A serving batch on quantized weights.
        {"name": "sunny_step_int4_b32", "kind": "sunny_step", "model": "100m", "weights": "int4", "B": 32,
         "prompt": 16},
        # One user's prompt of an odd length on quantized weights.
        {"name": "sunny_prefill_int4_b1", "kind": "sunny_prefill", "model": "100m", "weights": "int4",
         "B": 1, "T": 999},
        # Scoring a batch: the logits of every position.
        {"name": "sunny_forward_fp32_b16", "kind": "sunny_forward", "model": "100m", "weights": "fp32",
         "B": 16, "T": 512},
        # One user's decode on the RWKV-7 model of the benchmark.
        {"name": "rwkv_step_int4_b1", "kind": "rwkv_step", "model": "12x768", "weights": "int4", "B": 1,
         "prompt": 16},
        # A full serving batch of it.
        {"name": "rwkv_step_int4_b64", "kind": "rwkv_step", "model": "12x768", "weights": "int4", "B": 64,
         "prompt": 16},
        # The benchmark's 512-token prompt of it.
        {"name": "rwkv_prefill_int4", "kind": "rwkv_prefill", "model": "12x768", "weights": "int4", "T": 512},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["scan", "scan_train", "core_train", "sunny_step", "sunny_step", "sunny_prefill",
                       "sunny_forward", "rwkv_step", "rwkv_prefill"])
    if kind in ("scan", "scan_train", "core_train"):
        # up to 2^24 values (2^26 forward only), widths from a tenth of the small model's on
        B, T = _log(rng, 1, 16), _log(rng, 16, 4096)
        N = min(_log(rng, 24, 2048), (1 << (26 if kind == "scan" else 24)) // (B * T))
        if rng.random() < 0.5:
            N = max(64, N // 64 * 64)        # a model's width
        if kind == "scan":
            return {"kind": kind, "gated": rng.random() < 0.7, "B": B, "T": T, "N": N}
        if kind == "scan_train":
            return {"kind": kind, "B": B, "T": T, "N": N}
        return {"kind": kind, "B": B, "T": T, "D": max(8, N // 8 * 8)}
    if kind.startswith("sunny"):
        model = rng.choice(["small", "100m", "100m"])
        weights = rng.choice(["fp32", "int4", "fp16"])
        if kind == "sunny_step":
            return {"kind": kind, "model": model, "weights": weights, "B": _log(rng, 1, 64),
                    "prompt": _log(rng, 4, 64)}
        B = _log(rng, 1, 16)
        rows = 8192 if kind == "sunny_forward" else 16384
        return {"kind": kind, "model": model, "weights": weights, "B": B,
                "T": min(_log(rng, 8, 2048), rows // B)}
    model = rng.choice(["tiny", "12x768", "12x768"])
    weights = rng.choice(["int4", "int4", "stored"])
    if kind == "rwkv_step":
        return {"kind": kind, "model": model, "weights": weights, "B": _log(rng, 1, 64),
                "prompt": _log(rng, 4, 64)}
    return {"kind": kind, "model": model, "weights": weights, "T": _log(rng, 8, 512)}


# ---- weights -----------------------------------------------------------------
@functools.lru_cache(maxsize=None)
def _sunny_weights(model):
    """Gaussian matrices N(0, 0.02^2) (the INT4 workload's), everything else as
    the model initialises it; gains and centres moved off 1 and 0."""
    cfg = PRESETS[model]
    g = torch.Generator().manual_seed(7)
    D, I, R, K, V = cfg.dim, cfg.inner, cfg.rank, cfg.taps, cfg.vocab_size

    def rn(*shape, std=0.02, mean=0.0):
        return mean + std * torch.randn(*shape, generator=g)

    layers = [SunnyLayerWeights(
        ni_g=rn(D, std=0.1, mean=1.0), ni_c=rn(D, std=0.05), nm_g=rn(I, std=0.1, mean=1.0),
        nm_c=rn(I, std=0.05), dw=rn(D, 1, K, std=0.1), V=rn(R, D), U=rn(2 * D, R), W_z=rn(I, D),
        W_c=rn(D, I), W_s=rn(D, D), circ=torch.tensor([0.25, 0.5, 0.25]), theta=horizon_logit(D),
        a=torch.tensor(0.5), b_gain=torch.tensor(0.5)) for _ in range(cfg.layers)]
    return SunnyWeights(cfg=cfg, embed=rn(V, D), layers=layers, no_g=rn(D, std=0.1, mean=1.0),
                        no_c=rn(D, std=0.05))


@functools.lru_cache(maxsize=None)
def _rwkv_weights(model):
    return init_rwkv7(RWKV[model], 2)


@functools.lru_cache(maxsize=None)
def _blob(family, model):
    """The model's weight file, held in memory for the life of the process."""
    buf = pack_sunny_blob(_sunny_weights(model)) if family == "sunny" else pack_rwkv7_blob(_rwkv_weights(model))
    fd = os.memfd_create(f"{family}-{model}")
    view = memoryview(buf)
    while view:
        view = view[os.write(fd, view):]
    return f"/proc/self/fd/{fd}"


def _sunny(case):
    c = PRESETS[case["model"]]
    return HipModel(_blob("sunny", case["model"]), c.vocab_size, c.dim, c.inner, c.rank, c.taps, c.layers,
                    group=c.group, max_batch=case["B"], weights=case["weights"], block=INT4_BLOCK)


def _tokens(case, seed, shape):
    cfg = RWKV[case["model"]] if case["kind"].startswith("rwkv") else PRESETS[case["model"]]
    vocab = cfg.vocab if case["kind"].startswith("rwkv") else cfg.vocab_size
    g = torch.Generator().manual_seed(seed)
    return torch.randint(0, vocab, shape, generator=g, dtype=torch.int32)


def _decay(n, dtype=torch.float32):
    """1 / horizon per channel, horizons from 2 to 8192 steps (the model's range)."""
    t = torch.arange(n, device=DEV, dtype=dtype) / max(1, n - 1)
    return 1.0 / (2.0 * 4096.0 ** t)


# ---- inputs ------------------------------------------------------------------
def prepare(case, seed):
    kind = case["kind"]
    if kind in ("scan", "scan_train", "core_train"):
        g = torch.Generator(device=DEV).manual_seed(seed)

        def rn(*shape):
            return torch.randn(*shape, generator=g, device=DEV)

        B, T = case["B"], case["T"]
        if kind == "core_train":
            D = case["D"]
            return {"kind": kind, "q": rn(B, T, 2 * D).requires_grad_(), "delta": _decay(D).requires_grad_(),
                    "s0": rn(B, D).requires_grad_(), "du": rn(B, T, D), "dst": rn(B, T, D)}
        N = case["N"]
        if kind == "scan" and not case["gated"]:
            a = 0.9 + 0.1 * torch.rand(B, T, N, generator=g, device=DEV)
        else:
            a = rn(B, T, N).sigmoid_().mul_(_decay(N).neg()).add_(1.0)
        st = {"kind": kind, "gated": case.get("gated", True), "a": a, "b": rn(B, T, N), "s0": rn(B, N)}
        if kind == "scan_train":
            for k in ("a", "b", "s0"):
                st[k].requires_grad_()
            st["dout"], st["dsend"] = rn(B, T, N), rn(B, N)
        return st
    if kind == "sunny_step":
        toks = _tokens(case, seed, (case["B"], case["prompt"] + STEPS)).to(DEV)
        h = _sunny(case)
        h.reset()
        h.prefill_batch(toks[:, :case["prompt"]].contiguous(), logits=False)
        return {"kind": kind, "h": h, "steps": [toks[:, case["prompt"] + i].contiguous() for i in range(STEPS)]}
    if kind in ("sunny_prefill", "sunny_forward"):
        return {"kind": kind, "h": _sunny(case), "toks": _tokens(case, seed, (case["B"], case["T"])).to(DEV)}
    h = HipRwkv7(_blob("rwkv", case["model"]), max_batch=case.get("B", 1), weights=case["weights"],
                 block=INT4_BLOCK)
    h.reset()
    if kind == "rwkv_prefill":
        return {"kind": kind, "h": h, "toks": _tokens(case, seed, (case["T"],)).tolist()}
    toks = _tokens(case, seed, (case["B"], case["prompt"] + STEPS)).to(DEV)
    for i in range(case["prompt"]):
        h.step_batch(toks[:, i].contiguous())
    return {"kind": kind, "h": h, "steps": [toks[:, case["prompt"] + i].contiguous() for i in range(STEPS)]}


# ---- one pass ----------------------------------------------------------------
def run(st):
    kind = st["kind"]
    if kind == "scan":
        return scan(st["a"], st["b"], st["s0"], gated=st["gated"])
    if kind == "scan_train":
        out, send = gated_scan(st["a"], st["b"], st["s0"])
        return (out, send) + torch.autograd.grad((out, send), (st["a"], st["b"], st["s0"]),
                                                 (st["dout"], st["dsend"]))
    if kind == "core_train":
        u, states = core_forward(st["q"], st["delta"], st["s0"])
        return (u, states) + torch.autograd.grad((u, states), (st["q"], st["delta"], st["s0"]),
                                                 (st["du"], st["dst"]))
    h = st["h"]
    if kind in ("sunny_step", "rwkv_step"):
        # a few given tokens, then the sequences' state is put aside
        for t in st["steps"]:
            logits = h.step_batch(t)
        return (logits,) + tuple(h.get_state(int(t.shape[0])))
    if kind == "sunny_prefill":
        h.reset()
        logits = h.prefill_batch(st["toks"])
        return (logits,) + tuple(h.get_state(int(st["toks"].shape[0])))
    if kind == "sunny_forward":
        logits, state = HipSunnyNet(h).forward(st["toks"], return_state=True)
        return logits, state.s, state.hist
    h.reset()
    logits = h.prefill(st["toks"])
    return (np.asarray(logits, np.float32),) + tuple(h.get_state(1))


# ---- what a pass cannot do without --------------------------------------------
def _rwkv_params(c):
    """The matrix weights without the head."""
    return c.matmul_params() - c.vocab * c.dim


def work(case):
    kind = case["kind"]
    if kind in ("scan", "scan_train", "core_train"):
        B, T, N = case["B"], case["T"], case.get("N", case.get("D"))
        n = B * T * N
        if kind == "scan":
            return {"bytes": 12 * n + 8 * B * N, "flops": (4 if case["gated"] else 2) * n}
        if kind == "scan_train":     # p, nu, dout in; out, dp, dnu out
            return {"bytes": 24 * n + 16 * B * N, "flops": 11 * n}
        # q (two values a channel), du, dstate in; u, states, dq out
        return {"bytes": 32 * n + 8 * B * N, "flops": 60 * n}
    if kind.startswith("sunny"):
        c = PRESETS[case["model"]]
        D, L, V, B, K = c.dim, c.layers, c.vocab_size, case["B"], c.taps
        per = {"fp32": 4.0, "fp16": 2.0, "int4": 0.5 + 4.0 / INT4_BLOCK}[case["weights"]]
        body, head = matmul_params(c) - V * D, V * D
        state = B * L * K * D * 4
        if kind == "sunny_step":
            return {"bytes": STEPS * (per * (body + head) + 2 * state + 4 * B * (D + V)) + 2 * state,
                    "flops": STEPS * 2 * B * (body + head)}
        rows = B * case["T"]
        heads = rows if kind == "sunny_forward" else B
        return {"bytes": per * (body + head) + state + 4 * (rows * D + heads * V),
                "flops": 2 * rows * body + 2 * heads * head}
    c = RWKV[case["model"]]
    per = 0.5 + 4.0 / INT4_BLOCK if case["weights"] == "int4" else 4.0
    body, head = _rwkv_params(c), c.vocab * c.dim
    B, T = case.get("B", 1), case.get("T", STEPS)
    state = B * c.layers * (c.dim * c.head_size + 2 * c.dim) * 4
    mix = 8 * c.layers * c.dim * c.head_size         # the state update and read-out, per token
    if kind == "rwkv_step":
        return {"bytes": STEPS * (per * (body + head) + 2 * state + 4 * B * (c.dim + c.vocab)) + 2 * state,
                "flops": STEPS * B * (2 * (body + head) + mix)}
    return {"bytes": per * (body + head) + state + 4 * (T * c.dim + c.vocab),
            "flops": T * (2 * body + mix) + 2 * head}


def tolerance(case):
    kind = case["kind"]
    if kind in ("scan", "scan_train"):
        return "exact"       # the entry points promise the reference's rounding, step by step
    if kind.startswith("rwkv"):
        return "exact"       # so does the default RWKV-7 step
    if kind == "core_train":
        # horizons of thousands of steps gather the rounding of as many: up to
        # 2.7e-5 from the 64-bit result, and other roundings of exp move it as far
        return {"rel": 1e-4, "max": 4e-3}
    # 32-bit sums through every layer: up to 2.4e-6 from the 64-bit result
    return {"rel": 1e-5, "max": 1e-4}


# ---- the same in 64 bits -------------------------------------------------------
def _f64(t):
    if isinstance(t, np.ndarray):
        t = torch.from_numpy(t)
    return t.detach().to(device=DEV, dtype=torch.float64)


def _int4(w, block):
    """Symmetric INT4 groups along the input, as the loaders quantize: in 32
    bits, on the host (whose divisions are the correctly rounded ones)."""
    g = np.asarray(w.detach() if isinstance(w, torch.Tensor) else w, np.float32)
    g = g.reshape(g.shape[0], -1, block)
    amax = np.abs(g).max(axis=2, keepdims=True)
    scale = np.where(amax == 0, np.float32(1), amax / np.float32(7))
    q = np.clip(np.rint(g * (np.float32(1) / scale)), -8, 7)
    return torch.from_numpy((q * scale).reshape(w.shape))


def _scan64(p, b, s0, out=None):
    s = s0
    rows = []
    for t in range(p.shape[1]):
        s = p[:, t] * s + b[:, t]
        if out is None:
            rows.append(s)
        else:
            out[:, t] = s
    return torch.stack(rows, 1) if out is None else out


def _compete64(gate, G):
    g = gate.reshape(*gate.shape[:-1], -1, G)
    w = torch.sigmoid(g - torch.roll(g, -1, -1)) * torch.sigmoid(g - torch.roll(g, -2, -1))
    return w.reshape(gate.shape)


def _norm64(x, g, c, eps):
    return torch.nn.functional.layer_norm(x, (x.shape[-1],), g, c, eps)


def _sunny64(case, toks, every):
    """Logits (of every position, or the last), s and newest-first history of
    the sequences `toks` (B, T) from the zero state."""
    w = _sunny_weights(case["model"])
    c = w.cfg
    fmt = case["weights"]

    def mat(m):
        m = m.detach().float()
        if fmt == "int4":
            m = _int4(m, INT4_BLOCK)
        elif fmt == "fp16":
            m = m.half().float()
        return _f64(m)

    eps = 0.02 * 0.02 + 1e-5
    B, T = toks.shape
    D, K = c.dim, c.taps
    embed = _f64(w.embed)
    x = embed[toks.long()]
    ss, hh = [], []
    span = math.log(c.h_max / c.h_min)
    for L in w.layers:
        W = L.W_s
        eff = L.circ[0] * torch.roll(W, -1, 1) + L.circ[1] * W + L.circ[2] * torch.roll(W, 1, 1)
        delta = _f64(1.0 / (c.h_min * torch.exp(span * torch.sigmoid(L.theta))))
        raw = _norm64(x, _f64(L.ni_g), _f64(L.ni_c), eps)
        dw = _f64(L.dw)[:, 0]
        pad = torch.cat([raw.new_zeros(B, K - 1, D), raw], 1)
        at = raw + sum(pad[:, j:j + T] * dw[:, j] for j in range(K))
        q = (at @ mat(L.V).T) @ mat(L.U).T
        u, gate = q[..., :D], q[..., D:]
        u = u * _compete64(gate, c.group)
        p = 1.0 - delta * (1.0 - torch.sigmoid(gate))
        s = _scan64(p, (1.0 - p) * u, raw.new_zeros(B, D), torch.empty_like(u))
        z = u @ mat(L.W_z).T
        a = _f64(torch.tanh(L.a))
        y = _norm64(z * (1.0 + 0.5 * a / (1.0 + z.abs())), _f64(L.nm_g), _f64(L.nm_c), eps)
        prev = torch.cat([s.new_zeros(B, 1, D), s[:, :-1]], 1)
        x = y @ mat(L.W_c).T + float(L.b_gain) * s + prev @ mat(eff).T + x
        ss.append(s[:, -1])
        hh.append(torch.flip(pad[:, T:], [1]))
    x = _norm64(x if every else x[:, -1], _f64(w.no_g), _f64(w.no_c), eps)
    return x @ mat(w.embed).T, torch.stack(ss, 1), torch.stack(hh, 1)


def _rwkv64(case, toks):
    """Last logits, S and shift of the sequences `toks` (B, T) from zero."""
    w = _rwkv_weights(case["model"])
    c = w.cfg
    B, T = toks.shape
    D, H, Z = c.dim, c.n_head, c.head_size

    def lin(x, m):
        if case["weights"] == "int4" and m.shape[1] % INT4_BLOCK == 0:
            return x @ _f64(_int4(m, INT4_BLOCK)).T
        return x @ _f64(m).T

    def back(x):
        return torch.cat([x.new_zeros(B, 1, D), x[:, :-1]], 1)

    x = _norm64(_f64(w.embed)[toks.long()], _f64(w.en_w), _f64(w.en_b), c.eps)
    first, SS, shifts = None, [], []
    for L in w.layers:
        V = {k: _f64(v) for k, v in L.items() if v.ndim == 1 or k == "lerp"}
        xn = _norm64(x, V["ln1_w"], V["ln1_b"], c.eps)
        dd = back(xn) - xn
        xr, xw, xk, xv, xa, xg = (xn + V["lerp"][i] * dd for i in range(6))
        r, k, v = lin(xr, L["r"]), lin(xk, L["k"]), lin(xv, L["v"])
        dec = torch.exp(-torch.sigmoid(lin(torch.tanh(lin(xw, L["w1"])), L["w2"]) + V["w0"]) * math.exp(-0.5))
        if first is None:
            first = v
        else:
            v = v + (first - v) * torch.sigmoid(lin(lin(xv, L["v1"]), L["v2"]) + V["v0"])
        a = torch.sigmoid(lin(lin(xa, L["a1"]), L["a2"]) + V["a0"])
        g = lin(torch.sigmoid(lin(xg, L["g1"])), L["g2"])
        kk = (k * V["kk"]).reshape(B, T, H, Z)
        kk = kk / kk.norm(dim=-1, keepdim=True).clamp_min(1e-12)
        k = k + k * (a - 1.0) * V["ka"]
        rh, kh, vh, ah, dh = (t.reshape(B, T, H, Z) for t in (r, k, v, a, dec))
        S = x.new_zeros(B, H, Z, Z)
        y = torch.empty_like(rh)
        kka = kk * ah
        for t in range(T):
            pv = S @ kk[:, t, :, :, None]
            S = S * dh[:, t, :, None, :] + (vh[:, t, :, :, None] * kh[:, t, :, None, :] - pv * kka[:, t, :, None, :])
            y[:, t] = (S @ rh[:, t, :, :, None])[..., 0]
        y = (y - y.mean(-1, keepdim=True)) / torch.sqrt(y.var(-1, unbiased=False, keepdim=True) + 64e-5)
        y = y.reshape(B, T, D) * V["lnx_w"] + V["lnx_b"]
        dot = (rh * kh * V["rk"].reshape(H, Z)).sum(-1, keepdim=True)
        y = (y + (dot * vh).reshape(B, T, D)) * g
        x = x + lin(y, L["o"])
        xn2 = _norm64(x, V["ln2_w"], V["ln2_b"], c.eps)
        x = x + lin(torch.relu(lin(xn2 + V["cmk_lerp"] * (back(xn2) - xn2), L["cmk"])) ** 2, L["cmv"])
        SS.append(S)
        shifts.append(torch.stack([xn[:, -1], xn2[:, -1]], 1))
    logits = lin(_norm64(x[:, -1], _f64(w.on_w), _f64(w.on_b), c.eps), w.head)
    return logits, torch.stack(SS, 1), torch.stack(shifts, 1)


def exact(case, seed):
    kind = case["kind"]
    if kind == "scan":
        st = prepare(case, seed)
        a, b = _f64(st["a"]), _f64(st["b"])
        if st["gated"]:
            b.mul_(1.0 - a)
        out = _scan64(a, b, _f64(st["s0"]), torch.empty_like(a))
        return out, out[:, -1]
    if kind == "scan_train":
        st = prepare(case, seed)
        a, b, s0 = (_f64(st[k]).requires_grad_() for k in ("a", "b", "s0"))
        out = _scan64(a, (1.0 - a) * b, s0)
        send = out[:, -1]
        return (out.detach(), send.detach()) + torch.autograd.grad(
            (out, send), (a, b, s0), (_f64(st["dout"]), _f64(st["dsend"])))
    if kind == "core_train":
        st = prepare(case, seed)
        D = case["D"]
        q, delta, s0 = (_f64(st[k]).requires_grad_() for k in ("q", "delta", "s0"))
        gate = q[..., D:]
        u = q[..., :D] * _compete64(gate, 8)
        p = delta * torch.sigmoid(gate) + (1.0 - delta)
        out = _scan64(p, (1.0 - p) * u, s0)
        return (u.detach(), out.detach()) + torch.autograd.grad(
            (u, out), (q, delta, s0), (_f64(st["du"]), _f64(st["dst"])))
    with torch.no_grad():
        if kind == "sunny_step":
            return _sunny64(case, _tokens(case, seed, (case["B"], case["prompt"] + STEPS)).to(DEV), False)
        if kind == "sunny_prefill":
            return _sunny64(case, _tokens(case, seed, (case["B"], case["T"])).to(DEV), False)
        if kind == "sunny_forward":
            logits, s, hist = _sunny64(case, _tokens(case, seed, (case["B"], case["T"])).to(DEV), True)
            return logits, s, torch.flip(hist, [-2])
        if kind == "rwkv_step":
            return _rwkv64(case, _tokens(case, seed, (case["B"], case["prompt"] + STEPS)).to(DEV))
        logits, S, shift = _rwkv64(case, _tokens(case, seed, (case["T"],))[None].to(DEV))
        return logits[0], S, shift
