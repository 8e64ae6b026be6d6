"""Performance cases of the library: the calls a serving program makes, over the sizes it makes them at.

The model shapes are the repository's own: the Qwen2-0.5B decode stack (24 layers, hidden 896, vocab 151936), the
flow head (hidden 1024, 8 blocks) and the VAE decoder (24 layers, hidden 896, n_fft 3528).  Each
case is a dict with an "op" and its sizes:

  decode     one token of the whole 24-layer stack on a contiguous cache of `ctx` rows, 4-bit or bf16 weights,
             with the logits: what every generated token of one request costs
  prefill    a prompt of `L` rows through four layers (every layer of the stack does the same), in chunks of 512
             rows as a server sets them: what a request costs before its first token
  batch      one token of each of `n` requests of ragged length (`lo`..`hi` cached rows) through four layers of
             the stack over the paged cache, with the tied head and all logits
  flow       the flow head's ten Euler steps for `n` requests (n = 1: ming_cfm_sample, else the batched call)
  vae        the decoder from `T` latents to samples, bf16 or 4-bit weights: short chunks when audio is streamed,
             long ones when an utterance is decoded at once

Linear weights are N(0, 0.02) in bf16, quantized to groups of 64 at 4 bits where the case says so; the projections
back into the residual stream are scaled by 1 / sqrt(2 * 24), as such stacks are initialised.
"""
import ctypes
import importlib
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)
ming = importlib.import_module("ming-tts-serve_amd")
S = importlib.import_module("ming-tts-serve_amd.synthetic")

DEV = "cuda"
BF = torch.bfloat16
STD = 0.02
RES = STD / math.sqrt(2 * 24)
STACK_LAYERS = 4
CHUNK = 512
LM = S.LmSpec()
DIT = S.DitSpec()
VAE = S.VaeSpec()


# ---- the cases ------------------------------------------------------------------------------------------------


def listed():
    return [
        # a short prompt's first tokens: almost all of the step is hand-offs between dependent stages
        {"name": "decode_bf16_ctx77", "op": "decode", "quant": False, "ctx": 77},
        # the headline step: 4-bit weights, a cache of 2048 rows
        {"name": "decode_q4_ctx2048", "op": "decode", "quant": True, "ctx": 2048},
        # a sentence without a voice prompt
        {"name": "prefill_19", "op": "prefill", "L": 19},
        # a prompt that fills one chunk
        {"name": "prefill_512", "op": "prefill", "L": 512},
        # a long prompt: four chunks, the last one ragged
        {"name": "prefill_2041", "op": "prefill", "L": 2041},
        # a lightly loaded server
        {"name": "batch_13", "op": "batch", "n": 13, "lo": 64, "hi": 1500},
        # a full server
        {"name": "batch_64", "op": "batch", "n": 64, "lo": 64, "hi": 2047},
        # one request's flow head (the largest part of a token)
        {"name": "flow_1", "op": "flow", "n": 1, "temperature": 0.0},
        # a lightly loaded server, the stochastic sampler on
        {"name": "flow_13", "op": "flow", "n": 13, "temperature": 0.5},
        # a full server
        {"name": "flow_64", "op": "flow", "n": 64, "temperature": 0.0},
        # one audio chunk of a stream, 4-bit weights
        {"name": "vae_q4_7", "op": "vae", "quant": True, "T": 7},
        # eight seconds of audio decoded at once
        {"name": "vae_bf16_100", "op": "vae", "quant": False, "T": 100},
    ]


def draw(rng):
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    op = rng.choice(["decode", "prefill", "batch", "flow", "vae"])
    if op == "decode":
        return {"op": op, "quant": rng.random() < 0.7, "ctx": log_int(1, 4000)}
    if op == "prefill":
        return {"op": op, "L": log_int(2, 2041)}
    if op == "batch":
        hi = log_int(100, 2047)
        return {"op": op, "n": log_int(1, 64), "lo": rng.randint(0, hi // 2), "hi": hi}
    if op == "flow":
        return {"op": op, "n": log_int(1, 64), "temperature": rng.choice([0.0, 0.5, 1.0])}
    return {"op": op, "quant": rng.random() < 0.3, "T": log_int(1, 100)}


# ---- inputs, from the seed alone ----------------------------------------------------------------------------------


class Draws:
    def __init__(self, seed):
        self.g = torch.Generator(device=DEV)
        self.g.manual_seed(int(seed))

    def bf16(self, shape, std=1.0, mean=0.0):
        t = torch.randn(shape, device=DEV, generator=self.g)
        return t.mul_(std).add_(mean).to(BF)

    def ints(self, lo, hi, shape):
        return torch.randint(lo, hi, shape, device=DEV, generator=self.g, dtype=torch.int32)

    def linear(self, n, k, std, quant):
        """A bf16 weight [n, k], or the triplet (packed u32 as i32, scales, biases) of its groups of 64."""
        w = self.bf16((n, k), std)
        if not quant:
            return {"w": w}
        f = w.float().view(n, k // 64, 64)
        lo, hi = f.amin(-1), f.amax(-1)
        s, b = ((hi - lo) / 15).to(BF), lo.to(BF)
        q = ((f - b.float()[..., None]) / s.float()[..., None]).round_().clamp_(0, 15).to(torch.int32)
        q = q.view(n, k // 8, 8) << torch.arange(0, 32, 4, device=DEV, dtype=torch.int32)
        return {"w": q.sum(-1, dtype=torch.int32), "s": s, "b": b}


def full(t):
    """A linear's weight in 64 bits."""
    if "s" not in t:
        return t["w"].double()
    n, words = t["w"].shape
    q = (t["w"].unsqueeze(-1) >> torch.arange(0, 32, 4, device=DEV, dtype=torch.int32)) & 15
    q = q.view(n, words // 8, 64).double()
    return (q * t["s"].double().unsqueeze(-1) + t["b"].double().unsqueeze(-1)).view(n, words * 8)


def qwen_layer(d, spec, quant):
    h, kvd, inter = spec.hidden, spec.kvd, spec.inter
    lin = lambda n, k, std=STD: d.linear(n, k, std, quant)
    return {"ln1": d.bf16((h,), 0.1, 1.0), "ln2": d.bf16((h,), 0.1, 1.0), "q": lin(h, h), "k": lin(kvd, h),
            "v": lin(kvd, h), "o": lin(h, h, RES), "gate": lin(inter, h), "up": lin(inter, h),
            "down": lin(h, inter, RES), "bq": d.bf16((h,), STD), "bk": d.bf16((kvd,), STD),
            "bv": d.bf16((kvd,), STD)}


def lm_weights(d, layers, quant):
    return {"embed": d.linear(LM.vocab, LM.hidden, STD, quant), "norm": d.bf16((LM.hidden,), 0.1, 1.0),
            "layers": [qwen_layer(d, LM, quant) for _ in range(layers)]}


def cfm_weights(d):
    D, F, lat, H = DIT.hidden, DIT.ff, DIT.latent, DIT.lm_hidden
    lin = lambda n, k: (d.bf16((n, k), STD), d.bf16((n,), STD))
    block = lambda: {"n1": d.bf16((D,), 0.1, 1.0), "n2": d.bf16((D,), 0.1, 1.0), "q": lin(D, D), "k": lin(D, D),
                     "v": lin(D, D), "o": lin(D, D), "f1": lin(F, D), "f2": lin(D, F)}
    return {"blocks": [block() for _ in range(DIT.cfm_blocks)], "x": lin(D, lat), "c": lin(D, H), "t0": lin(D, 256),
            "t2": lin(D, D), "norm": d.bf16((D,), 0.1, 1.0), "final": lin(lat, D)}


def make(case, seed):
    """Everything a case's call reads, as tensors."""
    d, op = Draws(seed), case["op"]
    if op == "decode":
        shape = (LM.n_layers, LM.kv_heads, case["ctx"] + 1, LM.head_dim)
        return {"lm": lm_weights(d, LM.n_layers, case["quant"]), "k": d.bf16(shape), "v": d.bf16(shape),
                "token": d.ints(0, LM.vocab, (1,))}
    if op == "prefill":
        pages = (case["L"] + 63) // 64
        return {"lm": lm_weights(d, STACK_LAYERS, True), "tokens": d.ints(0, LM.vocab, (case["L"],)),
                "table": torch.randperm(pages, device=DEV, generator=d.g).to(torch.int32).view(1, pages)}
    if op == "batch":
        n, per = case["n"], case["hi"] // 64 + 1
        pool = (STACK_LAYERS, n * per, LM.kv_heads, 64, 64)
        return {"lm": lm_weights(d, STACK_LAYERS, True), "tokens": d.ints(0, LM.vocab, (n,)),
                "table": torch.randperm(n * per, device=DEV, generator=d.g).to(torch.int32).view(n, per),
                "pos": d.ints(case["lo"], case["hi"] + 1, (n,)), "k": d.bf16(pool), "v": d.bf16(pool)}
    if op == "flow":
        n = case["n"]
        return {"cfm": cfm_weights(d), "z": d.bf16((n, DIT.lm_hidden)), "hist": d.bf16((n, DIT.latent)),
                "noise": d.bf16((n, DIT.latent)), "sde": d.bf16((n, 10, DIT.latent))}
    q = case["quant"]
    P = VAE.n_fft + 2
    return {"fc1": d.linear(VAE.hidden, VAE.latent, 0.1, q), "fc1_bias": d.bf16((VAE.hidden,), STD),
            "layers": [qwen_layer(d, VAE, q) for _ in range(VAE.n_layers)], "norm": d.bf16((VAE.hidden,), 0.1, 1.0),
            "head": d.linear(P, VAE.hidden, STD, q), "head_bias": d.bf16((P,), STD),
            "window": torch.from_numpy(S.hann_window(VAE.n_fft)).to(DEV), "latents": d.bf16((case["T"], VAE.latent))}


# ---- what a program keeps between calls ---------------------------------------------------------------------------


def _lin(t):
    return ming.linear(t["w"], t["s"], t["b"]) if "s" in t else ming.linear(t["w"])


def _layer(l):
    return ming.LmLayerW(l["ln1"].data_ptr(), l["ln2"].data_ptr(), *(_lin(l[k]) for k in
                         ("q", "k", "v", "o", "gate", "up", "down")), *(l[k].data_ptr() for k in ("bq", "bk", "bv")))


def _lm(ctx, w):
    spec = S.LmSpec(n_layers=len(w["layers"]))
    e = _lin(w["embed"])
    return spec, ming.LmModel(ctx, spec.cfg(), [_layer(l) for l in w["layers"]], w["norm"], e, e)


def _pages(spec, i, n):
    pages = S.PagedKv(spec, n, i["table"].shape[1])
    pages.set_table(i["table"].cpu().numpy())
    return pages


def prepare(case, seed):
    op, i = case["op"], make(case, seed)
    ctx = ming.Context(0)
    ctx.set_exclusive(True)  # the serving process has the device to itself
    st = {"case": case, "in": i, "ctx": ctx}
    hid = lambda n: torch.zeros((n, LM.hidden), dtype=BF, device=DEV)
    if op == "decode":
        spec, st["model"] = _lm(ctx, i["lm"])
        st["kv"] = ming.Kv(i["k"].data_ptr(), i["v"].data_ptr(), spec.n_layers, spec.kv_heads, spec.head_dim,
                           case["ctx"] + 1, case["ctx"])
        st["hidden"] = hid(1)
        st["logits"] = torch.zeros(LM.vocab, dtype=torch.float32, device=DEV)
        st["argmax"] = torch.zeros(1, dtype=torch.int32, device=DEV)
    elif op == "prefill":
        L = case["L"]
        spec, st["model"] = _lm(ctx, i["lm"])
        st["pages"] = _pages(spec, i, 1)
        st["batch"] = ming.LmBatch(st["model"], CHUNK, 64 * i["table"].shape[1])
        st["hidden"] = hid(L)
    elif op == "batch":
        n = case["n"]
        spec, st["model"] = _lm(ctx, i["lm"])
        st["pages"] = _pages(spec, i, n)
        st["pages"].k.copy_(i["k"])
        st["pages"].v.copy_(i["v"])
        st["batch"] = ming.LmBatch(st["model"], n, 64 * i["table"].shape[1])
        st["pos"] = i["pos"].clone()
        st["hidden"] = hid(n)
        st["logits"] = torch.zeros((n, LM.vocab), dtype=torch.float32, device=DEV)
    elif op == "flow":
        w, names = i["cfm"], ("q", "k", "v", "o", "f1", "f2")
        blocks = (ming.DitBlockW * DIT.cfm_blocks)(*(
            ming.DitBlockW(b["n1"].data_ptr(), b["n2"].data_ptr(), *(ming.linear(b[k][0]) for k in names),
                           *(b[k][1].data_ptr() for k in names)) for b in w["blocks"]))
        st["keep"] = (blocks, DIT.inv_freq())
        st["model"] = ming.CfmModel(ctx, ming.CfmW(
            DIT.cfg(), DIT.cfm_blocks, ctypes.cast(blocks, ctypes.c_void_p), st["keep"][1].ctypes.data,
            *(ming.linear(w[k][0]) for k in ("x", "c", "t0", "t2", "final")),
            *(w[k][1].data_ptr() for k in ("x", "c", "t0", "t2")), w["norm"].data_ptr(), w["final"][1].data_ptr()))
        st["out"] = torch.zeros((case["n"], DIT.latent), dtype=BF, device=DEV)
    else:
        layers = (ming.LmLayerW * VAE.n_layers)(*(_layer(l) for l in i["layers"]))
        st["keep"] = layers
        w = ming.VaeW(_lin(i["fc1"]), i["fc1_bias"].data_ptr(), ctypes.cast(layers, ctypes.c_void_p),
                      i["norm"].data_ptr(), _lin(i["head"]), i["head_bias"].data_ptr(), i["window"].data_ptr())
        st["model"] = ming.VaeModel(ctx, VAE.cfg(), w, case["T"])
        st["out"] = torch.zeros(case["T"] * VAE.patch * VAE.hop, dtype=torch.float32, device=DEV)
    return st


def run(st):
    op, i, case = st["case"]["op"], st["in"], st["case"]
    if op == "decode":
        st["kv"].len = case["ctx"]
        st["model"].step(st["kv"], token=i["token"], hidden=st["hidden"], logits=st["logits"], argmax=st["argmax"])
        return {"logits": st["logits"], "hidden": st["hidden"], "k": i["k"], "v": i["v"]}
    if op == "prefill":
        st["batch"].prefill(st["pages"], st["pages"].table[0], 0, tokens=i["tokens"], hidden=st["hidden"])
        return {"hidden": st["hidden"], "k": st["pages"].k, "v": st["pages"].v}
    if op == "batch":
        st["pos"].copy_(i["pos"])  # the scheduler's positions of this step
        st["batch"].step(st["pages"], st["pages"].table, st["pos"], tokens=i["tokens"], hidden=st["hidden"],
                         logits=st["logits"])
        return {"logits": st["logits"], "hidden": st["hidden"], "k": st["pages"].k, "v": st["pages"].v}
    if op == "flow":
        a = (i["z"], i["hist"], i["noise"], i["sde"], 2.0, 0.25, case["temperature"], st["out"])
        st["model"].sample(*a) if case["n"] == 1 else st["model"].sample_batch(case["n"], *a)
        return {"latents": st["out"]}
    st["model"].decode(case["T"], i["latents"], st["out"])
    return {"wave": st["out"]}


# ---- what a pass cannot do without ----------------------------------------------------------------------------------


def work(case):
    op, H, kvd, inter = case["op"], LM.hidden, LM.kvd, LM.inter
    layer, head = 2 * H * H + 2 * kvd * H + 3 * H * inter, LM.vocab * H
    row = 2 * kvd * 2  # one cached position of one layer
    if op == "decode":
        b = 0.5625 if case["quant"] else 2.0
        c, n = case["ctx"], LM.n_layers
        return {"bytes": int((n * layer + head) * b + n * row * (c + 1) + LM.vocab * 4 + 2 * H),
                "flops": 2 * (n * layer + head) + n * 4 * H * (c + 1)}
    if op == "prefill":
        n, L = STACK_LAYERS, case["L"]
        return {"bytes": int(n * layer * 0.5625 + L * (H * 0.5625 + n * row + 2 * H)),
                "flops": 2 * n * layer * L + n * 4 * H * L * (L + 1) // 2}
    if op == "batch":
        n, seqs, mean = STACK_LAYERS, case["n"], (case["lo"] + case["hi"]) // 2
        return {"bytes": int((n * layer + head) * 0.5625 + seqs * (n * row * (mean + 1) + LM.vocab * 4 + 2 * H)),
                "flops": 2 * (n * layer + head) * seqs + n * 4 * H * seqs * (mean + 1)}
    if op == "flow":
        D, F, lat, n = DIT.hidden, DIT.ff, DIT.latent, case["n"]
        block = 4 * D * D + 2 * D * F
        # the weights are read once a sample; each Euler step takes six rows a request through every block
        return {"bytes": int(2 * (DIT.cfm_blocks * block + D * (DIT.lm_hidden + 2 * lat)) + n * 2 * (H + 13 * lat)),
                "flops": 10 * 2 * n * (6 * DIT.cfm_blocks * block + 3 * D * lat)}
    F, P = case["T"] * VAE.patch, VAE.n_fft + 2
    params = VAE.n_layers * layer + P * H + H * VAE.latent
    # the inverse transform as the 5 n log2 n operations of a fast one
    return {"bytes": int(params * (0.5625 if case["quant"] else 2.0) + F * VAE.hop * 4 + case["T"] * VAE.latent * 2),
            "flops": int(2 * F * (params + VAE.n_layers * 2 * H * min(F, VAE.window))
                         + F * 2.5 * VAE.n_fft * math.log2(VAE.n_fft))}


# ---- how exact a pass has to be ---------------------------------------------------------------------------------------


def tolerance(case):
    # Measured distance to exact(): decode 0.034 (24 layers of bf16 roundings), prefill and batch 0.013 (four layers),
    # flow 0.008 (ten Euler steps of eight blocks).  Another order of the f32 sums takes some of those roundings
    # elsewhere, so two correct implementations can be about that far apart.  The decoder is 32-bit throughout but for
    # fc1, whose bf16 result turns a last-bit difference into one of 2^-9 in that value: 8e-7, and 3.5e-5 where one does.
    op = case["op"]
    if op == "decode":
        return {"rel": 0.03, "max": 0.3}
    if op in ("prefill", "batch"):
        return {"rel": 0.02, "max": 0.2}
    if op == "flow":
        return {"rel": 0.03, "max": 0.3}
    return {"rel": 1e-4, "max": 4e-3}


# ---- the same values in 64 bits -----------------------------------------------------------------------------------------


def _rms(x, w, eps=1e-6):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps) * w.double()


def _rope(x, pos):
    """Heads x [rows, heads, 64] at positions pos [rows]: pairs (d, d + 32)."""
    inv = 1e6 ** (-torch.arange(32, device=DEV, dtype=torch.float64) / 32)
    a = pos.double()[:, None, None] * inv
    x1, x2 = x[..., :32], x[..., 32:]
    return torch.cat([x1 * a.cos() - x2 * a.sin(), x1 * a.sin() + x2 * a.cos()], -1)


def _attend(q, k, v, seen):
    """q [rows, 14, 64] on k, v [keys, 2, 64]; seen [rows, keys]."""
    rows, keys = q.shape[0], k.shape[0]
    q = q.view(rows, 2, 7, 64).permute(1, 2, 0, 3).reshape(2, 7 * rows, 64)
    s = torch.matmul(q, k.permute(1, 2, 0).contiguous()).view(2, 7, rows, keys) / 8
    s = s.masked_fill_(~seen, -math.inf).softmax(-1).view(2, 7 * rows, keys)
    o = torch.matmul(s, v.permute(1, 0, 2).contiguous())
    return o.view(2, 7, rows, 64).permute(2, 0, 1, 3).reshape(rows, 896)


def _qkv(x, l, pos):
    h = _rms(x, l["ln1"])
    q, k, v = (h @ full(l[a]).T + l["b" + a].double() for a in "qkv")
    return _rope(q.view(-1, 14, 64), pos), _rope(k.view(-1, 2, 64), pos), v.view(-1, 2, 64)


def _rest(x, o, l):
    x = x + o @ full(l["o"]).T
    h = _rms(x, l["ln2"])
    return x + (torch.nn.functional.silu(h @ full(l["gate"]).T) * (h @ full(l["up"]).T)) @ full(l["down"]).T


def _rows(t, tokens):
    idx = tokens.long()
    return full({k: v[idx] for k, v in t.items()})


def _logits(h, t):
    return torch.cat([h @ full({k: v[r:r + 16384] for k, v in t.items()}).T for r in range(0, LM.vocab, 16384)], -1)


def exact(case, seed):
    op, i = case["op"], make(case, seed)
    if op == "decode":
        c, w = case["ctx"], i["lm"]
        x, pos = _rows(w["embed"], i["token"]), torch.tensor([c], device=DEV)
        kc, vc = i["k"].double(), i["v"].double()
        for n, l in enumerate(w["layers"]):
            q, k, v = _qkv(x, l, pos)
            kc[n, :, c], vc[n, :, c] = k[0], v[0]
            x = _rest(x, _attend(q, kc[n].transpose(0, 1), vc[n].transpose(0, 1), torch.ones(1, c + 1, dtype=torch.bool, device=DEV)), l)
        h = _rms(x, w["norm"])
        return {"logits": _logits(h, w["embed"])[0], "hidden": h, "k": kc, "v": vc}
    if op == "prefill":
        L, w, table = case["L"], i["lm"], i["table"][0].long()
        pages = table.numel()
        x, pos = _rows(w["embed"], i["tokens"]), torch.arange(L, device=DEV)
        kp = torch.zeros((STACK_LAYERS, pages, 2, 64, 64), dtype=torch.float64, device=DEV)
        vp = torch.zeros_like(kp)
        for n, l in enumerate(w["layers"]):
            q, k, v = _qkv(x, l, pos)
            kp[n, table[pos // 64], :, pos % 64] = k
            vp[n, table[pos // 64], :, :, pos % 64] = v
            x = _rest(x, _attend(q, k, v, pos[None, :] <= pos[:, None]), l)
        return {"hidden": _rms(x, w["norm"]), "k": kp, "v": vp}
    if op == "batch":
        w, table, pos = i["lm"], i["table"].long(), i["pos"].long()
        x = _rows(w["embed"], i["tokens"])
        kp, vp = i["k"].double(), i["v"].double()
        at = table.gather(1, (pos // 64)[:, None])[:, 0]
        for n, l in enumerate(w["layers"]):
            q, k, v = _qkv(x, l, pos)
            kp[n, at, :, pos % 64] = k
            vp[n, at, :, :, pos % 64] = v
            o = []
            for s, c in enumerate(pos.tolist()):
                t = table[s, :c // 64 + 1]
                ks = kp[n, t].permute(0, 2, 1, 3).reshape(-1, 2, 64)[:c + 1]
                vs = vp[n, t].permute(0, 3, 1, 2).reshape(-1, 2, 64)[:c + 1]
                o.append(_attend(q[s:s + 1], ks, vs, torch.ones(1, c + 1, dtype=torch.bool, device=DEV)))
            x = _rest(x, torch.cat(o), l)
        h = _rms(x, w["norm"])
        return {"logits": _logits(h, w["embed"]), "hidden": h, "k": kp, "v": vp}
    return _exact_flow(case, i) if op == "flow" else _exact_vae(case, i)


def _schedule():
    """The schedule's bf16 constants: t (11), dt and sqrt |dt| (10)."""
    r = lambda v: v.to(BF).float()
    t = torch.tensor([0, 2, 4, 6, 8, 12, 16, 20, 24, 28, 32], dtype=torch.float32) / 32
    sway = r(r(r(torch.cos(r(r(torch.tensor(math.pi / 2)) * t))) - 1) + t)
    t = r(t - sway)
    dt = r(t[1:] - t[:-1])
    return t, dt, r(dt.abs().sqrt())


def _exact_flow(case, i):
    w, n, D = i["cfm"], case["n"], DIT.hidden
    lin = lambda x, p: x @ p[0].double().T + p[1].double()
    t, dt, sq = _schedule()
    shift = float(torch.tensor(0.25 * math.sqrt(case["temperature"])).to(BF))
    inv = torch.from_numpy(DIT.inv_freq()).to(DEV).double()
    ang = torch.arange(3, device=DEV, dtype=torch.float64)[:, None] * inv
    cos, sin = ang.cos()[:, None], ang.sin()[:, None]

    def rot(x):
        e, o = x[..., 0::2], x[..., 1::2]
        return torch.stack([e * cos - o * sin, e * sin + o * cos], -1).flatten(-2)

    freq = torch.exp(-torch.arange(128, device=DEV, dtype=torch.float64) * (math.log(1e4) / 127))
    ce = torch.stack([lin(i["z"].double(), w["c"]), w["c"][1].double().expand(n, D)], 1)  # [n, 2, D]
    xh = lin(i["hist"].double(), w["x"])
    y = i["noise"].double()
    for s in range(10):
        a = float((1000 * t[s]).to(BF)) * freq
        te = lin(torch.nn.functional.silu(lin(torch.cat([a.sin(), a.cos()]), w["t0"])), w["t2"])
        h = torch.stack([te + ce, xh[:, None].expand(n, 2, D), lin(y, w["x"])[:, None].expand(n, 2, D)], 2)
        for b in w["blocks"]:
            g = _rms(h, b["n1"])
            q, k, v = (lin(g, b[c]).view(n, 2, 3, 16, 64) for c in "qkv")
            q, k, v = (c.permute(0, 1, 3, 2, 4).contiguous() for c in (rot(q), rot(k), v))
            p = (torch.matmul(q, k.transpose(-1, -2).contiguous()) / 8).softmax(-1)
            h = h + lin(torch.matmul(p, v).permute(0, 1, 3, 2, 4).reshape(n, 2, 3, D), b["o"])
            f = torch.nn.functional.gelu(lin(_rms(h, b["n2"]), b["f1"]), approximate="tanh")
            h = h + lin(f, b["f2"])
        o = lin(_rms(h[:, :, 2], w["norm"]), w["final"])
        y = y + float(dt[s]) * (o[:, 0] + (o[:, 0] - o[:, 1]) * 2.0)
        if shift:
            y = y + shift * float(sq[s]) * i["sde"][:, s].double()
    return {"latents": y}


def _exact_vae(case, i):
    T, N, hop = case["T"], VAE.n_fft, VAE.hop
    F = T * VAE.patch
    # fc1 works in bf16 by definition; all that follows is 32-bit
    x = i["latents"].double() @ full(i["fc1"]).T
    x = ((x.to(BF).double() if case["quant"] else x) + i["fc1_bias"].double()).to(BF).double()
    at = (torch.arange(F, device=DEV, dtype=torch.float64) + 0.5) / VAE.patch - 0.5
    left = at.floor()
    wr = (at - left)[:, None]
    left = left.long()
    x = x[left.clamp(0, T - 1)] * (1 - wr) + x[(left + 1).clamp(0, T - 1)] * wr
    pos = torch.arange(F, device=DEV)
    seen = (pos[None, :] <= pos[:, None]) & (pos[None, :] > pos[:, None] - VAE.window)
    for l in i["layers"]:
        q, k, v = _qkv(x, l, pos)
        x = _rest(x, _attend(q, k, v, seen), l)
    p = _rms(x, i["norm"]) @ full(i["head"]).T + i["head_bias"].double()
    nb = N // 2 + 1
    mag, ph = p[:, :nb].exp().clamp(max=100.0).cpu().numpy(), p[:, nb:].cpu().numpy()
    win = i["window"].double().cpu().numpy()
    fr = np.fft.irfft(mag * np.cos(ph) + 1j * mag * np.sin(ph), n=N, axis=-1) * win
    wave, env = np.zeros((F + 3) * hop), np.zeros((F + 3) * hop)
    for f in range(F):
        wave[f * hop:f * hop + N] += fr[f]
        env[f * hop:f * hop + N] += win * win
    pad = (N - hop) // 2
    out = wave[pad:pad + F * hop] / np.maximum(env[pad:pad + F * hop], 1e-11)
    return {"wave": torch.from_numpy(out)}
