"""The work that a user of this package has it do, as measurable cases.

Kinds of case (each through a public entry point, at sizes of the repository's own configurations):

* ``decode``          one single-token step of the delta rule for B streams (``decode_step``), state in place;
* ``block``           one single-token step of the whole mixer block for B streams (``fused_decode_step``);
* ``serving_decode``  the serving layer's static decode step, captured once into a graph and replayed a step;
* ``serving_extend``  the serving layer's eager call: fresh prompts beside requests that continue their slots;
* ``prefill``         chunked prefill of B sequences of T tokens (``chunk_fwd``), bf16 or fp32;
* ``packed``          chunked prefill of packed sequences of different lengths;
* ``layer``           the model's mixer layer (``layer.gdn``): projections, conv, delta rule, gated norm;
* ``attnres``         the residual routing over S sources;
* ``accent``          the accent adapters' shift of a projection's rows, in place.

``exact`` states each result in float64 from the definitions, without this package's code.
"""

from __future__ import annotations

import importlib
import itertools
import math
from types import SimpleNamespace

import torch
import torch.nn.functional as F

DTYPES = {"bf16": torch.bfloat16, "f32": torch.float32}
CHUNK = 64
HEADS, HEAD_DIM, HIDDEN = 4, 128, 1024  # the release model's mixer
INNER = HEADS * HEAD_DIM


def listed():
    return [
        # a couple of voices spoken at once: latency and the launch itself count
        {"name": "decode_b2", "kind": "decode", "B": 2, "Hk": 16, "Hv": 16, "D": 128, "dtype": "bf16"},
        # the headline decode step: a server's batch of streams
        {"name": "decode_b64", "kind": "decode", "B": 64, "Hk": 16, "Hv": 16, "D": 128, "dtype": "bf16"},
        # streaming decode of the whole block for a large batch, q/k heads shared by two value heads
        {"name": "block_b256", "kind": "block", "B": 256, "Hk": 8, "Hv": 16, "dtype": "bf16"},
        # a serving engine's decode step of 32 requests with 100-row prompts, one graph replay a step
        {"name": "serving_decode_bs32", "kind": "serving_decode", "bs": 32, "prompt": 100},
        # a serving engine's eager step: four new prompts and two requests that go on, ragged lengths
        {"name": "serving_extend", "kind": "serving_extend", "rows": "301,77,512,40,128,9", "cached": "0,0,0,0,90,200"},
        # one long prompt, the headline prefill
        {"name": "prefill_t4096", "kind": "prefill", "B": 1, "T": 4096, "Hk": 16, "Hv": 16, "D": 128, "dtype": "bf16",
         "raw": False},
        # a batch of prompts of every length up to 2048 packed into one stream, with states carried in
        {"name": "packed_32", "kind": "packed", "n": 32, "lo": 64, "hi": 2048, "pick": 1004, "Hk": 16, "Hv": 16},
        # the fp32 model's short prompt (the configuration that is compared with the CPU)
        {"name": "prefill_f32_t256", "kind": "prefill", "B": 1, "T": 256, "Hk": 4, "Hv": 4, "D": 64, "dtype": "f32",
         "raw": False},
        # the fp32 model's long prompt
        {"name": "prefill_f32_t4096", "kind": "prefill", "B": 1, "T": 4096, "Hk": 16, "Hv": 16, "D": 128,
         "dtype": "f32", "raw": False},
        # the mixer layer of the release model on a long prompt, projections included
        {"name": "layer_t4096", "kind": "layer", "T": 4096, "carried": False},
        # the last residual mix of the release model (embedding + 22 sublayers) over a long prompt
        {"name": "attnres_s23", "kind": "attnres", "S": 23, "T": 4096, "dim": 1024, "dtype": "bf16"},
        # accent adapters on the mixer's input projection over a long prompt
        {"name": "accent_4096", "kind": "accent", "rows": 4096, "n_in": 1024, "n_out": 2056, "K": 64},
    ]


def _log(rng, lo, hi):
    """A whole number of [lo, hi], spread over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["decode", "block", "serving_decode", "serving_extend", "prefill", "prefill", "packed", "layer",
                       "layer", "attnres", "accent"])
    if kind == "decode":
        hv = rng.choice([4, 8, 16])
        return {"kind": kind, "B": _log(rng, 1, 256), "Hk": hv // rng.choice([1, 2]), "Hv": hv,
                "D": rng.choice([128, 128, 64]), "dtype": rng.choice(["bf16", "bf16", "f32"])}
    if kind == "block":
        hk, hv = rng.choice([(4, 4), (4, 8), (8, 16), (8, 8)])
        return {"kind": kind, "B": _log(rng, 1, 256), "Hk": hk, "Hv": hv, "dtype": rng.choice(["bf16", "bf16", "f32"])}
    if kind == "serving_decode":
        return {"kind": kind, "bs": _log(rng, 1, 64), "prompt": rng.randint(5, 200)}
    if kind == "serving_extend":
        n = rng.randint(1, 8)
        return {"kind": kind, "rows": ",".join(str(_log(rng, 1, 700)) for _ in range(n)),
                "cached": ",".join(str(rng.choice([0, 0, rng.randint(1, 300)])) for _ in range(n))}
    if kind == "prefill":
        hv, dtype = rng.choice([4, 8, 16]), rng.choice(["bf16", "bf16", "f32"])
        B = rng.choice([1, 1, 2, 4])
        return {"kind": kind, "B": B, "T": _log(rng, 40, 65536 // (hv * B)), "Hk": hv // rng.choice([1, 1, 2]),
                "Hv": hv, "D": rng.choice([128, 128, 64]), "dtype": dtype, "raw": rng.choice([False, True])}
    if kind == "packed":
        hv = rng.choice([4, 8, 16])
        n = rng.randint(2, 32)
        return {"kind": kind, "n": n, "lo": rng.randint(1, 100), "hi": _log(rng, 128, 1800), "pick": rng.randrange(10**6),
                "Hk": hv // rng.choice([1, 1, 2]), "Hv": hv}
    if kind == "layer":
        return {"kind": kind, "T": _log(rng, 1, 4096), "carried": rng.choice([False, True])}
    if kind == "attnres":
        return {"kind": kind, "S": rng.randint(2, 23), "T": _log(rng, 1, 4096), "dim": rng.choice([1024, 1024, 512]),
                "dtype": rng.choice(["bf16", "bf16", "f32"])}
    n_in, n_out = rng.choice([(1024, 2056), (512, 1024)])
    return {"kind": kind, "rows": _log(rng, 1, 4096), "n_in": n_in, "n_out": n_out, "K": rng.choice([8, 16, 24, 64])}


# ------------------------------------------------------------------------------------------------- inputs


def _lengths(c):
    g = torch.Generator().manual_seed(c["pick"])
    return torch.randint(c["lo"], c["hi"] + 1, (c["n"],), generator=g).tolist()


def _ints(text):
    return [int(x) for x in text.split(",")]


class _Rand:
    """Seeded normal tensors on the GPU."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(int(seed))

    def __call__(self, *shape, dtype=torch.float32, std=1.0, mean=0.0):
        return (torch.randn(*shape, generator=self.g, device="cuda") * std + mean).to(dtype)


def _unit(x):
    return x * torch.rsqrt(x.square().sum(-1, keepdim=True) + 1e-6)


def _delta_inputs(c, r, B, T, n_states):
    """q, k, v, g, beta and the start states of a delta-rule call: unit q, k, log decays and betas of the
    model's gate; with ``raw`` the rows before their norm and the gate's own inputs."""
    dt = DTYPES[c.get("dtype", "bf16")]
    D, hk, hv = c.get("D", 128), c["Hk"], c["Hv"]
    d = {"q": r(B, T, hk, D), "k": r(B, T, hk, D), "v": r(B, T, hv, D, dtype=dt)}
    a, b = r(B, T, hv), r(B, T, hv)
    if c.get("raw"):
        d.update(q=d["q"].to(dt), k=d["k"].to(dt), g=a.to(dt), beta=b.to(dt), A_log=r(hv, std=0.2), dt_bias=r(hv, std=0.2))
    else:
        d.update(q=_unit(d["q"]).to(dt), k=_unit(d["k"]).to(dt), g=-F.softplus(a), beta=b.sigmoid())
    if n_states:
        d["s0"] = r(n_states, hv, D, D, std=0.02)
    return d


def _mixer_weights(r):
    """The release model's mixer weights (bf16; the gate's vectors fp32)."""
    bf = torch.bfloat16
    return {"in_proj": r(4 * INNER + 2 * HEADS, HIDDEN, std=0.02, dtype=bf), "conv": r(3 * INNER, 1, 4, std=0.2, dtype=bf),
            "out_weight": r(HEAD_DIM, std=0.1, mean=1.0, dtype=bf), "A_log": r(HEADS, std=0.2),
            "dt_bias": r(HEADS, std=0.2), "wo": r(HIDDEN, INNER, std=0.02, dtype=bf)}


def _inputs(c, seed):
    """A case's inputs as tensors on the GPU, from the seed alone."""
    r, kind = _Rand(seed), c["kind"]
    dt = DTYPES[c.get("dtype", "bf16")]
    if kind == "decode":
        return _delta_inputs(c, r, c["B"], 1, c["B"])
    if kind == "prefill":
        return _delta_inputs(c, r, c["B"], c["T"], 0)
    if kind == "packed":
        return _delta_inputs(c, r, 1, sum(_lengths(c)), c["n"])
    if kind == "block":
        B, hk, hv, D = c["B"], c["Hk"], c["Hv"], HEAD_DIM
        C = 2 * hk * D + hv * D
        return {"x": r(B, C, dtype=dt), "z": r(B, hv, D, dtype=dt), "a": r(B, hv, dtype=dt), "b": r(B, hv, dtype=dt),
                "w": r(C, 4, std=0.2, dtype=dt), "cache": r(B, C, 3, dtype=dt), "state": r(B, hv, D, D, std=0.02),
                "nw": r(D, std=0.1, mean=1.0, dtype=dt), "A_log": r(hv, std=0.2), "dt_bias": r(hv, std=0.2)}
    if kind == "serving_decode":
        return {"w": _mixer_weights(r), "prompts": r(c["bs"], c["prompt"], HIDDEN, dtype=dt), "x": r(c["bs"], HIDDEN, dtype=dt)}
    if kind == "serving_extend":
        rows, cached = _ints(c["rows"]), _ints(c["cached"])
        return {"w": _mixer_weights(r), "before": [r(n, HIDDEN, dtype=dt) for n in cached], "x": r(sum(rows), HIDDEN, dtype=dt)}
    if kind == "layer":
        d = {"w": _mixer_weights(r), "x": r(c["T"], HIDDEN, dtype=dt)}
        if c["carried"]:
            d.update(conv=r(3 * INNER, 3, dtype=dt), state=r(HEADS, HEAD_DIM, HEAD_DIM, std=0.02))
        return d
    if kind == "attnres":
        return {"sources": [r(c["T"], c["dim"], dtype=dt) for _ in range(c["S"])], "query": r(c["dim"], std=0.3, dtype=dt)}
    if kind == "accent":
        rows, n_in, n_out, K = c["rows"], c["n_in"], c["n_out"], c["K"]
        on = torch.rand(rows, K, generator=r.g, device="cuda") < 0.5
        return {"x": r(rows, n_in, dtype=dt), "down": r(K, n_in, std=n_in**-0.5, dtype=dt), "up": r(K, n_out, std=K**-0.5, dtype=dt),
                "mask": on.to(dt), "y": r(rows, n_out, dtype=dt)}
    raise ValueError(kind)


# ---------------------------------------------------------------------------------------- prepare and run


def _package(name=""):
    return importlib.import_module("zonos3-mini_amd" + name)


def _tables(lengths):
    """cu_seqlens and the chunk table of packed sequences, as a program with the lengths on the host makes them."""
    cu = list(itertools.accumulate(lengths, initial=0))
    rows = [[i, j] for i, n in enumerate(lengths) for j in range(-(-n // CHUNK))]
    return (torch.tensor(cu, dtype=torch.int32, device="cuda"), torch.tensor(rows, dtype=torch.int32, device="cuda"))


def _request(slot, cached, new):
    return SimpleNamespace(table_idx=slot, uid=slot, is_cfg_uncond=False, cached_len=cached, device_len=cached + new,
                           extend_len=new)


def _serving_layer(w, slots):
    serving = _package(".serving")
    batch = SimpleNamespace(is_decode=False, padded_size=0, gdn_prefill=None, reqs=[], padded_reqs=[])
    layer = serving.OriginalGDN(SimpleNamespace(hidden_size=HIDDEN), 0, batch_source=lambda: batch)
    for name in ("in_proj", "conv", "wo"):
        getattr(layer, name).weight = w[name]
    layer.out_weight, layer.A_log, layer.dt_bias = w["out_weight"], w["A_log"], w["dt_bias"]
    layer.allocate_cache(slots, "cuda", torch.bfloat16)
    return layer, batch


def _caches(layer):
    return {"commit_state": layer._recurrent_state, "commit_conv": layer._conv_state, "live_state": layer._live_state,
            "live_conv": layer._live_conv, "win_len": layer._win_len}


def prepare(case, seed):
    c, d = case, _inputs(case, seed)
    kind = c["kind"]
    s = {"c": c, "d": d, "gdn": _package()}
    if kind == "decode":
        for n in ("q", "k", "v", "g", "beta"):
            d[n] = d[n][:, 0].contiguous()
    elif kind == "packed":
        s["cu"], s["chunks"] = _tables(_lengths(c))
    elif kind == "serving_decode":
        bs, P = c["bs"], c["prompt"]
        layer, batch = _serving_layer(d["w"], bs)
        batch.reqs = batch.padded_reqs = [_request(i, 0, P) for i in range(bs)]
        layer.forward(d["prompts"].reshape(bs * P, HIDDEN))
        slots = torch.arange(bs, device="cuda")
        layer.enable_graph_decode(slots, type(layer).static_tables("cuda", [bs]))
        layer.set_static_mode(True)
        batch.is_decode, batch.padded_size = True, bs
        kept = [layer._recurrent_state, layer._conv_state, layer._live_state, layer._live_conv, layer._window, layer._win_len]
        saved = [t.clone() for t in kept]
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):  # the engine's warm-up, then the capture
            layer.forward(d["x"])
        torch.cuda.current_stream().wait_stream(side)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            y = layer.forward(d["x"])
        for t, was in zip(kept, saved):
            t.copy_(was)
        s.update(layer=layer, batch=batch, slots=slots, graph=graph, y=y)
    elif kind == "serving_extend":
        rows, cached = _ints(c["rows"]), _ints(c["cached"])
        layer, batch = _serving_layer(d["w"], len(rows))
        going = [i for i, n in enumerate(cached) if n]
        if going:
            batch.reqs = batch.padded_reqs = [_request(i, 0, cached[i]) for i in going]
            layer.forward(torch.cat([d["before"][i] for i in going]))
        s.update(layer=layer, batch=batch, rows=rows, at=list(cached), going=going)
    elif kind == "layer":
        w = d["w"]
        att = SimpleNamespace(in_proj=SimpleNamespace(weight=w["in_proj"]), conv=SimpleNamespace(weight=w["conv"]),
                              out_weight=w["out_weight"], A_log=w["A_log"], dt_bias=w["dt_bias"],
                              wo=SimpleNamespace(weight=w["wo"]))
        model = SimpleNamespace(layers=[SimpleNamespace(attention=att)], _capture=None,
                                _lin=lambda name, x, weight, bias=None: F.linear(x, weight, bias))
        _package(".layer").patch(model)
        s["model"] = model
    return s


def run(state):
    c, d, gdn = state["c"], state["d"], state["gdn"]
    kind = c["kind"]
    if kind == "decode":
        o = gdn.decode_step(d["q"], d["k"], d["v"], d["g"], d["beta"], d["s0"])
        return {"o": o, "state": d["s0"]}
    if kind == "block":
        out = gdn.fused_decode_step(d["x"], d["z"], d["a"], d["b"], d["w"], d["cache"], d["state"], d["nw"], d["A_log"],
                                    d["dt_bias"])
        return {"out": out, "cache": d["cache"], "state": d["state"]}
    if kind == "prefill":
        more = dict(A_log=d["A_log"], dt_bias=d["dt_bias"], use_qk_l2norm=True, beta_is_logit=True) if c["raw"] else {}
        o, final = gdn.chunk_fwd(d["q"], d["k"], d["v"], d["g"], d["beta"], **more)
        return {"o": o, "state": final}
    if kind == "packed":
        o, final = gdn.chunk_fwd(d["q"], d["k"], d["v"], d["g"], d["beta"], initial_state=d["s0"], cu_seqlens=state["cu"],
                                 chunk_indices=state["chunks"])
        return {"o": o, "state": final}
    if kind == "serving_decode":
        state["graph"].replay()
        return {"y": state["y"], **_caches(state["layer"])}
    if kind == "serving_extend":
        layer, batch, rows, at = state["layer"], state["batch"], state["rows"], state["at"]
        batch.reqs = batch.padded_reqs = [_request(i, at[i], n) for i, n in enumerate(rows)]
        y = layer.forward(d["x"])
        for i in state["going"]:
            at[i] += rows[i]
        return {"y": y, **_caches(layer)}
    if kind == "layer":
        cache = SimpleNamespace(gdn_state={}, conv_state={})
        if c["carried"]:
            cache.gdn_state[0], cache.conv_state[0] = d["state"], d["conv"]
        y = state["model"]._gdn(d["x"], 0, cache)
        return {"y": y, "conv": cache.conv_state[0], "state": cache.gdn_state[0]}
    if kind == "attnres":
        return {"mix": _package(".attnres").full_attnres_route(d["sources"], d["query"], 1e-5)}
    return {"y": gdn.ops.accent_shift(d["x"], d["down"], d["up"], d["mask"], y=d["y"], out=d["y"])}


# --------------------------------------------------------------------------------------- work, tolerance


def _size(d):
    if isinstance(d, torch.Tensor):
        return d.numel() * d.element_size()
    return sum(_size(x) for x in (d.values() if isinstance(d, dict) else d))


def _delta_flops(tokens, heads, D):
    """The chunked form's matrix products, per token and value head (64-token chunks)."""
    return tokens * heads * (2 * CHUNK * 5 * D + 6 * D * D + CHUNK**2 / 3)


def work(case):
    c, kind = case, case["kind"]
    e = 2 if c.get("dtype", "bf16") == "bf16" else 4
    D = c.get("D", HEAD_DIM)
    if kind in ("decode", "block"):
        B, hk, hv = c["B"], c["Hk"], c["Hv"]
        state = 2 * B * hv * D * D * 4
        if kind == "decode":
            return {"bytes": state + B * (2 * hk + 2 * hv) * D * e + 2 * B * hv * 4, "flops": 8.0 * B * hv * D * D}
        C = 2 * hk * D + hv * D
        return {"bytes": state + 2 * B * C * 3 * e + B * C * e + 2 * B * hv * D * e + 2 * B * hv * e + C * 4 * e,
                "flops": 8.0 * B * hv * D * D}
    if kind in ("prefill", "packed"):
        tokens = c["B"] * c["T"] if kind == "prefill" else sum(_lengths(c))
        hk, hv = c["Hk"], c["Hv"]
        states = (c["B"] if kind == "prefill" else 2 * c["n"]) * hv * D * D * 4
        gates = 2 * tokens * hv * (e if c.get("raw") else 4)
        return {"bytes": tokens * (2 * hk + 2 * hv) * D * e + gates + states, "flops": _delta_flops(tokens, hv, D)}
    if kind == "attnres":
        return {"bytes": (c["S"] + 1) * c["T"] * c["dim"] * e, "flops": 8.0 * c["S"] * c["T"] * c["dim"]}
    if kind == "accent":
        rows, n_in, n_out, K = c["rows"], c["n_in"], c["n_out"], c["K"]
        return {"bytes": 2 * (rows * n_in + 2 * rows * n_out + rows * K + K * (n_in + n_out)),
                "flops": 2.0 * rows * K * (n_in + n_out)}
    # the mixer with its projections
    rows = c["bs"] if kind == "serving_decode" else sum(_ints(c["rows"])) if kind == "serving_extend" else c["T"]
    n = c["bs"] if kind == "serving_decode" else len(_ints(c["rows"])) if kind == "serving_extend" else 1
    width = 4 * INNER + 2 * HEADS
    weights = 2 * (width * HIDDEN + INNER * HIDDEN + 3 * INNER * 4 + HEAD_DIM)
    states = n * (HEADS * D * D * 4 + 3 * INNER * 3 * 2)
    reads = 0 if kind == "layer" and not c["carried"] else states
    gemms = 2.0 * rows * (width + INNER) * HIDDEN
    core = 8.0 * rows * HEADS * D * D if kind == "serving_decode" else _delta_flops(rows, HEADS, D)
    return {"bytes": weights + 2 * rows * HIDDEN * 2 + states + reads, "flops": gemms + core}


def tolerance(case):
    """About four times the distance from float64 that the path shows, or the data type's own where that is less."""
    c, kind = case, case["kind"]
    if c.get("dtype") == "f32":  # fp32 throughout (about 1e-6 from float64)
        return {"rel": 1e-5, "max": 1e-3}
    if kind == "decode":  # fp32 arithmetic on bf16 rows, the output rounded once (1.7e-3)
        return {"rel": 7e-3, "max": 4e-2}
    if kind in ("prefill", "packed", "accent"):  # bf16 operands of the matrix products (2.2e-3 to 2.9e-3)
        return {"rel": 1e-2, "max": 0.15}
    return {"rel": 1.5e-2, "max": 0.2}  # several roundings to bf16 in a row (4.4e-3 to 7.2e-3)


# ------------------------------------------------------------------------------------------------- exact


def _delta(q, k, v, g, beta, scale, S, mark=None):
    """The token loop in float64 over N sequences: q, k, v [N, T, H, D], g, beta [N, T, H], S [N, H, V, K].
    Returns (o, S, S after ``mark`` tokens of each sequence)."""
    o = torch.empty_like(v)
    S = S.clone()
    at = torch.zeros_like(S)
    marks = set() if mark is None else set(mark)
    for t in range(q.shape[1]):
        S = S * g[:, t].exp()[:, :, None, None]
        kt = k[:, t, :, None, :]
        u = beta[:, t, :, None] * (v[:, t] - (S * kt).sum(-1))
        S = S + u[..., None] * kt
        o[:, t] = scale * (S * q[:, t, :, None, :]).sum(-1)
        if t + 1 in marks:
            for i, m in enumerate(mark):
                if m == t + 1:
                    at[i] = S[i]
    return o, S, at


def _heads(x, hv):
    return x.double().repeat_interleave(hv // x.shape[-2], dim=-2)


def _gates(d):
    if "A_log" not in d:
        return d["g"].double(), d["beta"].double()
    g = -d["A_log"].double().exp() * F.softplus(d["g"].double() + d["dt_bias"].double())
    return g, d["beta"].double().sigmoid()


def _mixer(x, w, hist, S, mark=None):
    """The mixer layer in float64 on N sequences of T rows: x [N, T, hidden], hist [N, C, 3] raw rows before
    the first. Returns (y, raw q|k|v rows with the history before them, S, S after ``mark`` rows)."""
    w = {n: t.double() for n, t in w.items()}
    N, T = x.shape[:2]
    mixed = x.double() @ w["in_proj"].T
    qkv, z, a, b = mixed.split((3 * INNER, INNER, HEADS, HEADS), -1)
    raw = torch.cat((hist.double().transpose(1, 2), qkv), 1)
    taps = w["conv"].reshape(3 * INNER, 4)
    conv = F.silu(sum(raw[:, i:i + T] * taps[:, i] for i in range(4)))
    q, k, v = (t.reshape(N, T, HEADS, HEAD_DIM) for t in conv.split(INNER, -1))
    g = -w["A_log"].exp() * F.softplus(a + w["dt_bias"])
    o, S, at = _delta(_unit(q), _unit(k), v, g, b.sigmoid(), HEAD_DIM**-0.5, S, mark)
    o = o * torch.rsqrt(o.square().mean(-1, keepdim=True) + 1e-5) * w["out_weight"]
    o = o * F.silu(z.reshape(N, T, HEADS, HEAD_DIM))
    return o.reshape(N, T, INNER) @ w["wo"].T, raw, S, at


def _zeros(*shape):
    return torch.zeros(*shape, dtype=torch.float64, device="cuda")


def _last_raw(raw, T, n=4):
    """The last ``n`` of the first T raw rows (``raw`` has 3 rows of history in front), zeros before the first."""
    rows = raw[3:3 + T]
    return torch.cat((rows.new_zeros(n, rows.shape[1]), rows))[-n:].T


def exact(case, seed):
    c, d = case, _inputs(case, seed)
    kind = c["kind"]
    D = c.get("D", HEAD_DIM)
    if kind in ("decode", "prefill", "packed"):
        hv = c["Hv"]
        q, k, v = _heads(d["q"], hv), _heads(d["k"], hv), d["v"].double()
        g, beta = _gates(d)
        if c.get("raw"):
            q, k = _unit(q), _unit(k)
        if kind == "packed":  # a sequence a row, padded with tokens that change nothing
            lengths = _lengths(c)

            def rows(x):
                return torch.nn.utils.rnn.pad_sequence(x[0].split(lengths), batch_first=True)

            o, S, _ = _delta(rows(q), rows(k), rows(v), rows(g), rows(beta), D**-0.5, d["s0"].double())
            return {"o": torch.cat([o[i, :n] for i, n in enumerate(lengths)])[None], "state": S}
        S = d["s0"].double() if "s0" in d else _zeros(c["B"], hv, D, D)
        o, S, _ = _delta(q, k, v, g, beta, D**-0.5, S)
        return {"o": o[:, 0] if kind == "decode" else o, "state": S}
    if kind == "block":
        hk, hv = c["Hk"], c["Hv"]
        raw = torch.cat((d["cache"], d["x"][..., None]), -1).double()
        q, k, v = (t.reshape(c["B"], 1, -1, D) for t in F.silu((raw * d["w"].double()).sum(-1)).split((hk * D, hk * D, hv * D), -1))
        g, beta = _gates({"A_log": d["A_log"], "dt_bias": d["dt_bias"], "g": d["a"][:, None], "beta": d["b"][:, None]})
        o, S, _ = _delta(_heads(_unit(q), hv), _heads(_unit(k), hv), v, g, beta, D**-0.5, d["state"].double())
        o = o[:, 0] * torch.rsqrt(o[:, 0].square().mean(-1, keepdim=True) + 1e-6) * d["nw"].double()
        return {"out": o * F.silu(d["z"].double()), "cache": raw[..., 1:], "state": S}
    if kind == "serving_decode":
        bs, P = c["bs"], c["prompt"]
        x = torch.cat((d["prompts"], d["x"][:, None]), 1)
        done = (P + 1) // CHUNK * CHUNK
        y, raw, S, at = _mixer(x, d["w"], _zeros(bs, 3 * INNER, 3), _zeros(bs, HEADS, D, D), [done] * bs)
        return {"y": y[:, -1], "commit_state": at, "commit_conv": torch.stack([_last_raw(t, done) for t in raw]),
                "live_state": S, "live_conv": torch.stack([_last_raw(t, P + 1) for t in raw]), "win_len": None}
    if kind == "serving_extend":
        rows, cached = _ints(c["rows"]), _ints(c["cached"])
        got = {n: [] for n in ("y", "commit_state", "commit_conv", "live_state", "live_conv")}
        for x, before in zip(d["x"].split(rows), d["before"]):
            T = len(before) + len(x)
            done = T // CHUNK * CHUNK
            y, raw, S, at = _mixer(torch.cat((before, x))[None], d["w"], _zeros(1, 3 * INNER, 3), _zeros(1, HEADS, D, D), [done])
            for n, t in zip(got, (y[0, len(before):], at[0], _last_raw(raw[0], done), S[0], _last_raw(raw[0], T))):
                got[n].append(t)
        return {n: torch.cat(t) if n == "y" else torch.stack(t) for n, t in got.items()} | {"win_len": None}
    if kind == "layer":
        hist = d["conv"][None] if c["carried"] else _zeros(1, 3 * INNER, 3)
        S = d["state"][None].double() if c["carried"] else _zeros(1, HEADS, D, D)
        y, raw, S, _ = _mixer(d["x"][None], d["w"], hist, S)
        return {"y": y[0], "conv": raw[0, -3:].T, "state": S[0]}
    if kind == "attnres":
        bank = torch.stack(d["sources"]).double()
        keys = bank * torch.rsqrt(bank.square().mean(-1, keepdim=True) + 1e-5)
        return {"mix": (bank * (keys @ d["query"].double()).softmax(0)[..., None]).sum(0)}
    shift = ((d["x"].double() @ d["down"].double().T) * d["mask"].double()) @ d["up"].double()
    return {"y": d["y"].double() + shift}
