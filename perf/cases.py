"""
The work a user of this library has it do, as cases that can be timed: the MoE layers of a model
(one-token decode, batched decode, prefill chunks, the experts module of a patched transformers
model), the int8 dense layers around them, the store build that quantises experts, and decode
with the experts offloaded to host memory.

Each case goes through the library's public entry points as a program calls them: MoEDecoder and
GroupedLayer captured in one HIP graph per step (every call of theirs is capturable), GroupedTokens
and GroupedLayer called eagerly on prefill chunks, HipMoE.run_layer as a model's experts module
calls it, QLinear, encode_record_, OffloadDecoder. The model shapes are the library's own benchmark
configurations: OLMoE, Qwen3-30B-A3B and Qwen3-Next-80B-A3B.

The experts are N(0, 0.02) weights quantised here in plain torch in the store's packing, so
`exact` can rebuild them in 64 bits from the seed; hidden states are N(0, 1) (a normalised residual
stream), routers N(0, 0.02).
"""

from __future__ import annotations

import math
import sys
from functools import lru_cache
from pathlib import Path

import torch

ROOT = Path(__file__).resolve().parents[1]
PKG = ROOT / "moe-offload-lab_amd"
if str(PKG) not in sys.path:
    sys.path.insert(0, str(PKG))

DEV = "cuda:0"
DT = {"fp16": torch.float16, "bf16": torch.bfloat16}

# d_model, d_ff, experts, top-k, renormalised top-k, shared expert
SHAPES = {
    "olmoe": dict(H=2048, I=1024, E=64, k=8, renorm=False, shared=False),
    "qwen3-30b": dict(H=2048, I=768, E=128, k=8, renorm=True, shared=False),
    "qwen3-next": dict(H=2048, I=512, E=512, k=10, renorm=True, shared=True),
}
# records per expert, most precise first; "mixed" is the two-precision store (fp16 from a routed
# weight of T1 on, else int4)
PRECS = {"int4": ["int4"], "int8": ["int8"], "fp8": ["fp8"], "fp16": ["fp16"], "mixed": ["fp16", "int4"]}
T1 = 0.15
HI_VOTE = 0.5   # a batch's expert runs at the level that at least this share of its tokens asks for
STD = 0.02
CHUNK = 64      # experts generated at a time
MAX_TOKENS = 512  # tokens per call of the experts module (HipMoE's own default)


def listed() -> list[dict]:
    return [
        # the headline: one decode token through the 16 MoE layers of OLMoE, int4, one HIP graph
        dict(name="decode-olmoe-int4", kind="decode", shape="olmoe", prec="int4", layers=16, tokens=1, dtype="fp16"),
        # one decode token of an FP8 checkpoint's layers: 512 experts, top-10 and the shared expert
        dict(name="decode-qwen3next-fp8", kind="decode", shape="qwen3-next", prec="fp8", layers=4, tokens=1,
             dtype="bf16"),
        # a small serving batch on the two-precision store (a vote per expert)
        dict(name="batch8-olmoe-mixed", kind="batch", shape="olmoe", prec="mixed", layers=8, tokens=8, dtype="fp16"),
        # a larger serving batch, many experts with one or two tokens each, shared expert
        dict(name="batch32-qwen3next-int4", kind="batch", shape="qwen3-next", prec="int4", layers=2, tokens=32,
             dtype="bf16"),
        # the usual prefill chunk: ~32 tokens per expert
        dict(name="prefill512-qwen3-30b", kind="prefill", shape="qwen3-30b", prec="int4", layers=1, tokens=512,
             dtype="bf16"),
        # a long prompt in one chunk: 256 tokens per expert
        dict(name="prefill2048-olmoe", kind="prefill", shape="olmoe", prec="int4", layers=1, tokens=2048, dtype="fp16"),
        # a short prompt (ragged length) on an FP8 checkpoint with the shared expert: ~6 tokens per expert
        dict(name="chunk333-qwen3next-fp8", kind="chunk", shape="qwen3-next", prec="fp8", layers=1, tokens=333,
             dtype="bf16"),
        # a 1000-token prompt through a patched transformers model's experts module: two calls of
        # 512 and 488 tokens inside run_layer, two record precisions
        dict(name="experts1000-olmoe-mixed", kind="experts", shape="olmoe", prec="mixed", layers=1, tokens=1000,
             dtype="bf16"),
        # the smallest calls: the attention projections of a decode token (q, k, v, o of 16 layers),
        # int8, in the token's graph
        dict(name="dense1-projections", kind="dense", rows=2048, cols=2048, matrices=64, tokens=1, dtype="fp16"),
        # the LM head of a 32-token decode batch
        dict(name="dense32-head", kind="dense", rows=151936, cols=2048, matrices=1, tokens=32, dtype="bf16"),
        # building a store: a checkpoint's experts to int4 records with the default (mse) scale search
        dict(name="encode-olmoe-int4", kind="encode", shape="olmoe", prec="int4", experts=8),
        # decode with the experts in host memory: 39 % of the records fit the device budget, the
        # next layer's experts predicted by its gate; 6 tokens of a correlated stream per pass
        dict(name="offload-olmoe-int4", kind="offload", shape="olmoe", prec="int4", layers=4, tokens=6, dtype="bf16",
             resident=0.39),
    ]


def _log_int(rng, lo: int, hi: int) -> int:
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng) -> dict:
    kind = rng.choice(["decode", "decode", "batch", "batch", "prefill", "prefill", "chunk", "chunk", "experts",
                       "dense", "dense", "encode", "offload"])
    shape = rng.choice(list(SHAPES))
    dtype = rng.choice(["fp16", "bf16"])
    big = shape == "qwen3-next"
    if kind == "decode":
        prec = rng.choice(["int4", "int8", "fp8", "mixed"])
        return dict(kind=kind, shape=shape, prec=prec, layers=rng.randint(2, 3 if big else 8), tokens=1, dtype=dtype)
    if kind == "batch":
        prec = rng.choice(["int4", "int8", "fp8", "mixed"])
        return dict(kind=kind, shape=shape, prec=prec, layers=rng.randint(1, 2 if big else 6),
                    tokens=_log_int(rng, 2, 64), dtype=dtype)
    if kind == "prefill":
        return dict(kind=kind, shape=shape, prec="int4", layers=1, tokens=_log_int(rng, 65, 2000), dtype=dtype)
    if kind == "chunk":
        prec = rng.choice(["int4", "int8", "fp8", "fp16", "mixed"])
        return dict(kind=kind, shape=shape, prec=prec, layers=1, tokens=_log_int(rng, 65, 1100), dtype=dtype)
    if kind == "experts":
        tokens = _log_int(rng, 1, 1400)
        prec = rng.choice(["int4", "int8", "fp8", "mixed"])
        return dict(kind=kind, shape=shape, prec=prec, layers=3 if tokens < 32 else 1, tokens=tokens, dtype=dtype)
    if kind == "dense":
        tokens = _log_int(rng, 1, 500)
        if rng.random() < 0.4:
            return dict(kind=kind, rows=rng.choice([50304, 151936]), cols=2048, matrices=1, tokens=tokens, dtype=dtype)
        rows, cols = rng.choice([(2048, 2048), (4096, 2048), (2048, 4096), (512, 2048), (1024, 2048)])
        return dict(kind=kind, rows=rows, cols=cols, matrices=rng.randint(8, 48), tokens=tokens, dtype=dtype)
    if kind == "encode":
        return dict(kind=kind, shape=shape, prec=rng.choice(["int4", "int8", "fp8"]), experts=rng.randint(2, 16))
    return dict(kind=kind, shape=rng.choice(["olmoe", "qwen3-30b"]), prec="int4", layers=rng.randint(2, 4),
                tokens=rng.randint(3, 8), dtype=dtype, resident=round(rng.uniform(0.3, 0.6), 3))


# ---------------------------------------------------------------------------------------------
# inputs: from the seed alone, in plain torch
# ---------------------------------------------------------------------------------------------
def _gen(seed: int, *at: int) -> torch.Generator:
    s = seed
    for a in at:
        s = (s * 1000003 + a + 1) % (1 << 61)
    return torch.Generator(device=DEV).manual_seed(s)


def _expert_weights(sh: dict, seed: int, layer: int, e0: int, n: int):
    """gate_up (n, 2I, H) and down (n, H, I) fp32 of experts e0 .. e0 + n - 1."""
    g = _gen(seed, 7, layer, e0)
    return (torch.randn(n, 2 * sh["I"], sh["H"], device=DEV, generator=g) * STD,
            torch.randn(n, sh["H"], sh["I"], device=DEV, generator=g) * STD)


def _quantise(w: torch.Tensor, prec: str):
    """(values, scales) of w (..., O, K): int4 / int8 integers with fp16 scales per 64 columns
    (absmax), fp8 e4m3 bytes with fp32 scales per 128 x 128 block, fp16 values (no scales)."""
    if prec == "fp16":
        return w.half(), None
    *lead, O, K = w.shape
    if prec == "fp8":
        b = w.reshape(*lead, O // 128, 128, K // 128, 128)
        s = b.abs().amax(dim=(-3, -1)) / 448.0
        q = (b / s[..., :, None, :, None]).clamp_(-448.0, 448.0).to(torch.float8_e4m3fn)
        return q.reshape(*lead, O, K).view(torch.uint8), s
    qmax = 7.0 if prec == "int4" else 127.0
    b = w.reshape(*lead, O, K // 64, 64)
    s = (b.abs().amax(dim=-1) / qmax).half()
    q = (b / s.float()[..., None]).round_().clamp_(-qmax, qmax)
    return q.reshape(*lead, O, K).to(torch.int8), s


def _double(q: torch.Tensor, s, prec: str) -> torch.Tensor:
    """The float64 matrix (O, K) of one expert's (values, scales)."""
    if prec == "fp16":
        return q.double()
    if prec == "fp8":
        O, K = q.shape
        b = q.view(torch.float8_e4m3fn).float().double().reshape(O // 128, 128, K // 128, 128)
        return (b * s.double()[:, None, :, None]).reshape(O, K)
    O, K = q.shape
    return (q.double().reshape(O, K // 64, 64) * s.double()[..., None]).reshape(O, K)


def _bytes(q: torch.Tensor, prec: str) -> torch.Tensor:
    """The stored bytes of the values (int4: two per byte, low nibble first, + 8)."""
    if prec == "int4":
        u = (q + 8).to(torch.uint8)
        return u[..., 0::2] | (u[..., 1::2] << 4)
    return q


def _write(blobs: torch.Tensor, layout: dict, mats: dict) -> None:
    """Fields {name: tensor (n, ...)} into the records blobs (n, record_bytes)."""
    for name, _, _, off in layout["fields"]:
        t = mats[name].contiguous()
        raw = t.view(torch.uint8).reshape(t.shape[0], -1)
        blobs[:, off:off + raw.shape[1]].copy_(raw)


def _fields(gu: torch.Tensor, dn: torch.Tensor, prec: str) -> dict:
    out = {}
    for name, w in (("gate_up", gu), ("down", dn)):
        q, s = _quantise(w, prec)
        if s is None:
            out[name] = q
        else:
            out[f"{name}.q"], out[f"{name}.s"] = _bytes(q, prec), s
    return out


def _routers(sh: dict, seed: int, layers: int, dt):
    return [(torch.randn(sh["E"], sh["H"], device=DEV, generator=_gen(seed, 11, l)) * STD).to(dt) for l in range(layers)]


def _states(sh: dict, seed: int, layers: int, tokens: int, dt) -> torch.Tensor:
    return torch.randn(layers, tokens, sh["H"], device=DEV, generator=_gen(seed, 13)).to(dt)


def _shared_gate(sh: dict, seed: int, layer: int, dt) -> torch.Tensor:
    return (torch.randn(sh["H"], device=DEV, generator=_gen(seed, 17, layer)) * 0.05).to(dt)


def _given_routing(sh: dict, seed: int, layer: int, tokens: int, dt):
    """idx (T, k) int64 and weights (T, k) in dt as a model's router hands them on."""
    g = _gen(seed, 19, layer)
    p = torch.softmax(torch.randn(tokens, sh["E"], device=DEV, generator=g) * 0.9, dim=-1)
    w, idx = torch.topk(p, sh["k"], dim=-1)
    if sh["renorm"]:
        w = w / w.sum(-1, keepdim=True)
    return idx.contiguous(), w.to(dt).contiguous()


def _stream(sh: dict, seed: int, layers: int, tokens: int, dt):
    """A correlated decode: routers with a Zipf-like popularity of the experts, and hidden states
    that change by 0.6-correlated steps from token to token and by 0.35 from layer to layer."""
    H, E = sh["H"], sh["E"]
    g = _gen(seed, 23)
    u = torch.randn(H, device=DEV, generator=g)
    u /= u.norm()
    routers = []
    for _ in range(layers):
        rank = torch.rand(E, device=DEV, generator=g).argsort().float()
        W = torch.randn(E, H, device=DEV, generator=g) / math.sqrt(H) - torch.log(rank + 1.0)[:, None] * u[None, :]
        routers.append(W.to(dt).contiguous())
    xs = torch.empty(layers, tokens, H, dtype=dt, device=DEV)
    z = torch.randn(H, device=DEV, generator=g)
    for t in range(tokens):
        z = 0.6 * z + 0.8 * torch.randn(H, device=DEV, generator=g)
        zl = z.clone()
        for l in range(layers):
            xs[l, t] = (u + zl).to(dt)
            zl = zl + 0.35 * torch.randn(H, device=DEV, generator=g)
    return routers, xs


def _policy(prec: str):
    from moelab_hip.policy import PrecisionPolicy

    return PrecisionPolicy("weight", t1=T1, upgrade=False) if prec == "mixed" else PrecisionPolicy("lo")


def _layouts(sh: dict, prec: str) -> dict:
    from moelab_hip.store import record_layout

    return {p: record_layout(p, sh["H"], sh["I"], 64, scale="absmax" if p in ("int4", "int8") else None)
            for p in PRECS[prec]}


def _store(sh: dict, prec: str, layers: int, seed: int):
    """A ResidentStore holding every expert of every layer."""
    from moelab_hip.layer import ResidentStore

    lays = _layouts(sh, prec)
    E = sh["E"]
    st = ResidentStore(lays, layers, E, DEV)
    for l in range(layers):
        for e0 in range(0, E, CHUNK):
            n = min(CHUNK, E - e0)
            gu, dn = _expert_weights(sh, seed, l, e0, n)
            for p, lay in lays.items():
                rb = lay["record_bytes"]
                o = (l * E + e0) * rb
                _write(st.arena[p][o:o + n * rb].view(n, rb), lay, _fields(gu, dn, p))
        for pi, p in enumerate(st.precisions):
            rb = lays[p]["record_bytes"]
            st.rtab[l, pi] = st.arena[p].data_ptr() + (l * E + torch.arange(E, device=DEV)) * rb
    st.present[:] = True
    return st


def _shared(sh: dict, st, seed: int, dt):
    if not sh["shared"]:
        return None
    out = []
    for l in range(st.L):
        gu, dn = _expert_weights(sh, seed, l, sh["E"], 1)
        rec = {}
        for p, lay in st.layouts.items():
            blob = torch.zeros(1, lay["record_bytes"], dtype=torch.uint8, device=DEV)
            _write(blob, lay, _fields(gu, dn, p))
            rec[p] = blob[0]
        out.append({"gate": _shared_gate(sh, seed, l, dt), "rec": rec})
    return out


def _captured(step):
    """`step` as one HIP graph (run once before, as a program warms up)."""
    step()
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        out = step()
    return g, out


def prepare(case: dict, seed: int) -> dict:
    from moelab_hip import _lib

    _lib.check_device(DEV)  # a program's set-up call (probes the device once)
    kind = case["kind"]
    if kind == "dense":
        return _prepare_dense(case, seed)
    if kind == "encode":
        return _prepare_encode(case, seed)
    if kind == "offload":
        return _prepare_offload(case, seed)
    sh, dt, T, L = SHAPES[case["shape"]], DT[case["dtype"]], case["tokens"], case["layers"]
    st = _store(sh, case["prec"], L, seed)
    xs = _states(sh, seed, L, T, dt)
    outs = torch.empty_like(xs)
    s = dict(kind=kind, store=st, xs=xs, outs=outs, layers=L)
    if kind == "experts":
        from moelab_hip.adapters import HipMoE

        s["moe"] = HipMoE(st, sh["k"], _policy(case["prec"]), dt, max_tokens=MAX_TOKENS)
        s["routing"] = [_given_routing(sh, seed, l, T, dt) for l in range(L)]
        s["act"] = torch.nn.functional.silu
        return s
    s["routers"] = _routers(sh, seed, L, dt)
    if kind == "prefill":
        from moelab_hip.prefill import GroupedTokens

        s["tokens"] = GroupedTokens(st.layouts["int4"], sh["E"], sh["k"], T, DEV)
        s["tabs"] = [s["tokens"].table(st.rtab[l, 0]).contiguous() for l in range(L)]
        s["renorm"] = sh["renorm"]
        return s
    shared = _shared(sh, st, seed, dt)
    pol = _policy(case["prec"])
    if kind == "decode":
        from moelab_hip.layer import MoEDecoder

        dec = MoEDecoder(st, sh["k"], pol, dt, router_weights=s["routers"], renorm=sh["renorm"], shared=shared)
    else:
        from moelab_hip.prefill import GroupedLayer

        dec = GroupedLayer(st, sh["k"], T, pol, dt, router_weights=s["routers"], renorm=sh["renorm"], shared=shared)
    s["dec"], s["shared"] = dec, shared
    if kind != "chunk":  # a decode step is one HIP graph
        def step():
            for l in range(L):
                dec.layer(l, xs[l], outs[l])

        s["graph"], _ = _captured(step)
    return s


def _prepare_dense(case: dict, seed: int) -> dict:
    from moelab_hip.denseq import QLinear

    O, K, T, dt = case["rows"], case["cols"], case["tokens"], DT[case["dtype"]]
    mods, xs = [], []
    for i in range(case["matrices"]):
        q, sc = _dense_weights(case, seed, i)
        mods.append(QLinear(q, sc, 64, None, dt))
        xs.append(torch.randn(T, K, device=DEV, generator=_gen(seed, 31, i)).to(dt))
    s = dict(kind="dense", mods=mods, xs=xs)
    if T == 1:  # part of the decode token's graph
        s["graph"], s["outs"] = _captured(lambda: [m(x) for m, x in zip(mods, xs)])
    return s


def _dense_weights(case: dict, seed: int, i: int):
    w = torch.randn(case["rows"], case["cols"], device=DEV, generator=_gen(seed, 29, i)) * STD
    return _quantise(w, "int8")


def _prepare_encode(case: dict, seed: int) -> dict:
    from moelab_hip.store import record_layout

    sh = SHAPES[case["shape"]]
    lay = record_layout(case["prec"], sh["H"], sh["I"], 64)  # the store's own choice of scale method
    ws = []
    for e in range(case["experts"]):
        gu, dn = _expert_weights(sh, seed, 0, e, 1)
        ws.append((gu[0].bfloat16(), dn[0].bfloat16()))  # as a checkpoint holds them
    blobs = torch.empty(case["experts"], lay["record_bytes"], dtype=torch.uint8, device=DEV)
    return dict(kind="encode", layout=lay, ws=ws, blobs=blobs)


def _prepare_offload(case: dict, seed: int) -> dict:
    from moelab_hip.offload import OffloadDecoder
    from moelab_hip.policy import PrecisionPolicy

    sh, dt, L, T = SHAPES[case["shape"]], DT[case["dtype"]], case["layers"], case["tokens"]
    st = _store(sh, "int4", L, seed)
    lay = st.layouts["int4"]
    rb, E = lay["record_bytes"], sh["E"]
    host = torch.empty(L * E * rb, dtype=torch.uint8, pin_memory=True)
    host.copy_(st.arena["int4"])
    routers, xs = _stream(sh, seed, L, T, dt)
    off = OffloadDecoder({"int4": lay}, L, E, sh["k"], lambda l, e, p: host[(l * E + e) * rb:(l * E + e + 1) * rb],
                         int(L * E * rb * case["resident"]), DEV, PrecisionPolicy("lo"), dt, router_weights=routers,
                         renorm=sh["renorm"], predictor="gate")
    return dict(kind="offload", off=off, host=host, xs=xs, outs=torch.empty_like(xs), layers=L, count=T)


# ---------------------------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------------------------
def run(s: dict):
    kind = s["kind"]
    if "graph" in s:
        s["graph"].replay()
        return s["outs"]
    if kind == "prefill":
        for l in range(s["layers"]):
            s["tokens"].layer(s["xs"][l], s["routers"][l], s["renorm"], s["tabs"][l], s["outs"][l])
        return s["outs"]
    if kind == "chunk":
        for l in range(s["layers"]):
            s["dec"].layer(l, s["xs"][l], s["outs"][l])
        return s["outs"]
    if kind == "experts":
        return [s["moe"].run_layer(l, s["xs"][l], *s["routing"][l], s["act"]) for l in range(s["layers"])]
    if kind == "dense":
        return [m(x) for m, x in zip(s["mods"], s["xs"])]
    if kind == "encode":
        from moelab_hip.store import encode_record_

        for blob, (gu, dn) in zip(s["blobs"], s["ws"]):
            encode_record_(s["layout"], blob, gu, dn)
        return s["blobs"]
    off, xs, outs = s["off"], s["xs"], s["outs"]
    for t in range(s["count"]):
        for l in range(s["layers"]):
            off.layer(l, xs[l, t:t + 1], outs[l, t:t + 1])
        off.tick()
    return outs


# ---------------------------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------------------------
def _record_bytes(sh: dict, p: str) -> float:
    v = 3 * sh["H"] * sh["I"]
    return {"int4": v / 2 + v / 64 * 2, "int8": v + v / 64 * 2, "fp8": v + v / 128 / 128 * 4, "fp16": v * 2.0}[p]


@lru_cache(maxsize=None)
def _records_run(shape: str, prec: str, tokens: int) -> float:
    """Bytes of the distinct (expert, precision) records that T tokens of one layer run, expected
    over random routing (logits N(0, 0.9)); counted on a few drawn batches."""
    sh, g, total, n = SHAPES[shape], torch.Generator().manual_seed(5), 0.0, 8
    for _ in range(n):
        p = torch.softmax(torch.randn(tokens, sh["E"], generator=g) * 0.9, dim=-1)
        w, idx = torch.topk(p, sh["k"], dim=-1)
        if sh["renorm"]:
            w = w / w.sum(-1, keepdim=True)
        cnt = torch.bincount(idx.reshape(-1), minlength=sh["E"])
        if prec == "mixed":
            hi = torch.bincount(idx[w >= T1], minlength=sh["E"])
            at0 = (cnt > 0) & (hi >= HI_VOTE * cnt)
            total += int(at0.sum()) * _record_bytes(sh, "fp16") + int(((cnt > 0) & ~at0).sum()) * _record_bytes(sh, "int4")
        else:
            total += int((cnt > 0).sum()) * _record_bytes(sh, prec)
    return total / n


def work(case: dict) -> dict:
    kind = case["kind"]
    if kind == "dense":
        O, K, T, n = case["rows"], case["cols"], case["tokens"], case["matrices"]
        return {"bytes": n * (O * K + O * K / 64 * 2 + 2 * T * (O + K)), "flops": n * 2.0 * O * K * T}
    sh = SHAPES[case["shape"]]
    H, I, E, k = sh["H"], sh["I"], sh["E"], sh["k"]
    if kind == "encode":  # bf16 weights in, records out
        return {"bytes": case["experts"] * (3 * H * I * 2 + _record_bytes(sh, case["prec"])), "flops": 0.0}
    T, L = case["tokens"], case["layers"]
    if kind == "offload":  # a token's records are read from device memory by its layer, wherever they were before
        recs = T * k * _record_bytes(sh, "int4")
        return {"bytes": L * (recs + T * (E * H * 2 + 4 * H)), "flops": L * T * (k * 6.0 * H * I + 2.0 * E * H)}
    shared = 1 if sh["shared"] and kind != "experts" else 0
    recs = _records_run(case["shape"], case["prec"], T) + shared * _record_bytes(sh, PRECS[case["prec"]][0])
    router = 0 if kind == "experts" else E * H * 2
    return {"bytes": L * (recs + router + T * 4 * H), "flops": L * T * ((k + shared) * 6.0 * H * I + (2.0 * E * H if router else 0.0))}


def tolerance(case: dict):
    """2-norm of the difference over 2-norm of the result; about four times what two correct
    orders of summation and roundings show at the output's precision (fp16 2^-11, bf16 2^-8)."""
    if case["kind"] == "encode":
        return "exact"
    return {"rel": 2e-3 if case["dtype"] == "fp16" else 1e-2}


# ---------------------------------------------------------------------------------------------
# the same in 64 bits, in plain torch
# ---------------------------------------------------------------------------------------------
def _route64(x, Wr, sh, dt):
    """The router as the model defines it (logits in the activation dtype, softmax, top-k with the
    lower index first among equals, weights in the activation dtype), on 64-bit products."""
    logits = (x.double() @ Wr.double().t()).to(dt)
    order = torch.sort(logits, dim=-1, descending=True, stable=True)[1][:, :sh["k"]]
    w = torch.softmax(logits.double(), dim=-1).gather(1, order)
    if sh["renorm"]:
        w = w / w.sum(-1, keepdim=True)
    return order, w.to(dt)


def _expert64(x, gu, dn):
    g, u = (x @ gu.t()).chunk(2, dim=-1)
    return (torch.nn.functional.silu(g) * u) @ dn.t()


def _layer64(sh: dict, prec: str, seed: int, layer: int, x, idx, w, gate) -> torch.Tensor:
    """Sum over each token's routed experts (and the shared one) of weight * expert(x), float64."""
    x64, out = x.double(), torch.zeros(x.shape, dtype=torch.float64, device=DEV)
    T = x.shape[0]
    used = set(idx.reshape(-1).tolist())
    precs = PRECS[prec]
    for e0 in range(0, sh["E"], CHUNK):
        n = min(CHUNK, sh["E"] - e0)
        if not any(e0 <= e < e0 + n for e in used):
            continue
        gu, dn = _expert_weights(sh, seed, layer, e0, n)
        for e in range(e0, e0 + n):
            if e not in used:
                continue
            tok, slot = (idx == e).nonzero(as_tuple=True)
            we = w[tok, slot]
            p = precs[0]
            if prec == "mixed":  # one token: its own weight; several: the vote
                hi = int((we.float() >= T1).sum())
                p = precs[0] if hi >= (HI_VOTE - 1e-9) * tok.numel() else precs[1]
            q = [_double(*_quantise(m[e - e0], p), p) for m in (gu, dn)]
            out.index_add_(0, tok, _expert64(x64[tok], *q) * we.double()[:, None])
    if gate is not None:
        gu, dn = _expert_weights(sh, seed, layer, sh["E"], 1)
        q = [_double(*_quantise(m[0], precs[0]), precs[0]) for m in (gu, dn)]
        logit = (x64 @ gate.double()).to(x.dtype).double()
        out += torch.sigmoid(logit).to(x.dtype).double()[:, None] * _expert64(x64, *q)
    return out


def exact(case: dict, seed: int):
    kind = case["kind"]
    if kind == "encode":
        return None
    dt, T = DT[case["dtype"]], case["tokens"]
    if kind == "dense":
        outs = []
        for i in range(case["matrices"]):
            x = torch.randn(T, case["cols"], device=DEV, generator=_gen(seed, 31, i)).to(dt).double()
            q, s = _dense_weights(case, seed, i)
            outs.append(torch.cat([x @ _double(q[r:r + 16384], s[r:r + 16384], "int8").t()
                                   for r in range(0, case["rows"], 16384)], dim=1))
        return outs
    sh, L = SHAPES[case["shape"]], case["layers"]
    if kind == "offload":
        routers, xs = _stream(sh, seed, L, T, dt)
    else:
        xs = _states(sh, seed, L, T, dt)
        routers = None if kind == "experts" else _routers(sh, seed, L, dt)
    outs = []
    for l in range(L):
        shared = sh["shared"] and kind in ("decode", "batch", "chunk")
        gate = _shared_gate(sh, seed, l, dt) if shared else None
        if kind == "experts":
            idx, w = _given_routing(sh, seed, l, T, dt)
            outs.append(torch.cat([_layer64(sh, case["prec"], seed, l, xs[l, t:t + MAX_TOKENS], idx[t:t + MAX_TOKENS],
                                            w[t:t + MAX_TOKENS], None) for t in range(0, T, MAX_TOKENS)]))
        else:
            idx, w = _route64(xs[l], routers[l], sh, dt)
            outs.append(_layer64(sh, case["prec"], seed, l, xs[l], idx, w, gate))
    return outs if kind == "experts" else torch.stack(outs)
