"""What a user of this framework has it do, as cases that can be timed and checked.

The framework runs the FFN half of a quantised mixture-of-experts model: a decode step (one token through a stack of
layers, replayed from a HIP graph as an engine does), the speculative-verify step, prompt chunks, the leading dense
FFN blocks, the output head, and the separate calls that an engine written against the kernel-launch API makes. Each
kind goes through the public entry points of flintnsteel_amd.ops (or the C ABI itself for the separate calls), with
weights, workspaces and outputs allocated once, as an engine holds them.

A case is a dict:
  kind     "layer" (MoeLayer: decode at tokens = 1, verify at 2..4), "calls" (the seven separate decode calls),
           "prefill" (MoePrefill), "dense" (DenseFfn, decode form), "dense_prefill" (DenseFfn, prefill form),
           "head" (Q8_1 of the hidden rows, then one wide mmvq)
  tokens   tokens of one call
  layers   resident layers one pass goes through; over 1 they are captured in one HIP graph and the pass replays it
  hidden, inter, experts, k, gu, down   shapes and ggml block types (gate and up share one)
  block    True: the whole block (RMSNorm, bf16 router, sigmoid gating, F16 guard, residual, a shared expert of
           width 2 * inter); False: fp32 router, softmax gating
  skew     (prefill) True: a Dirichlet(0.3) router bias, so that the experts' loads differ as in real prompts
"""
from __future__ import annotations

import ctypes
import math

import numpy as np
import torch

from flintnsteel_amd import ops, synth
from flintnsteel_amd._lib import call

Q8_0, Q3_K, Q4_K, Q5_K, Q6_K = 8, 11, 12, 13, 14
IQ3_XXS, IQ3_S, IQ4_XS = 18, 21, 23
BLOCK = {Q8_0: 272, Q3_K: 110, Q4_K: 144, Q5_K: 176, Q6_K: 210, IQ3_XXS: 98, IQ3_S: 110, IQ4_XS: 136}  # per 256 values
EPS = 1e-6
VOCAB = 150144


def listed() -> list[dict]:
    moe = {"hidden": 2048, "inter": 768, "experts": 128, "k": 8, "block": False}
    flint = {"hidden": 2048, "inter": 512, "experts": 256, "k": 6, "block": True}
    return [
        # one layer called by itself without a graph, mixed 3-bit weights: an engine's debug or first step
        {"name": "decode-call-q3k-q5k", "kind": "layer", "tokens": 1, "layers": 1, "gu": Q3_K, "down": Q5_K, **moe},
        # the headline: a token through a stack of Q4_K layers, one graph replay per token
        {"name": "decode-q4k-x16", "kind": "layer", "tokens": 1, "layers": 16, "gu": Q4_K, "down": Q4_K, **moe},
        # the same for the reference model's whole block in the formats its checkpoints ship
        {"name": "decode-block-iq3xxs-iq4xs-x16", "kind": "layer", "tokens": 1, "layers": 16, "gu": IQ3_XXS,
         "down": IQ4_XS, **flint},
        # speculative decoding: 1 accepted and 3 drafted tokens verified per step
        {"name": "verify4-q4k-x8", "kind": "layer", "tokens": 4, "layers": 8, "gu": Q4_K, "down": Q4_K, **moe},
        # the same token through an engine that makes the kernel-launch API's seven calls per layer
        {"name": "decode-calls-q4k-x16", "kind": "calls", "tokens": 1, "layers": 16, "gu": Q4_K, "down": Q4_K, **moe},
        # the end of a prompt, or a short one: a ragged chunk whose experts get a token or two each
        {"name": "prefill-37-block-q4k-q5k", "kind": "prefill", "tokens": 37, "layers": 1, "gu": Q4_K, "down": Q5_K,
         "skew": False, **flint},
        # a prompt chunk with uneven expert loads
        {"name": "prefill-512-q4k", "kind": "prefill", "tokens": 512, "layers": 1, "gu": Q4_K, "down": Q4_K,
         "skew": True, **moe},
        # a prompt chunk of odd length through the reference model's whole block
        {"name": "prefill-1021-block-q4k-q5k", "kind": "prefill", "tokens": 1021, "layers": 1, "gu": Q4_K,
         "down": Q5_K, "skew": False, **flint},
        # a long prompt at once
        {"name": "prefill-4096-q4k-q6k", "kind": "prefill", "tokens": 4096, "layers": 1, "gu": Q4_K, "down": Q6_K,
         "skew": True, **moe},
        # the leading dense FFN blocks: a token ...
        {"name": "dense-decode-q8_0-x8", "kind": "dense", "tokens": 1, "layers": 8, "gu": Q8_0, "down": Q8_0,
         "hidden": 2048, "inter": 6144},
        # ... and a prompt chunk
        {"name": "dense-prefill-512-q8_0", "kind": "dense_prefill", "tokens": 512, "layers": 1, "gu": Q8_0,
         "down": Q8_0, "hidden": 2048, "inter": 6144},
        # the output head's logits for one token
        {"name": "head-q8_0", "kind": "head", "tokens": 1, "layers": 1, "gu": Q8_0, "hidden": 2048, "inter": VOCAB},
    ]


def _log_int(rng, lo: int, hi: int) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw(rng) -> dict:
    kind = rng.choice(["layer", "layer", "calls", "prefill", "prefill", "prefill", "dense", "dense_prefill", "head"])
    if kind == "head":
        return {"kind": kind, "tokens": rng.choice([1, 1, 2, 3, 4]), "layers": 1,
                "gu": rng.choice([Q8_0, Q8_0, Q6_K]), "hidden": 256 * rng.randint(4, 12),
                "inter": _log_int(rng, 20000, VOCAB)}
    if kind in ("dense", "dense_prefill"):
        t = rng.choice([Q8_0, Q8_0, Q4_K, Q6_K])
        pre = kind == "dense_prefill"
        return {"kind": kind, "tokens": _log_int(rng, 5, 2048) if pre else rng.choice([1, 1, 2, 4]),
                "layers": 1 if pre else rng.randint(4, 8), "gu": t, "down": t, "hidden": 256 * rng.randint(4, 12),
                "inter": 256 * rng.randint(8, 32)}
    block = rng.random() < 0.5 and kind != "calls"
    gu, down = rng.choice([(Q4_K, Q4_K), (Q3_K, Q5_K), (Q4_K, Q6_K), (Q4_K, Q5_K), (Q5_K, Q6_K), (IQ3_XXS, IQ4_XS),
                           (IQ3_S, IQ4_XS)])
    c = {"kind": kind, "gu": gu, "down": down, "block": block, "hidden": 256 * rng.randint(4, 16),
         "inter": 256 * rng.randint(1, 6), "experts": rng.choice([16, 32, 60, 64, 128, 160, 256]),
         "k": rng.randint(2, 8)}
    if kind == "prefill":
        return {**c, "tokens": _log_int(rng, 5, 4096), "layers": 1, "skew": rng.random() < 0.5}
    if kind == "layer":
        c = {**c, "tokens": rng.choice([1, 1, 1, 2, 3, 4]), "layers": rng.choice([1, 4, 6, 8])}
        pad = (c["inter"] + 511) // 512 * 512  # MoeLayer takes 64 KiB of 8-bit act rows (over 1.5 bytes a column)
        return c if c["tokens"] * c["k"] * pad * 1.625 <= 65536 else _draw(rng)
    return {**c, "tokens": 1, "layers": rng.choice([4, 8]), "inter": min(c["inter"], 1024)}


def draw(rng) -> dict:
    """A case of the same kinds and ranges that costs no more (weights to make, bytes, products) than the listed ones."""
    works = [work(c) for c in listed()]
    top = {key: max(w[key] for w in works) for key in ("bytes", "flops")}
    while True:
        c = _draw(rng)
        w = work(c)
        if w["bytes"] <= top["bytes"] and w["flops"] <= top["flops"] and _weight_bytes(c) * c["layers"] <= 6e9:
            return c


# ---- what a pass cannot do without ----------------------------------------------------------------------------------

def _mat(qtype: int, n: int, m: int) -> int:
    return n * m // 256 * BLOCK[qtype]


def _expert_bytes(c: dict) -> int:
    return 2 * _mat(c["gu"], c["inter"], c["hidden"]) + _mat(c["down"], c["hidden"], c["inter"])


def _weight_bytes(c: dict) -> int:
    if c["kind"] == "head":
        return _mat(c["gu"], c["inter"], c["hidden"])
    return _expert_bytes(c) * c.get("experts", 1)


def work(case: dict) -> dict:
    c = case
    T, H, F, L = c["tokens"], c["hidden"], c["inter"], c["layers"]
    if c["kind"] == "head":
        return {"bytes": _weight_bytes(c) + 4 * T * (H + F), "flops": 2 * T * H * F}
    io = 4 * T * H * 2
    if c["kind"] in ("dense", "dense_prefill"):
        return {"bytes": L * (_expert_bytes(c) + 4 * H + io), "flops": L * 6 * T * H * F}
    E, k = c["experts"], c["k"]
    distinct = E * (1 - (1 - k / E) ** T)  # expected number of experts that T tokens select
    if c.get("skew"):  # the router bias makes an expert's share follow the square root of its load
        share = np.sqrt(np.random.default_rng(0).dirichlet(np.full(E, 0.3)))
        distinct = float(np.sum(1 - (1 - np.minimum(1, k * share / share.sum())) ** T))
    byts = distinct * _expert_bytes(c) + E * H * (2 if c["block"] else 4) + io
    flops = 2 * T * (E * H + k * 3 * H * F)
    if c["block"]:
        sh = 2 * F
        byts += 2 * _mat(c["gu"], sh, H) + _mat(c["down"], H, sh) + 4 * H
        flops += 6 * T * H * sh
    return {"bytes": L * byts, "flops": L * flops}


def tolerance(case: dict) -> dict:
    """Products of quantised blocks are exact and their sums 32-bit, so the head's logits agree to about 1e-7. In a layer,
    activations are quantised to 8 bits (the layer's input after RMSNorm, act before down), and a 32-bit sum that
    differs in its last bits moves a code that lies on a rounding boundary by one step of 127: against 64 bits, most
    outputs are within 2e-4, and one token whose largest codes moved, or whose router rounded an activation to bf16 the
    other way, was 1.8e-3 off (400 drawn cases). The IQ formats' decode products also round each 32-column sum to a
    whole number of scale steps."""
    if case["kind"] == "head":
        return {"rel": 1e-6, "max": 1e-5}
    return {"rel": 4e-3, "max": 0.1}


# ---- states ---------------------------------------------------------------------------------------------------------

def _grids():
    """Seeded codebooks of the IQ formats' shapes (a checkpoint's runtime brings its own)."""
    rng = np.random.default_rng(11)
    a = rng.choice(np.array([4, 12, 20, 28, 36, 44, 52, 62], np.uint8), size=(256, 4))
    b = rng.choice(np.arange(1, 16, 2, dtype=np.uint8), size=(512, 4))
    c = rng.choice(np.array([8, 25, 43], np.uint8), size=(1024, 8))
    return a, b, c


_registered = False


def _register_grids() -> None:
    global _registered
    if not _registered:
        grids = _grids()
        call("fns_hip_set_iq_grids", *(g.ctypes.data_as(ctypes.c_void_p) for g in grids))
        _registered = True


def _matrix(qtype: int, n_mat: int, nrows: int, ncols: int, seed: int, out: torch.Tensor) -> None:
    """out [n_mat][bytes] <- N(0, 0.02) quantised to the K-quants and Q8_0, random blocks of that size for the IQ types."""
    if qtype in synth.IQ_BLOCK_BYTES:
        blocks = torch.empty(n_mat * nrows * ncols // 256 * BLOCK[qtype], dtype=torch.uint8, device="cuda")
        synth.random_iq_blocks(qtype, n_mat * nrows * ncols // 256, seed, blocks)
        out.copy_(blocks.view(n_mat, -1))
    else:
        synth.quantized_matrices(qtype, n_mat, nrows, ncols, seed, 0.02, out)


def _plain(qtype: int, nrows: int, ncols: int, seed: int) -> torch.Tensor:
    t = torch.empty(_mat(qtype, nrows, ncols), dtype=torch.uint8, device="cuda")
    _matrix(qtype, 1, nrows, ncols, seed, t.view(1, -1))
    return t


def _normal(shape, seed: int, mean: float = 0.0, std: float = 1.0) -> torch.Tensor:
    g = torch.Generator(device="cuda")
    g.manual_seed(seed & 0x7FFFFFFFFFFFFFFF)
    return torch.empty(*shape, device="cuda").normal_(mean, std, generator=g)


def _moe_layer(c: dict, seed: int, l: int) -> ops.MoeLayer:
    s = lambda kind: synth.tensor_seed(seed + 1, l, kind)  # noqa: E731
    H, F, E = c["hidden"], c["inter"], c["experts"]
    router = _normal((E, H), s(0), std=0.02)
    slots = ops.ExpertSlots(E, _mat(c["gu"], F, H), _mat(c["gu"], F, H), _mat(c["down"], H, F))
    _matrix(c["gu"], E, F, H, s(1), slots.view("gate"))
    _matrix(c["gu"], E, F, H, s(2), slots.view("up"))
    _matrix(c["down"], E, H, F, s(3), slots.view("down"))
    bias = None
    if c.get("skew"):
        load = np.random.default_rng(s(4)).dirichlet(np.full(E, 0.3))
        bias = torch.from_numpy((np.log(load + 1e-6) * 0.5).astype(np.float32)).cuda()
    if not c["block"]:
        return ops.MoeLayer(router, slots, c["gu"], c["down"], H, F, c["k"], router_bias=bias)
    shexp = {"gate": _plain(c["gu"], 2 * F, H, s(5)), "up": _plain(c["gu"], 2 * F, H, s(6)),
             "down": _plain(c["down"], H, 2 * F, s(7)), "inter": 2 * F, "gu_type": c["gu"], "down_type": c["down"]}
    return ops.MoeLayer(router.to(torch.bfloat16), slots, c["gu"], c["down"], H, F, c["k"], router_bias=bias,
                        gating=ops.GATING_SIGMOID, guard=True, ffn_norm=_normal((H,), s(8), 1.0, 0.1), norm_eps=EPS,
                        shexp=shexp)


def _inputs(case: dict, seed: int):
    """(layers or matrices, x of every layer)."""
    c = case
    if {c["gu"], c.get("down")} & set(synth.IQ_BLOCK_BYTES):
        _register_grids()
    L, H = c["layers"], c["hidden"]
    xs = [_normal((c["tokens"], H), synth.tensor_seed(seed + 1, l, 20)) for l in range(L)]
    if c["kind"] == "head":
        return _plain(c["gu"], c["inter"], H, synth.tensor_seed(seed + 1, 0, 1)), xs
    if c["kind"] in ("dense", "dense_prefill"):
        F, ffns = c["inter"], []
        for l in range(L):
            s = lambda kind: synth.tensor_seed(seed + 1, l, kind)  # noqa: E731
            ffns.append(ops.DenseFfn(_plain(c["gu"], F, H, s(1)), _plain(c["gu"], F, H, s(2)),
                                     _plain(c["down"], H, F, s(3)), c["gu"], c["gu"], c["down"], H, F,
                                     ffn_norm=_normal((H,), s(8), 1.0, 0.1), norm_eps=EPS))
        return ffns, xs
    layers = [_moe_layer(c, seed, l) for l in range(L)]
    if c["kind"] == "layer":  # an engine names the bytes that the next layer reads first
        for l, layer in enumerate(layers):
            nxt = layers[(l + 1) % L].router_w
            layer.desc.prefetch, layer.desc.prefetch_bytes = nxt.data_ptr(), nxt.numel() * nxt.element_size()
    return layers, xs


def _calls(layers, xs, outs, c: dict):
    """The decode step of an engine on the kernel-launch API: seven calls per layer on the engine's own buffers."""
    H, F, E, k = c["hidden"], c["inter"], c["experts"], c["k"]
    P = ctypes.c_void_p
    buf = {"logits": torch.empty(E, device="cuda"), "ids": torch.empty(k, dtype=torch.int32, device="cuda"),
           "w": torch.empty(k, device="cuda"), "act": torch.empty(k, F, device="cuda"),
           "xq": torch.zeros(k, ops.q8_1_row_bytes(max(H, F)), dtype=torch.uint8, device="cuda"),
           "esc": torch.empty(k, device="cuda"), "dexp": torch.empty(k, H, device="cuda")}
    logits, ids, w, act, xq, esc, dexp = (P(buf[n].data_ptr()) for n in ("logits", "ids", "w", "act", "xq", "esc", "dexp"))

    def step():
        st = P(torch.cuda.current_stream().cuda_stream)
        for layer, x, out in zip(layers, xs, outs):
            s = layer.slots
            xp, op, table = P(x.data_ptr()), P(out.data_ptr()), P(s.table.data_ptr())
            call("fns_hip_gemv_router", 0, P(layer.router_w.data_ptr()), xp, logits, H, E, 1, st)
            call("fns_hip_route_topk", logits, ids, w, E, k, 1, 0, 1, st)
            call("fns_hip_quantize_q8_1", xp, xq, H, 1, st)
            call("fns_hip_mmvq_experts_swiglu", c["gu"], table, s.gate_off, s.up_off, H, F, xq, 1, ids, k, act, st)
            call("fns_hip_amax_guard_q8_1", act, esc, xq, F, k, st)
            call("fns_hip_mmvq_experts", c["down"], table, s.down_off, F, H, xq, k, ids, k, dexp, st)
            call("fns_hip_moe_combine", dexp, esc, w, None, xp, op, H, k, 1, st)

    return step, buf


def prepare(case: dict, seed: int) -> dict:
    c = case
    mods, xs = _inputs(c, seed)
    T, state = c["tokens"], {"case": c, "mods": mods, "xs": xs}
    if c["kind"] == "head":
        state["xq"] = torch.zeros(T, ops.q8_1_row_bytes(c["hidden"]), dtype=torch.uint8, device="cuda")
        state["outs"] = [torch.empty(T, c["inter"], device="cuda")]
        return state
    outs = state["outs"] = [torch.empty_like(x) for x in xs]
    if c["kind"] == "calls":
        step, state["buf"] = _calls(mods, xs, outs, c)
    else:
        if c["kind"] == "prefill":
            state["mods"] = mods = [ops.MoePrefill(m) for m in mods]
        wss = state["wss"] = [m.workspace(T) for m in mods]
        if c["kind"] in ("dense", "dense_prefill"):
            pre = c["kind"] == "dense_prefill"

            def step():
                for m, x, o, w in zip(mods, xs, outs, wss):
                    m(x, out=o, ws=w, prefill=pre)
        elif c["block"]:
            def step():
                for m, x, o, w in zip(mods, xs, outs, wss):
                    m(x, out=o, ws=w, x_resid=x)
        else:
            def step():
                for m, x, o, w in zip(mods, xs, outs, wss):
                    m(x, out=o, ws=w)
    state["step"] = step
    if c["layers"] > 1:
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            step()
        torch.cuda.current_stream().wait_stream(side)
        torch.cuda.synchronize()
        state["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(state["graph"]):
            step()
    return state


def run(state: dict):
    if state["case"]["kind"] == "head":
        c, x = state["case"], state["xs"][0]
        ops.quantize_q8_1(x, state["xq"])
        ops.mmvq(c["gu"], state["mods"], c["hidden"], c["inter"], state["xq"], c["tokens"], dst=state["outs"][0])
    elif "graph" in state:
        state["graph"].replay()
    else:
        state["step"]()
    return state["outs"]


# ---- the same in 64 bits --------------------------------------------------------------------------------------------

def _f16(b: torch.Tensor) -> torch.Tensor:
    """The f16 in bytes b[..., 0:2], as f64 [..., 1]."""
    return b.contiguous().view(torch.float16).double()


def _scale_min(s: torch.Tensor):
    """The 8 six-bit scales and minima in 12 bytes."""
    lo, hi, top = s[:, 0:4], s[:, 4:8], s[:, 8:12]
    sc = torch.cat([lo & 63, (top & 15) | ((lo >> 6) << 4)], 1)
    mn = torch.cat([hi & 63, (top >> 4) | ((hi >> 6) << 4)], 1)
    return sc.double(), mn.double()


def _dequantize(qtype: int, data: torch.Tensor, nrows: int, ncols: int) -> torch.Tensor:
    """GGUF blocks -> f64 [nrows][ncols]."""
    b = data.reshape(-1, 34 if qtype == Q8_0 else BLOCK[qtype])
    n = b.shape[0]
    if qtype == Q8_0:
        y = _f16(b[:, 0:2]) * b[:, 2:34].contiguous().view(torch.int8).double()
        return y.view(nrows, ncols)
    if qtype in (Q4_K, Q5_K):
        d, dmin = _f16(b[:, 0:2]), _f16(b[:, 2:4])
        sc, mn = _scale_min(b[:, 4:16].int())
        qs = b[:, -128:].view(n, 4, 1, 32)
        q = torch.cat([qs & 15, qs >> 4], 2).view(n, 8, 32)
        if qtype == Q5_K:
            bit = torch.arange(8, device=b.device, dtype=torch.uint8).view(1, 8, 1)
            q = q + (((b[:, 16:48].view(n, 1, 32) >> bit) & 1) << 4)
        y = (d * sc).view(n, 8, 1) * q.double() - (dmin * mn).view(n, 8, 1)
    elif qtype == Q6_K:
        ql, qh = b[:, 0:128].view(n, 2, 2, 32), b[:, 128:192].view(n, 2, 1, 32)
        low = torch.cat([ql & 15, ql >> 4], 2)                                     # [n][half][4][32]
        two = torch.arange(0, 8, 2, device=b.device, dtype=torch.uint8).view(1, 1, 4, 1)
        q = (low | (((qh >> two) & 3) << 4)).double() - 32
        sc = b[:, 192:208].contiguous().view(torch.int8).double()
        y = (_f16(b[:, 208:210]) * sc).view(n, 16, 1) * q.view(n, 16, 16)
    elif qtype == Q3_K:
        two = torch.arange(0, 8, 2, device=b.device, dtype=torch.uint8).view(1, 1, 4, 1)
        q = ((b[:, 32:96].view(n, 2, 1, 32) >> two) & 3).double()
        bit = torch.arange(8, device=b.device, dtype=torch.uint8).view(1, 2, 4, 1)
        q = q - 4 * (1 - ((b[:, 0:32].view(n, 1, 1, 32) >> bit) & 1).double())
        s = b[:, 96:108].int()
        lo = torch.cat([s[:, 0:8] & 15, s[:, 0:8] >> 4], 1)
        hi = torch.cat([(s[:, 8:12] >> (2 * j)) & 3 for j in range(4)], 1)
        sc = ((lo | (hi << 4)) - 32).double()
        y = (_f16(b[:, 108:110]) * sc).view(n, 16, 1) * q.reshape(n, 16, 16)
    elif qtype == IQ4_XS:
        values = torch.tensor([-127, -104, -83, -65, -49, -35, -22, -10, 1, 13, 25, 38, 53, 69, 89, 113],
                              dtype=torch.float64, device=b.device)
        h = b[:, 2].int() | (b[:, 3].int() << 8)
        ls = torch.stack([((b[:, 4 + j // 2].int() >> (4 * (j % 2))) & 15) | (((h >> (2 * j)) & 3) << 4)
                          for j in range(8)], 1).double() - 32
        qs = b[:, 8:136].view(n, 8, 16)
        y = (_f16(b[:, 0:2]) * ls).view(n, 8, 1) * values[torch.cat([qs & 15, qs >> 4], 2).long()]
    else:
        grid = torch.from_numpy(_grids()[0 if qtype == IQ3_XXS else 1]).to(b.device).double()
        if qtype == IQ3_XXS:
            aux = b[:, 66:98].contiguous().view(torch.int32).long() & 0xFFFFFFFF     # [n][8]
            db = (0.5 + (aux >> 28).double()) * 0.5
            v = torch.stack([(aux >> (7 * l)) & 127 for l in range(4)], 2)           # [n][8][4]
            bits = torch.stack([(v >> j) & 1 for j in range(7)], 3)
            neg = torch.cat([bits, bits.sum(3, keepdim=True) & 1], 3)                # an even number of signs
            idx = b[:, 2:66].long()
        else:
            s = b[:, 106:110].int()
            db = 1 + 2 * torch.stack([(s[:, j // 2] >> (4 * (j % 2))) & 15 for j in range(8)], 1).double()
            sg = b[:, 74:106].int()
            neg = torch.stack([(sg >> j) & 1 for j in range(8)], 2)
            qh = torch.stack([(b[:, 66:74].int() >> l) & 1 for l in range(8)], 2).view(n, 64)
            idx = b[:, 2:66].long() | (qh.long() << 8)
        g = grid[idx].view(n, 8, 32) * (1 - 2 * neg.reshape(n, 8, 32).double())
        y = (_f16(b[:, 0:2]) * db).view(n, 8, 1) * g
    return y.reshape(nrows, ncols)


def _q8_1(x: torch.Tensor) -> torch.Tensor:
    """x through 8-bit blocks of 32 (codes x / (amax / 127) rounded half away from zero, a scale stored in f16), f64."""
    v = x.float().view(-1, 32)
    d = v.abs().amax(1, keepdim=True) / 127
    r = torch.where(d > 0, v / d, torch.zeros_like(v))
    q = torch.sign(r) * torch.floor(r.abs() + 0.5)
    return (q.double() * d.half().double()).view(x.shape)


def _ffn(xq, gate, up, down, c: dict, inter: int) -> torch.Tensor:
    H = c["hidden"]
    g = xq @ _dequantize(c["gu"], gate, inter, H).T
    u = xq @ _dequantize(c["gu"], up, inter, H).T
    return _q8_1(u * g * torch.sigmoid(g)) @ _dequantize(c["down"], down, H, inter).T


def _rms(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    x = x.double()
    return x / torch.sqrt((x * x).mean(1, keepdim=True) + EPS) * w.double()


def _moe(layer: ops.MoeLayer, x: torch.Tensor, c: dict) -> torch.Tensor:
    h = _rms(x, layer.ffn_norm).float() if c["block"] else x
    # prompts' bf16 routers take the activations in bf16, as the reference's BF16 GEMM does
    hr = h.to(torch.bfloat16) if c["block"] and c["kind"] == "prefill" else h
    logits = hr.double() @ layer.router_w.double().T
    if layer.router_bias is not None:
        logits = logits + layer.router_bias.double()
    p = torch.sigmoid(logits) if c["block"] else torch.softmax(logits, 1)
    w, ids = torch.topk(p, c["k"], dim=1)
    w = w / w.sum(1, keepdim=True).clamp_min(6.103515625e-5)
    xq, slots = _q8_1(h), layer.slots
    out = x.double() if c["block"] or c["kind"] == "calls" else torch.zeros_like(x, dtype=torch.float64)
    if c["block"]:
        sh = layer.shexp
        out = out + _ffn(xq, sh["gate"], sh["up"], sh["down"], c, sh["inter"])
    for e in ids.unique().tolist():
        t, j = (ids == e).nonzero(as_tuple=True)
        y = _ffn(xq[t], slots.view("gate")[e], slots.view("up")[e], slots.view("down")[e], c, c["inter"])
        out = out.index_add(0, t, y * w[t, j].unsqueeze(1))
    return out


def exact(case: dict, seed: int):
    c = case
    mods, xs = _inputs(c, seed)
    if c["kind"] == "head":
        xq, out = _q8_1(xs[0]), []
        row = c["hidden"] // 256 * BLOCK[c["gu"]]
        for r in range(0, c["inter"], 8192):
            n = min(8192, c["inter"] - r)
            out.append(xq @ _dequantize(c["gu"], mods[r * row: (r + n) * row], n, c["hidden"]).T)
        return [torch.cat(out, 1)]
    if c["kind"] in ("dense", "dense_prefill"):
        return [x.double() + _ffn(_q8_1(_rms(x, m.ffn_norm)), m.gate, m.up, m.down, c, c["inter"])
                for m, x in zip(mods, xs)]
    return [_moe(m, x, c) for m, x in zip(mods, xs)]
