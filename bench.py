#!/usr/bin/env python3
"""bench.py - MI355X MoE FFN decode benchmark (BASELINE.json metric: us/token per MoE layer + achieved HBM GB/s,
batch 1, Q4_K experts).

    python bench.py [--gpus 1] [--steps K] [--warmup W] [--layers L] [--no-cpu] [--no-extra]

Workload (config 0): one MoE FFN layer at batch 1 - hidden 2048, 128 experts, top-8 softmax gating with
renormalisation, SwiGLU experts of width 768, gate/up/down Q4_K (ggml reference quantiser on N(0, 0.02)), fp32
router N(0, 0.02), x ~ N(0, 1) fresh per layer and step. A "step" is one token through L resident copies of that
layer (distinct weights, L * 340 MB > the 256 MB Infinity Cache, so every layer streams its experts from HBM);
value = step time / L. All inputs are resident in HBM before the timed region; each layer is the library's
fns_hip_moe_layer call, replayed from a HIP graph, with the read-ahead hint naming the next layer's router.

The JSON line also carries:
  roofline     - for the dominant kernel (k_layer_fused: routing, gate/up + SwiGLU, Q8_1 of act, down, combine):
                 algorithmic bytes per launch (8 experts x gate + up + down Q4_K = 21,233,664 B) / its average
                 duration, timed with HIP events on the launch stream over back-to-back launches on rotating layers;
                 peak 8 TB/s (MI355X HBM3E); traffic from the committed rocprofv3 FETCH_SIZE / WRITE_SIZE summary
                 (profiles/) when present.
  cpu_baseline - the oracle's OpenMP CPU restatement of the same layer (int8 x K-quant dot products, not ggml), timed
                 on this host's cores on a bounded sample.
  extra        - configs 1 (Q3_K/Q5_K mix), 2 (4-token speculative verify), 3 (48-layer Q4_K/Q6_K stack) and 4
                 (512-token prefill through the grouped GEMM on int8 MFMA, Dirichlet(0.3)-skewed router bias; MFMA
                 utilisation = 38.65 G int8 ops per layer / time / 5.0 POP/s dense int8 peak), the reference
                 model's whole MoE block (RMSNorm, 256 experts top-6 sigmoid, width 512, shared expert) at decode with
                 K-quant and with IQ3_XXS / IQ3_S gate/up + IQ4_XS down experts, and its dense FFN block (2048 ->
                 6144, Q8_0) at 512 prefill tokens.
"""
from __future__ import annotations

import argparse
import json
import os
import re
import sys
import time
import warnings
from pathlib import Path

ROOT = Path(__file__).resolve().parent
sys.path.insert(0, str(ROOT))

H, F, NE, K_TOP = 2048, 768, 128, 8
SEED = 20261022
Q3_K, Q4_K, Q5_K, Q6_K = 11, 12, 13, 14
BLOCK = {Q3_K: 110, Q4_K: 144, Q5_K: 176, Q6_K: 210}
PEAK_GBS = 8000.0


def expert_bytes(gu: int, dn: int) -> int:
    return 2 * F * (H // 256) * BLOCK[gu] + H * (F // 256) * BLOCK[dn]


def layer_bytes(gu: int, dn: int, n_distinct: int = K_TOP) -> int:
    """Algorithmic HBM bytes of one layer-token: the selected experts' gate/up/down blocks + the fp32 router."""
    return n_distinct * expert_bytes(gu, dn) + NE * H * 4


def log(msg: str) -> None:
    print(msg, file=sys.stderr, flush=True)


def build_layers(synth, n: int, gu: int, dn: int, seed_base: int):
    return link_prefetch([synth.build_layer(H, F, NE, K_TOP, gu, dn, SEED, layer=seed_base + l) for l in range(n)])


def link_prefetch(layers):
    """Each layer's read-ahead hint names the next layer's router (FnsMoeLayer.prefetch), as an engine stepping
    through its layers would pass it; the outputs do not depend on it."""
    for l, layer in enumerate(layers):
        nxt = layers[(l + 1) % len(layers)].router_w
        layer.desc.prefetch, layer.desc.prefetch_bytes = nxt.data_ptr(), nxt.numel() * nxt.element_size()
    return layers


def make_xs(synth, torch, n_tok: int, n_steps: int, n_layers: int, seed_layer0: int):
    """x[s][l] ~ N(0, 1) [n_tok][H]: fresh per (step, layer)."""
    xs = torch.empty(n_steps, n_layers, n_tok, H, device="cuda")
    for l in range(n_layers):
        for s in range(n_steps):
            xs[s, l].copy_(synth.activations(n_tok, H, SEED, layer=seed_layer0 + l, step=s))
    return xs


def capture(torch, layers, xs, outs, wss, steps_per_graph: int):
    g = torch.cuda.CUDAGraph()
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        for st in range(steps_per_graph):  # eager warm-up of every launch in the graph
            for l, layer in enumerate(layers):
                layer(xs[st, l], out=outs[l], ws=wss[l])
    torch.cuda.current_stream().wait_stream(s)
    torch.cuda.synchronize()
    with torch.cuda.graph(g):
        for st in range(steps_per_graph):
            for l, layer in enumerate(layers):
                layer(xs[st, l], out=outs[l], ws=wss[l])
    return g


IQ3_XXS, IQ3_S, IQ4_XS, Q8_0 = 18, 21, 23, 8
BLOCK.update({IQ3_XXS: 98, IQ3_S: 110, IQ4_XS: 136})


def run_flint(torch, synth, n_layers: int = 8, replays: int = 40, gu: int = Q4_K, dn: int = Q5_K) -> dict:
    """The reference model's MoE block shape (src/model.cpp:159-164: RMSNorm, bf16 router, sigmoid top-6 of 256
    experts of width 512, F16 guard, shared expert of width 1024; gate/up Q4_K, down Q5_K, or the checkpoint's IQ
    formats with random blocks and seeded codebooks), decode batch 1 through fns_hip_moe_layer with the residual
    added; n_layers resident copies replayed in one graph."""
    if gu in synth.IQ_BLOCK_BYTES or dn in synth.IQ_BLOCK_BYTES:
        synth.register_iq_grids()
        layers = [synth.build_iq_flint_layer(H, 512, 256, 6, 1024, gu, dn, SEED, layer=600 + l)
                  for l in range(n_layers)]
    else:
        layers = [synth.build_flint_layer(H, 512, 256, 6, 1024, gu, dn, SEED, layer=600 + l) for l in range(n_layers)]
    link_prefetch(layers)
    xs = [synth.activations(1, H, SEED, layer=700 + l) for l in range(n_layers)]
    outs = [torch.empty(1, H, device="cuda") for _ in layers]
    wss = [layer.workspace(1) for layer in layers]
    g = torch.cuda.CUDAGraph()
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        for l, layer in enumerate(layers):
            layer(xs[l], out=outs[l], ws=wss[l], x_resid=xs[l])
    torch.cuda.current_stream().wait_stream(s)
    torch.cuda.synchronize()
    with torch.cuda.graph(g):
        for l, layer in enumerate(layers):
            layer(xs[l], out=outs[l], ws=wss[l], x_resid=xs[l])
    us = time_graph(torch, g, replays, 3) * 1e3 / n_layers
    routed = 6 * (2 * 512 * (H // 256) * BLOCK[gu] + H * 2 * BLOCK[dn])
    shared = 2 * 1024 * (H // 256) * BLOCK[gu] + H * 4 * BLOCK[dn]
    byts = routed + shared + 256 * H * 2
    del g
    return {"us_per_layer": round(us, 3), "hbm_bytes_per_layer": byts, "hbm_gbs": round(byts / (us * 1e-6) / 1e9, 1)}


def time_graph(torch, g, replays: int, warmup: int) -> float:
    """ms per replay."""
    for _ in range(warmup):
        g.replay()
    torch.cuda.synchronize()
    e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    e0.record()
    for _ in range(replays):
        g.replay()
    e1.record()
    torch.cuda.synchronize()
    return e0.elapsed_time(e1) / replays


def replay_spread(torch, g, n: int, layers_per_replay: int) -> dict:
    """After the timed region: n replays of the same graph, each between its own pair of HIP events, as µs per
    layer (median, 10th and 90th percentile), so that the value's mean over a few replays can be read against the
    distribution."""
    evs = [(torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)) for _ in range(n)]
    for e0, e1 in evs:
        e0.record()
        g.replay()
        e1.record()
    torch.cuda.synchronize()
    v = sorted(e0.elapsed_time(e1) * 1e3 / layers_per_replay for e0, e1 in evs)
    return {"median": round(v[n // 2], 3), "p10": round(v[n // 10], 3), "p90": round(v[(9 * n) // 10], 3), "n": n}


def stage_times(torch, layers, xs, outs, wss, reps: int) -> list[float]:
    """Average duration (us) of each of the three kernels, timed with HIP events on the launch stream around graph
    replays of back-to-back launches of that kernel over the L rotating layers (each reads what the previous stage
    left in its workspace)."""
    L = len(layers)
    graphs = []
    for k in range(3):
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            for l, layer in enumerate(layers):
                layer.stage(k, xs[0, l], outs[l], wss[l])
        graphs.append(g)
    ev = [torch.cuda.Event(enable_timing=True) for _ in range(6)]
    tot = [0.0, 0.0, 0.0]
    for _ in range(2):
        for g in graphs:
            g.replay()
    torch.cuda.synchronize()
    for _ in range(reps):
        for k, g in enumerate(graphs):
            ev[2 * k].record()
            g.replay()
            ev[2 * k + 1].record()
        torch.cuda.synchronize()
        for k in range(3):
            tot[k] += ev[2 * k].elapsed_time(ev[2 * k + 1]) * 1e3 / L
    return [t / reps for t in tot]


def read_traffic() -> dict | None:
    """HBM bytes per k_gate_up launch from the committed rocprofv3 --pmc summary (calibrated), if present."""
    p = ROOT / "profiles" / "k_layer_fused_cfg0_traffic.md"
    if not p.exists():
        return None
    m = re.search(r"traffic_bytes_per_launch:\s*([0-9.eE+]+)", p.read_text())
    return {"bytes": round(float(m.group(1)))} if m else None


def cpu_baseline(torch, layer, budget_s: float = 15.0) -> dict:
    """Oracle CPU restatement of one config-0 layer on this host (bounded sample)."""
    import numpy as np

    from oracle import oracle as orc
    host = host_cpus()
    nthreads = host["threads"]
    router = layer.router_w.cpu().numpy()
    slots = [layer.slots.expert_bytes(e).cpu().numpy() for e in range(NE)]
    xs = [torch.randn(H, generator=torch.Generator().manual_seed(SEED + i)).numpy().astype(np.float32) for i in range(4)]
    args = (Q4_K, Q4_K, router, slots, layer.slots.gate_off, layer.slots.up_off, layer.slots.down_off)
    orc.cpu_moe_layer(*args, xs[0], H, F, K_TOP, nthreads)  # warm-up
    n, t0 = 0, time.perf_counter()
    while True:
        orc.cpu_moe_layer(*args, xs[n % 4], H, F, K_TOP, nthreads)
        n += 1
        dt = time.perf_counter() - t0
        if dt > budget_s:
            break
    return {"value": dt / n * 1e6, "unit": "us/layer", "cores": nthreads, "kind": "port",
            "sample": f"{n} batch-1 config-0 layers (Q4_K, 128 experts, top-8) with fresh x, {dt:.1f} s; OpenMP "
                      f"restatement in oracle/fns_oracle.c (int8 x K-quant integer dots), not ggml (llama.cpp is not "
                      f"on the box)", **{k: v for k, v in host.items() if k != "threads"}}


def host_cpus() -> dict:
    """The host's CPU model and counts, and the threads the baseline runs: every CPU this process may use (its
    affinity mask and cgroup CPU quota), or OMP_NUM_THREADS when the job sets it (the GPU boxes allot 16 cores per
    GPU that way)."""
    model = ""
    try:
        for line in open("/proc/cpuinfo"):
            if line.startswith("model name"):
                model = line.split(":", 1)[1].strip()
                break
    except OSError:
        pass
    affinity = len(os.sched_getaffinity(0))
    quota = None
    try:
        q, period = open("/sys/fs/cgroup/cpu.max").read().split()
        if q != "max":
            quota = int(q) / int(period)
    except (OSError, ValueError):
        pass
    threads = affinity if quota is None else max(1, min(affinity, int(quota)))
    omp = os.environ.get("OMP_NUM_THREADS", "")
    if omp.isdigit() and int(omp) > 0:
        threads = int(omp)
    return {"threads": threads, "cpu_model": model, "host_cpus": os.cpu_count(), "affinity_cpus": affinity,
            "cgroup_cpu_quota": quota, "omp_num_threads": omp or None}


def run_stack(torch, synth, gu: int, dn: int, n_layers: int, n_tok: int, steps: int, warmup: int, seed_base: int,
              steps_per_graph: int = 4):
    layers = build_layers(synth, n_layers, gu, dn, seed_base)
    xs = make_xs(synth, torch, n_tok, steps_per_graph, n_layers, seed_base + 500)
    outs = [torch.empty(n_tok, H, device="cuda") for _ in layers]
    wss = [layer.workspace(n_tok) for layer in layers]
    g = capture(torch, layers, xs, outs, wss, steps_per_graph)
    replays = max(1, steps // steps_per_graph)
    ms = time_graph(torch, g, replays, warmup)
    distinct = float(sum(len(torch.unique(layer.trace(ws, n_tok)["ids"])) for layer, ws in zip(layers, wss)) / n_layers)
    del g
    return layers, ms / steps_per_graph, distinct


def run_prefill(torch, synth, n_layers: int = 4, T: int = 512, replays: int = 10) -> dict:
    """Config 4: T tokens through n_layers resident Q4_K layers (distinct weights), each with its own seeded
    Dirichlet(0.3) router bias; one graph replay = one prefill of every layer."""
    import numpy as np

    from flintnsteel_amd import ops
    rng = np.random.default_rng(SEED)
    pres = []
    for l in range(n_layers):
        base = synth.build_layer(H, F, NE, K_TOP, Q4_K, Q4_K, SEED, layer=400 + l)
        bias = torch.from_numpy((np.log(rng.dirichlet(np.full(NE, 0.3)) + 1e-6) * 0.5).astype(np.float32)).cuda()
        pres.append(ops.MoePrefill(ops.MoeLayer(base.router_w, base.slots, Q4_K, Q4_K, H, F, K_TOP,
                                                router_bias=bias)))
    xs = [synth.activations(T, H, SEED, layer=500 + l) for l in range(n_layers)]
    outs = [torch.empty(T, H, device="cuda") for _ in range(n_layers)]
    wss = [p.workspace(T) for p in pres]
    g = torch.cuda.CUDAGraph()
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        for l in range(n_layers):
            pres[l](xs[l], out=outs[l], ws=wss[l])
    torch.cuda.current_stream().wait_stream(s)
    torch.cuda.synchronize()
    with torch.cuda.graph(g):
        for l in range(n_layers):
            pres[l](xs[l], out=outs[l], ws=wss[l])
    ms = time_graph(torch, g, replays, 2)
    us = ms * 1e3 / n_layers
    ids = [p.trace(w, T)["ids"].cpu().numpy() for p, w in zip(pres, wss)]
    touched = float(np.mean([len(np.unique(i)) for i in ids]))
    max_load = float(np.mean([np.bincount(i.ravel(), minlength=NE).max() for i in ids]))
    loads = [np.bincount(i.ravel(), minlength=NE) for i in ids]
    groups = float(np.mean([np.sum((n + 63) // 64) for n in loads]))       # workgroup row groups of 64
    tiles = float(np.mean([np.sum((n + 31) // 32) for n in loads]))        # 32-row MFMA tiles computed
    ops_per_layer = 2 * T * K_TOP * (2 * F * H + H * F)
    del g
    return {"us_per_layer": round(us, 2), "tokens_per_s": round(T / us * 1e6, 0), "experts_touched": touched,
            "max_expert_load": max_load, "row_groups": groups, "tile_fill": round(T * K_TOP / (32 * tiles), 3),
            "weight_gbs": round(touched * expert_bytes(Q4_K, Q4_K) / (us * 1e-6) / 1e9, 1),
            "int8_tops": round(ops_per_layer / (us * 1e-6) / 1e12, 2),
            "mfma_util": round(ops_per_layer / (us * 1e-6) / 5.0e15, 4)}


def run_dropin(torch, layers, replays: int = 40) -> dict:
    """The reference's decode MoE sequence (Engine::ffn_block, src/engine.cu:670-694, without RMSNorm and shared
    expert) as its seven separate calls through the drop-in C ABI - gemv router, route_topk, quantize_q8_1,
    mmvq_experts_swiglu, amax_guard_q8_1, mmvq_experts, moe_combine - on preallocated buffers (as the engine holds
    them), over the config-0 layers, replayed from one graph."""
    import ctypes

    from flintnsteel_amd import ops
    from flintnsteel_amd._lib import call
    L = len(layers)
    P = ctypes.c_void_p
    st = lambda: P(torch.cuda.current_stream().cuda_stream)  # noqa: E731
    xs = [torch.randn(1, H, device="cuda") for _ in range(L)]
    outs = [torch.empty(1, H, device="cuda") for _ in range(L)]
    logits = torch.empty(NE, device="cuda")
    ids = torch.empty(K_TOP, dtype=torch.int32, device="cuda")
    w = torch.empty(K_TOP, device="cuda")
    xq = torch.zeros(K_TOP, ops.q8_1_row_bytes(max(H, F)), dtype=torch.uint8, device="cuda")
    act = torch.empty(K_TOP, F, device="cuda")
    esc = torch.empty(K_TOP, device="cuda")
    dexp = torch.empty(K_TOP, H, device="cuda")
    p = lambda t: P(t.data_ptr())  # noqa: E731

    def step():
        for l, layer in enumerate(layers):
            s = layer.slots
            call("fns_hip_gemv_router", 0, p(layer.router_w), p(xs[l]), p(logits), H, NE, 1, st())
            call("fns_hip_route_topk", p(logits), p(ids), p(w), NE, K_TOP, 1, 0, 1, st())
            call("fns_hip_quantize_q8_1", p(xs[l]), p(xq), H, 1, st())
            call("fns_hip_mmvq_experts_swiglu", Q4_K, p(s.table), s.gate_off, s.up_off, H, F, p(xq), 1, p(ids), K_TOP,
                 p(act), st())
            call("fns_hip_amax_guard_q8_1", p(act), p(esc), p(xq), F, K_TOP, st())
            call("fns_hip_mmvq_experts", Q4_K, p(s.table), s.down_off, F, H, p(xq), K_TOP, p(ids), K_TOP, p(dexp), st())
            call("fns_hip_moe_combine", p(dexp), p(esc), p(w), None, p(xs[l]), p(outs[l]), H, K_TOP, 1, st())

    g = torch.cuda.CUDAGraph()
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        step()
    torch.cuda.current_stream().wait_stream(s)
    torch.cuda.synchronize()
    with torch.cuda.graph(g):
        step()
    us = time_graph(torch, g, replays, 3) * 1e3 / L
    del g
    return {"us_per_layer": round(us, 3), "launches_per_layer": 7}


def run_dense_q8_0(torch, n_layers: int = 4, T: int = 512, replays: int = 10) -> dict:
    """The reference model's dense FFN block (src/model.cpp:121-125,163: hidden 2048, FFN 6144, the leading two
    layers) with Q8_0 gate / up / down, prefill of T tokens through fns_hip_dense_ffn_prefill (RMSNorm, mmq of gate
    and up, SwiGLU, mmq of down, residual), and one Q8_0 mmq (2048 -> 6144) alone; n_layers resident copies."""
    from flintnsteel_amd import ops, synth
    FD = 6144
    ffns, mats = [], []
    for l in range(n_layers):
        g = torch.empty(FD * ops.row_bytes(Q8_0, H), dtype=torch.uint8, device="cuda")
        u, d = torch.empty_like(g), torch.empty(H * ops.row_bytes(Q8_0, FD), dtype=torch.uint8, device="cuda")
        for t, (nr, nc), kind in ((g, (FD, H), 1), (u, (FD, H), 2), (d, (H, FD), 3)):
            synth.quantized_matrices(Q8_0, 1, nr, nc, synth.tensor_seed(SEED, 800 + l, kind), 0.02, t.view(1, -1))
        norm = ops.fill_normal(torch.empty(H, device="cuda"), synth.tensor_seed(SEED, 800 + l, 9), mean=1.0, std=0.1)
        ffns.append(ops.DenseFfn(g, u, d, Q8_0, Q8_0, Q8_0, H, FD, ffn_norm=norm, norm_eps=1e-6))
        mats.append(g)
    xs = [synth.activations(T, H, SEED, layer=900 + l) for l in range(n_layers)]
    outs = [torch.empty(T, H, device="cuda") for _ in range(n_layers)]
    wss = [f.workspace(T) for f in ffns]
    ys = [torch.empty(T, FD, device="cuda") for _ in range(n_layers)]
    xq = torch.empty(ops.mmq_q8_1_bytes(H, T), dtype=torch.uint8, device="cuda")
    res = {}
    for name, fn in (("dense_ffn", lambda l: ffns[l](xs[l], out=outs[l], ws=wss[l], prefill=True)),
                     ("mmq", lambda l: ops.mmq(Q8_0, mats[l], H, FD, xs[l], xq=xq, out=ys[l]))):
        gr = torch.cuda.CUDAGraph()
        s = torch.cuda.Stream()
        s.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(s):
            for l in range(n_layers):
                fn(l)
        torch.cuda.current_stream().wait_stream(s)
        torch.cuda.synchronize()
        with torch.cuda.graph(gr):
            for l in range(n_layers):
                fn(l)
        res[name] = time_graph(torch, gr, replays, 2) * 1e3 / n_layers
        del gr
    wbytes = 3 * FD * H * 34 // 32
    flops = 2 * T * 3 * FD * H
    return {"dense_ffn_us": round(res["dense_ffn"], 2), "dense_ffn_weight_gbs": round(wbytes / (res["dense_ffn"] * 1e-6) / 1e9, 1),
            "dense_ffn_tops": round(flops / (res["dense_ffn"] * 1e-6) / 1e12, 2),
            "mmq_2048x6144_us": round(res["mmq"], 2),
            "mmq_tops": round(2 * T * FD * H / (res["mmq"] * 1e-6) / 1e12, 2)}


def main() -> int:
    ap = argparse.ArgumentParser(description=__doc__.split("\n")[0])
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=64)
    ap.add_argument("--warmup", type=int, default=8)
    ap.add_argument("--layers", type=int, default=16, help="resident copies of the config-0 layer (MALL defeat)")
    ap.add_argument("--no-cpu", action="store_true", help="skip the CPU baseline")
    ap.add_argument("--no-extra", action="store_true", help="skip configs 1-3")
    ap.add_argument("--profile-stages", type=int, default=0,
                    help="profiling mode for rocprofv3: only N back-to-back rounds of the three kernels + a 256 MiB copy")
    ap.add_argument("--profile-prefill", type=int, default=0,
                    help="profiling mode for rocprofv3: only N rounds of config-4 prefill over 2 layers + a 256 MiB copy")
    ap.add_argument("--profile-dense", type=int, default=0,
                    help="profiling mode for rocprofv3: only N rounds of the dense Q8_0 FFN prefill and Q8_0 mmq")
    args = ap.parse_args()
    if args.gpus != 1:
        print(f"bench.py: this build measures one GPU only (asked for --gpus {args.gpus}); the MoE layer would shard "
              f"experts across GPUs (one expert range per GPU, partial outputs summed by an all-reduce), which is not built "
              f"or measured here.", file=sys.stderr)
        return 2

    import torch

    from flintnsteel_amd import synth
    warnings.filterwarnings("ignore", message="The CUDA Graph is empty")
    torch.cuda.init()
    dev = torch.cuda.get_device_properties(0)
    log(f"device {dev.name} {dev.gcnArchName if hasattr(dev, 'gcnArchName') else ''} CUs {dev.multi_processor_count}")

    if args.profile_dense:
        r = run_dense_q8_0(torch, n_layers=2, replays=args.profile_dense)
        a = torch.empty(64 << 20, device="cuda")
        b = torch.empty_like(a)
        b.copy_(a)  # 256 MiB read + 256 MiB write: FETCH_SIZE / WRITE_SIZE calibration
        torch.cuda.synchronize()
        log(f"profile dense done: {r}")
        return 0

    if args.profile_prefill:
        r = run_prefill(torch, synth, n_layers=2, replays=args.profile_prefill)
        a = torch.empty(64 << 20, device="cuda")
        b = torch.empty_like(a)
        b.copy_(a)  # 256 MiB read + 256 MiB write: FETCH_SIZE / WRITE_SIZE calibration
        torch.cuda.synchronize()
        log(f"profile prefill done: {r}")
        return 0

    L = args.layers
    t0 = time.time()
    layers = build_layers(synth, L, Q4_K, Q4_K, 0)
    torch.cuda.synchronize()
    log(f"built {L} config-0 layers in {time.time() - t0:.1f} s")
    steps_per_graph = max(d for d in range(1, 9) if args.steps % d == 0)
    xs = make_xs(synth, torch, 1, steps_per_graph, L, 1000)
    outs = [torch.empty(1, H, device="cuda") for _ in layers]
    wss = [layer.workspace(1) for layer in layers]

    if args.profile_stages:
        for r in range(args.profile_stages):
            for k in range(3):
                for l, layer in enumerate(layers):
                    layer.stage(k, xs[r % steps_per_graph, l], outs[l], wss[l])
        a = torch.empty(64 << 20, device="cuda")
        b = torch.empty_like(a)
        b.copy_(a)  # 256 MiB read + 256 MiB write: FETCH_SIZE / WRITE_SIZE calibration
        torch.cuda.synchronize()
        log("profile rounds done")
        return 0

    g = capture(torch, layers, xs, outs, wss, steps_per_graph)
    replays = args.steps // steps_per_graph
    ms_replay = time_graph(torch, g, replays, max(1, args.warmup // steps_per_graph))
    ms_per_step = ms_replay / steps_per_graph
    us_layer = ms_per_step * 1e3 / L
    log(f"config 0: {us_layer:.2f} us/layer ({ms_per_step:.3f} ms per step of {L} layers)")
    spread = replay_spread(torch, g, 64, steps_per_graph * L)
    log(f"config 0, 64 replays timed one by one (us/layer): median {spread['median']} p10 {spread['p10']} "
        f"p90 {spread['p90']}")
    st = stage_times(torch, layers, xs, outs, wss, reps=16)
    log(f"per-kernel (us): router {st[0]:.2f}  gate/up {st[1]:.2f}  down+combine {st[2]:.2f}")
    ex_bytes = K_TOP * expert_bytes(Q4_K, Q4_K)
    ex_us = st[1] + st[2]  # the fused kernel is stage 1; stage 2 is then empty (its graph replay costs ~0.3 us)
    achieved = ex_bytes / (st[1] * 1e-6) / 1e9
    traffic = read_traffic()
    roofline = {"bound": "hbm", "kernel": "k_layer_fused (routing, gate/up + SwiGLU, Q8_1 of act, down, combine)",
                "achieved": round(achieved, 1), "peak": PEAK_GBS, "unit": "GB/s", "frac": round(achieved / PEAK_GBS, 4),
                "traffic": traffic["bytes"] if traffic else None, "algorithmic_bytes": ex_bytes,
                "avg_us": round(st[1], 3), "expert_stages_us": round(ex_us, 3)}
    layer_gbs = layer_bytes(Q4_K, Q4_K) / (us_layer * 1e-6) / 1e9
    del g

    extra = {"config0_layer_hbm_gbs": round(layer_gbs, 1), "config0_stage_us": [round(v, 3) for v in st],
             "config0_replays_us_per_layer": spread}
    if not args.no_extra:
        extra["config0_dropin_seven_calls"] = run_dropin(torch, layers)
        log(f"config0 through the seven drop-in calls: {extra['config0_dropin_seven_calls']}")
        for name, gu, dn in (("config1_q3k_q5k", Q3_K, Q5_K),):
            _, ms, _ = run_stack(torch, synth, gu, dn, L, 1, 16, 4, 100)
            us = ms * 1e3 / L
            extra[name] = {"us_per_layer": round(us, 3),
                           "hbm_gbs": round(layer_bytes(gu, dn) / (us * 1e-6) / 1e9, 1)}
            log(f"{name}: {us:.2f} us/layer")
        _, ms, distinct = run_stack(torch, synth, Q4_K, Q4_K, L, 4, 16, 4, 200)
        us = ms * 1e3 / L
        extra["config2_verify4"] = {"us_per_layer_step": round(us, 3), "distinct_experts": distinct,
                                    "hbm_gbs": round(layer_bytes(Q4_K, Q4_K, distinct) / (us * 1e-6) / 1e9, 1)}
        log(f"config2 (4-token verify): {us:.2f} us/layer, {distinct:.1f} distinct experts")
        del layers
        torch.cuda.empty_cache()
        t1 = time.time()
        stack, ms, _ = run_stack(torch, synth, Q4_K, Q6_K, 48, 1, 256, 8, 300, steps_per_graph=4)
        tok_s = 1e3 / ms
        per_tok = 48 * layer_bytes(Q4_K, Q6_K)
        extra["config3_stack48"] = {"tokens_per_s": round(tok_s, 1), "us_per_layer": round(ms * 1e3 / 48, 3),
                                    "hbm_gbs": round(per_tok * tok_s / 1e9, 1), "build_s": round(time.time() - t1, 1)}
        log(f"config3 (48 layers): {tok_s:.1f} tok/s")
        layers = stack[:1]
        del stack
        torch.cuda.empty_cache()
        extra["config4_prefill512"] = run_prefill(torch, synth)
        log(f"config4 (prefill 512): {extra['config4_prefill512']}")
        torch.cuda.empty_cache()
        extra["flint_block_decode"] = run_flint(torch, synth)
        log(f"flint block (decode): {extra['flint_block_decode']}")
        torch.cuda.empty_cache()
        for name, gu, dn in (("flint_block_iq3xxs_iq4xs", IQ3_XXS, IQ4_XS), ("flint_block_iq3s_iq4xs", IQ3_S, IQ4_XS)):
            extra[name] = run_flint(torch, synth, gu=gu, dn=dn)
            log(f"{name} (decode): {extra[name]}")
            torch.cuda.empty_cache()
        extra["dense_q8_0_prefill512"] = run_dense_q8_0(torch)
        log(f"dense Q8_0 prefill 512: {extra['dense_q8_0_prefill512']}")
    cpu = None
    if not args.no_cpu:
        if args.no_extra:
            cpu_layer = layers[0]
        else:
            cpu_layer = build_layers(synth, 1, Q4_K, Q4_K, 0)[0]
        cpu = cpu_baseline(torch, cpu_layer)
        log(f"cpu baseline: {cpu['value']:.1f} us/layer on {cpu['cores']} threads")

    line = {
        "metric": "us/token per MoE layer + achieved HBM GB/s (batch 1, Q4_K experts)",
        "value": round(us_layer, 3), "unit": "us/layer", "n_gpus": 1, "steps": args.steps, "warmup": args.warmup,
        "ms_per_step": round(ms_per_step, 4), "higher_is_better": False, "scaling": "weak", "vs_baseline": None,
        "dtype": "int8xK-quant dot, fp32 accumulate", "data": "synthetic (seeded Philox N(0,1) / N(0,0.02) on device)",
        "config": {"workload": "config 0: 1 MoE FFN layer, decode batch 1, hidden 2048, 128 experts top-8 softmax, "
                               f"inter 768, Q4_K gate/up/down, fp32 router; {L} resident layer copies per step",
                   "layers_per_step": L, "hbm_bytes_per_layer": layer_bytes(Q4_K, Q4_K),
                   "achieved_layer_hbm_gbs": round(layer_gbs, 1)},
        "roofline": roofline,
        "cpu_baseline": cpu,
        "extra": extra,
    }
    print(json.dumps(line), flush=True)
    return 0


if __name__ == "__main__":
    sys.exit(main())
