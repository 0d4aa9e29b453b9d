"""The grouped GEMM's int8 form (types whose scales change every 32 columns) through the dense FFN block's prefill:
every type, at the edges of its 32-row tiles and 64-row groups, both grid orders (few and many weight row blocks) and a
split K range, against the float64 chain of dequantised weights and activations.

Bars: act is re-quantised to 8 bits inside the block, so a code whose quotient lies on a rounding boundary may move one
step where two fp32 sums differ in their last bits (about one code in 10^4, so at most two in a row of 1024). One step
moves an output by at most max|act| / 127 * max|w_down|: two such steps plus 1e-5 of the largest output (32-bit sums, and
the residual's rounding) bound every element; the relative L2 bound is that of the independent chains in
tests/helpers.py."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import oracle as orc
from tests.helpers import CHAIN_L2_TOL, gaussian, rel_l2
from tests.iq_data import random_blocks, register_grids, register_grids_in_library

pytestmark = pytest.mark.gpu

TYPES = [orc.Q8_0, orc.Q4_K, orc.Q5_K, orc.IQ4_XS, orc.IQ3_XXS, orc.IQ3_S]


@pytest.fixture(scope="module")
def ops():
    from flintnsteel_amd import ops as o
    register_grids_in_library(register_grids())
    return o


def weights(qtype: int, nrows: int, ncols: int, seed: int) -> np.ndarray:
    if qtype in (orc.IQ4_XS, orc.IQ3_XXS, orc.IQ3_S):
        return random_blocks(qtype, nrows, ncols, seed)
    w = gaussian(np.random.default_rng(seed), (nrows, ncols), 0.02)
    w[:, 256:512] *= 3e-4   # small sub-block scales
    w[1, :256] = 0.0        # a block with d = 0
    return orc.quantize(qtype, w)


def dequant(qtype: int, w: np.ndarray, nrows: int, ncols: int) -> np.ndarray:
    return np.asarray(orc.dequantize(qtype, w.reshape(nrows, -1), ncols), np.float64).reshape(nrows, ncols)


# (T <= 130: every launch takes groups of 32 rows, 1 to 5 of them. 449: 64-row groups, the last of one row; gate/up with 34
# weight row blocks over the XCDs, not a multiple of 8; down with its columns split in four.)
SHAPES = [(1, 512, 768), (33, 512, 768), (65, 512, 768), (130, 2048, 1024)]


@pytest.mark.parametrize("qtype,T,H,F", [(t, *s) for t in TYPES for s in SHAPES] +
                         [(t, 449, 2048, 4352) for t in (orc.Q8_0, orc.Q4_K, orc.IQ4_XS)])
def test_dense_prefill_int8(ops, qtype, T, H, F):
    rng = np.random.default_rng(T + H)
    g, u, d = weights(qtype, F, H, 1), weights(qtype, F, H, 2), weights(qtype, H, F, 3)
    x = gaussian(rng, (T, H))
    x[0, :64] = 0.0  # blocks with amax = 0
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()  # noqa: E731
    ffn = ops.DenseFfn(dev(g), dev(u), dev(d), qtype, qtype, qtype, H, F)
    got = ffn(dev(x), prefill=True)
    torch.cuda.synchronize()
    xq = orc.dequantize_q8_1(orc.quantize_q8_1(x), H)
    gate, up = xq @ dequant(qtype, g, F, H).T, xq @ dequant(qtype, u, F, H).T
    act = (up * gate / (1 + np.exp(-gate))).astype(np.float32)
    down = dequant(qtype, d, H, F)
    ref = orc.dequantize_q8_1(orc.quantize_q8_1(act), F) @ down.T
    err = np.abs(got.cpu().numpy().astype(np.float64) - x - ref)
    bound = 2 * np.abs(act).max() / 127 * np.abs(down).max() + 1e-5 * np.abs(ref).max()
    l2 = rel_l2(got.cpu().numpy().astype(np.float64) - x, ref)
    assert err.max() <= bound and l2 <= CHAIN_L2_TOL, f"max err {err.max():.3e} (bound {bound:.3e}), rel L2 {l2:.3e}"


@pytest.mark.parametrize("gu,down", [(orc.Q4_K, orc.Q4_K), (orc.Q4_K, orc.Q6_K), (orc.Q5_K, orc.IQ4_XS),
                                     (orc.IQ3_XXS, orc.IQ3_S), (orc.Q8_0, orc.Q8_0), (orc.Q6_K, orc.Q5_K),
                                     (orc.Q3_K, orc.Q4_K), (orc.Q4_K, orc.Q3_K)])
@pytest.mark.parametrize("E,counts", [(8, (1, 2, 7, 8, 9)), (8, (32, 33, 40, 64, 72)),
                                      (256, (1, 2, 7, 8, 9, 32, 33, 40, 64, 72)), (256, (15, 16, 17, 24, 31, 48, 80, 81))])
def test_prefill_group_sizes(ops, gu, down, E, counts):
    """The prefill layer with experts of exactly these loads (a router that picks each token's expert): one tile, two
    tiles and their remainders, in one launch or two, gate/up and down in either form of the GEMM (8 experts: at most
    256 gate/up workgroups, the split form; 256 experts: the int8 form for the types that have it)."""
    H, F = 512, 256
    owner = np.concatenate([np.full(n, e) for e, n in enumerate(counts)])
    T = owner.size
    rng = np.random.default_rng(T + gu)
    router = np.zeros((E, H), np.float32)
    x = gaussian(rng, (T, H))
    for e in range(len(counts)):  # the first columns carry the choice
        router[e, e] = 50.0
    x[:, :len(counts)] = 0.0
    x[np.arange(T), owner] = 4.0
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()  # noqa: E731
    mats = []
    for k, (t, r, c) in enumerate([(gu, F, H), (gu, F, H), (down, H, F)]):
        used = [weights(t, r, c, 100 * k + e).reshape(-1) for e in range(len(counts))]
        mats.append(np.stack([used[e % len(used)] for e in range(E)]))
    slots = ops.ExpertSlots.from_tensors(*(torch.from_numpy(m) for m in mats))
    layer = ops.MoeLayer(dev(router), slots, gu, down, H, F, 1)
    pre = ops.MoePrefill(layer)
    ws, xd = pre.workspace(T), dev(x)
    out = pre(xd, ws=ws).cpu().numpy().astype(np.float64)
    tr = pre.trace(ws, T)
    assert np.array_equal(tr["ids"].cpu().numpy()[:, 0], owner)
    xq = orc.dequantize_q8_1(orc.quantize_q8_1(x), H)
    w = tr["w"].cpu().numpy().astype(np.float64)
    tight = []  # rows without a moved code: all but about one in forty (256 codes a row, one in 10^4 moves)
    for e in range(len(counts)):
        t = np.flatnonzero(owner == e)
        g, u, d = (dequant(ty, m[e], r, c) for m, (ty, r, c) in zip(mats, [(gu, F, H), (gu, F, H), (down, H, F)]))
        gate, up = xq[t] @ g.T, xq[t] @ u.T
        act = (up * gate / (1 + np.exp(-gate))).astype(np.float32)
        ref = orc.dequantize_q8_1(orc.quantize_q8_1(act), F) @ d.T * w[t]
        err = np.abs(out[t] - ref).max(axis=1)
        bound = 2 * np.abs(act).max() / 127 * np.abs(d).max() + 1e-5 * np.abs(ref).max()
        assert err.max() <= bound, f"expert {e} ({t.size} rows): {err.max():.3e} > {bound:.3e}"
        tight.append(err <= 1e-5 * np.abs(ref).max())
    assert np.concatenate(tight).mean() >= 0.8


@pytest.mark.parametrize("gu,down,guard,shared", [
    (orc.Q4_K, orc.Q4_K, False, None), (orc.Q4_K, orc.Q3_K, False, None), (orc.Q3_K, orc.Q4_K, False, None),
    (orc.Q4_K, orc.Q5_K, False, None), (orc.Q5_K, orc.Q6_K, True, None), (orc.IQ3_XXS, orc.IQ4_XS, False, None),
    (orc.IQ3_S, orc.IQ4_XS, True, (orc.IQ3_S, orc.IQ4_XS)), (orc.Q8_0, orc.Q8_0, False, (orc.Q8_0, orc.Q8_0)),
    (orc.Q4_K, orc.Q4_K, False, (orc.Q6_K, orc.Q4_K)), (orc.Q4_K, orc.Q5_K, False, (orc.Q4_K, orc.Q5_K))])
def test_prefill_token_alone_and_in_a_chunk(ops, gu, down, guard, shared):
    """A token's result does not depend on the call's length: 1000 tokens (64-row groups), their first 150 (64-row groups as
    two items where that fills no more than the GPU), 33 of them and single tokens give the same bits, for every type of
    the int8 form, one launch and two, each pair of image forms, and a shared expert of the routed types or others."""
    E, K, H, F, T = 16, 4, 1024, 768, 1000
    rng = np.random.default_rng(gu * 100 + down)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()  # noqa: E731
    mats = [np.stack([weights(t, r, c, 10 * k + e % 4).reshape(-1) for e in range(E)])
            for k, (t, r, c) in enumerate([(gu, F, H), (gu, F, H), (down, H, F)])]
    slots = ops.ExpertSlots.from_tensors(*(torch.from_numpy(m) for m in mats))
    shexp = None
    if shared:
        g, d = shared
        shexp = {"gate": dev(weights(g, 512, H, 91)), "up": dev(weights(g, 512, H, 92)), "down": dev(weights(d, H, 512, 93)),
                 "inter": 512, "gu_type": g, "down_type": d}
    layer = ops.MoeLayer(dev(gaussian(rng, (E, H), 0.05)), slots, gu, down, H, F, K, guard=guard, shexp=shexp,
                         ffn_norm=dev(gaussian(rng, (H,), 1.0)))
    pre = ops.MoePrefill(layer)
    x = dev(gaussian(rng, (T, H)))
    whole = pre(x).cpu().numpy()
    assert np.isfinite(whole).all() and np.abs(whole).max() > 0
    for t0, n in ((0, 150), (400, 33), (0, 1), (T - 1, 1)):
        part = pre(x[t0:t0 + n].contiguous()).cpu().numpy()
        assert np.array_equal(part, whole[t0:t0 + n]), f"{n} tokens from {t0}"


@pytest.mark.parametrize("T", [5, 70])
def test_prefill_split_x_int8_act(ops, T):
    """Q4_K experts beside a Q6_K shared gate/up: x in the split form, act in the int8 form, gate/up and down in one launch.
    Against the decode path of the same layer (other sums of the same products: the chain bounds)."""
    from tests.helpers import assert_close_chain
    E, K, H, F = 16, 4, 512, 768
    rng = np.random.default_rng(40 + T)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()  # noqa: E731
    mats = [np.stack([weights(orc.Q4_K, r, c, 10 * k + e).reshape(-1) for e in range(E)])
            for k, (r, c) in enumerate([(F, H), (F, H), (H, F)])]
    shexp = {"gate": dev(weights(orc.Q6_K, 256, H, 91)), "up": dev(weights(orc.Q6_K, 256, H, 92)),
             "down": dev(weights(orc.Q4_K, H, 256, 93)), "inter": 256, "gu_type": orc.Q6_K, "down_type": orc.Q4_K}
    layer = ops.MoeLayer(dev(gaussian(rng, (E, H), 0.05)), ops.ExpertSlots.from_tensors(*(torch.from_numpy(m) for m in mats)),
                         orc.Q4_K, orc.Q4_K, H, F, K, shexp=shexp)
    pre, x = ops.MoePrefill(layer), dev(gaussian(rng, (T, H)))
    ws, ws1 = pre.workspace(T), layer.workspace(1)
    out = pre(x, ws=ws).cpu().numpy()
    assert pre.status(ws, T) == 0
    one = np.stack([layer(x[t:t + 1].contiguous(), ws=ws1).cpu().numpy()[0] for t in range(T)])
    assert_close_chain(out, one, f"{T} tokens")


@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("H,E,T", [(256, 256, 993), (576 * 4, 250, 1025), (512, 33, 4097)])
def test_prefill_router_tiles(ops, bf16, H, E, T):
    """The router GEMM's 32 x 32 tiles (at least 256 of them) give every token the logits of the 16 x 16 tiles, which a
    call of fewer tokens takes, bit for bit: ragged token and expert counts, fewer column chunks than waves and more."""
    rng = np.random.default_rng(T)
    F = 256
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()  # noqa: E731
    router = dev(gaussian(rng, (E, H)))
    x = dev(gaussian(rng, (T, H)))
    mats = [np.repeat(weights(orc.Q4_K, r, c, k).reshape(1, -1), E, axis=0)
            for k, (r, c) in enumerate([(F, H), (F, H), (H, F)])]
    slots = ops.ExpertSlots.from_tensors(*(torch.from_numpy(m) for m in mats))
    layer = ops.MoeLayer(router.bfloat16() if bf16 else router, slots, orc.Q4_K, orc.Q4_K, H, F, 1)
    pre = ops.MoePrefill(layer)

    def logits(xs):
        ws = pre.workspace(xs.shape[0])
        pre(xs, ws=ws)
        return pre.trace(ws, xs.shape[0])["logits"].cpu().numpy()

    whole = logits(x)
    w64, x64 = (t.bfloat16().double() if bf16 else t.double() for t in (router, x))
    ref = (x64 @ w64.T).cpu().numpy()
    assert np.abs(whole - ref).max() <= 1e-5 * np.abs(ref).max()  # fp32 sums of at most 2304 products
    step = 300
    for t in range(0, T, step):
        assert np.array_equal(logits(x[t:t + step].contiguous()), whole[t:t + step]), f"tokens from {t}"
