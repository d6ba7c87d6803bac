"""GPU parity of the grouped-expert prefill (mnemo_moe_prefill).

Reference for the added delta out - out0: the reference's expert chain applied token by token
(src/forward.c:876-893 per expert, src/forward.c:1783-1830 per token) in the Q8_1 GEMM
semantics -- Oracle.moe_prefill (fp64, C) at test sizes and its torch restatement
(tests/torch_ref.py, fp64 on the GPU, pinned against the oracle on the CPU) at the benchmark
cfg5 shape.  Bar: relative L2 <= 1e-3.  The GEMMs sum every sub-block exactly,
so the remaining difference is the SwiGLU's exp rounding moving a requantized value by one
step now and then (measured ~1e-6); a wrong expert, slot or weight is an O(1) error.
The per-expert composition of the plain entry points is a second reference at the same bar.
Routing edge cases: experts with no tokens, an expert spanning several 128-row tiles, dropped
slots (id -1 or >= n_experts), one token.  The cfg5 shape is also checked for bitwise
run-to-run determinism."""
import numpy as np
import pytest
import torch

from mnemocuda_amd import synth
from tests.conftest import rel_l2
from tests import torch_ref
from tests.gpu_util import case, dev, host

pytestmark = pytest.mark.gpu
TOL = 1e-3
TOL_ORACLE = 1e-3


def _run(gpu, table, lay, down_type, x, idx, w, T, H, EFF, E, k, out0):
    stride, g_off, u_off, d_off = lay
    ws = torch.empty(gpu.ops.moe_prefill_workspace_bytes(T, H, EFF, E, k), dtype=torch.uint8, device="cuda")
    out = out0.clone()
    gpu.ops.moe_prefill(table, stride, g_off, u_off, d_off, down_type, x, idx, w, T, H, EFF, E, k, ws, out)
    return out


def _compose_plain(gpu, table, lay, DT, x, idx, w, T, H, EFF, out0):
    """out0 + sum_slot w * down(silu(gate x) * up x) through the plain GPU entry points."""
    stride, g_off, u_off, d_off = lay
    ops = gpu.ops
    xq = torch.empty(T * (H // 128) * 144, dtype=torch.uint8, device="cuda")
    ops.quantize_q8_1(x, xq, H, T)
    xq = xq.view(T, -1)
    ref = out0.clone().double().view(T, H)
    for e in np.unique(idx):
        tok, slot = np.nonzero(idx == e)
        if e < 0 or e * stride >= table.numel():
            continue
        n = tok.size
        a = xq[torch.from_numpy(tok).cuda()].contiguous()
        base = int(e) * stride
        g = torch.empty(n, EFF, device="cuda")
        u = torch.empty(n, EFF, device="cuda")
        ops.gemm(table[base + g_off: base + u_off], 12, a, g, EFF, H, n)
        ops.gemm(table[base + u_off: base + d_off], 12, a, u, EFF, H, n)
        act = (g / (1 + torch.exp(-g)) * u).contiguous()
        aq = torch.empty(n * (EFF // 128) * 144, dtype=torch.uint8, device="cuda")
        ops.quantize_q8_1(act, aq, EFF, n)
        d = torch.empty(n, H, device="cuda")
        ops.gemm(table[base + d_off: base + stride], DT, aq, d, H, EFF, n)
        ref.index_add_(0, torch.from_numpy(tok).cuda(),
                       d.double() * torch.from_numpy(w[tok, slot]).cuda()[:, None].double())
    return ref


@pytest.mark.parametrize("T,H,EFF,E,k,down_type,skew", [
    (64, 512, 256, 16, 4, 14, 1.1),
    (300, 256, 512, 4, 2, 12, 3.0),    # expert 0 spans several tiles
    (1, 256, 256, 8, 8, 14, 1.1),      # one token, every expert once
    (37, 768, 256, 32, 3, 14, 0.0),    # most experts empty or single-row
    # experts of one ragged tile, of a full one and a ragged one
    (130, 256, 256, 2, 1, 14, 0.0),
    (200, 512, 256, 5, 2, 12, 0.5),
    # K in whole 1024-value windows, one to five of them
    (48, 1024, 1024, 4, 2, 12, 0.5),
    (24, 2048, 256, 3, 2, 14, 1.1),
    (70, 3072, 256, 2, 1, 14, 0.0),
    (16, 5120, 1024, 2, 1, 12, 0.0),
    # Q6_K down rows of 3 blocks (630 B): rows and blocks alternate between 4-byte aligned
    # and 2 bytes past (the copies' window offsets)
    (40, 512, 768, 4, 2, 14, 0.5),
])
def test_moe_prefill_vs_oracle(gpu, oracle, T, H, EFF, E, k, down_type, skew):
    rng = np.random.default_rng(T * 1000 + E)
    table = synth.expert_table(rng, E, H, EFF, down_type)
    lay = synth.expert_layout(H, EFF, down_type)
    idx, w = synth.zipf_routing(rng, T, E, k, s=skew)
    if T > 4:  # dropped slots: an unfilled top-k slot (-1) and an id past the table
        idx[1, -1] = -1
        idx[3, 0] = E + 5
    x = rng.standard_normal((T, H)).astype(np.float32)
    if down_type == 12:
        # a Q4_K down projection takes its min term from the Q8_1 ds field (d8 * sum of the
        # SwiGLU values, an f16): with the benchmark weight distribution and x ~ N(0, 1) the
        # SwiGLU values reach ~1e3 and ds overflows to inf, in the reference's formula as here
        x *= np.float32(0.05)
    out0 = rng.standard_normal((T, H)).astype(np.float32)
    case(f"moe_prefill T={T} H={H} EFF={EFF} E={E} k={k} down={down_type}")
    out = _run(gpu, dev(table), lay, down_type, dev(x), dev(idx), dev(w), T, H, EFF, E, k, dev(out0))
    got_delta = host(out).astype(np.float64).reshape(T, H) - out0
    comp = host(_compose_plain(gpu, dev(table), lay, down_type, dev(x), idx, w, T, H, EFF, dev(out0))) - out0
    ref_delta = oracle.moe_prefill(table, *lay, down_type, x, idx, w, H, EFF, E)
    err_c, err_o = rel_l2(got_delta, comp), rel_l2(got_delta, ref_delta)
    print(f"rel_l2 vs plain composition={err_c:.2e} vs oracle={err_o:.2e} "
          f"(plain composition vs oracle {rel_l2(comp, ref_delta):.2e})")
    assert err_c < TOL
    assert err_o < TOL_ORACLE


# Tiles of every width: 1 .. 8 columns of 16 rows (5 and 7 run as 6 and 8), one row over and under,
# second tiles, an empty expert, a tile count that is no multiple of 8; K = 1280 ends a 1024-value
# window early.  9000 pairs: more than one batch of loads per wave in the routing, with a k
# that does not divide 64.
@pytest.mark.parametrize("counts,H,EFF,k,down_type", [
    ((1, 16, 17, 48, 0, 49, 64, 65, 96, 97, 112, 113, 128, 129, 200), 1280, 768, 1, 12),
    ((1, 16, 17, 48, 0, 49, 64, 65, 96, 97, 112, 113, 128, 129, 200), 1280, 768, 1, 14),
    ((375,) * 24, 256, 256, 6, 14),
])
def test_moe_prefill_tile_widths(gpu, counts, H, EFF, k, down_type):
    E = len(counts)
    rng = np.random.default_rng(sum(counts) + H)
    table = synth.expert_table(rng, E, H, EFF, down_type)
    lay = synth.expert_layout(H, EFF, down_type)
    if k == 1:
        idx = rng.permutation(np.repeat(np.arange(E, dtype=np.int32), counts)).reshape(-1, 1)
    else:  # every token k different experts
        T = sum(counts) // k
        idx = ((np.arange(T)[:, None] * 5 + np.arange(k)[None, :] * 3) % E).astype(np.int32)
    T = idx.shape[0]
    w = rng.random((T, k)).astype(np.float32)
    x = (0.05 * rng.standard_normal((T, H))).astype(np.float32)
    out0 = np.zeros((T, H), dtype=np.float32)
    case(f"moe_prefill widths T={T} H={H} EFF={EFF} E={E} k={k} down={down_type}")
    args = (gpu, dev(table), lay, down_type, dev(x), dev(idx), dev(w), T, H, EFF, E, k, dev(out0))
    got = host(_run(*args))
    assert np.array_equal(got, host(_run(*args)))
    comp = host(_compose_plain(gpu, dev(table), lay, down_type, dev(x), idx, w, T, H, EFF, dev(out0)))
    got, comp = got.reshape(T, H).astype(np.float64), comp.reshape(T, H)
    assert rel_l2(got, comp) < TOL
    # no token is lost among the others: each within ten times the bar
    err = np.linalg.norm(got - comp, axis=1) / np.linalg.norm(comp, axis=1)
    assert err.max() < 10 * TOL


@pytest.mark.parametrize("H", [512, 2048])
def test_moe_prefill_zero_d_blocks(gpu, oracle, H):
    """Gate/up Q4_K blocks with d = 0 (dmin kept, so only the min term survives), scattered
    and over whole rows, with K below one 1024-value window and K in two whole windows."""
    T, EFF, E, k, DT = 96, 256, 4, 2, 14
    rng = np.random.default_rng(H + 7)
    table = synth.expert_table(rng, E, H, EFF, DT)
    lay = synth.expert_layout(H, EFF, DT)
    stride, _, up_off, down_off = lay
    nb = H // 256
    t = table.reshape(E, stride)
    gu = t[:, :down_off].reshape(E, 2 * EFF * nb, 144)
    gu[:, :, 0:2][rng.random((E, 2 * EFF * nb)) < 0.15] = 0
    rows = gu.reshape(E, 2 * EFF, nb, 144)
    rows[:, 3, :, 0:2] = 0          # every block of gate row 3
    rows[:, EFF + 10, :, 0:2] = 0   # and of up row 10
    assert np.shares_memory(rows, t)
    table = t.reshape(-1)
    idx, w = synth.zipf_routing(rng, T, E, k, s=0.5)
    x = rng.standard_normal((T, H)).astype(np.float32)
    out0 = rng.standard_normal((T, H)).astype(np.float32)
    case(f"moe_prefill zero-d blocks H={H}")
    out = _run(gpu, dev(table), lay, DT, dev(x), dev(idx), dev(w), T, H, EFF, E, k, dev(out0))
    got_delta = host(out).astype(np.float64).reshape(T, H) - out0
    ref_delta = oracle.moe_prefill(table, *lay, DT, x, idx, w, H, EFF, E)
    err = rel_l2(got_delta, ref_delta)
    print(f"rel_l2 vs oracle={err:.2e}")
    assert err < TOL_ORACLE


def test_moe_prefill_bad_args(gpu):
    T, H, EFF, E, k = 4, 256, 256, 4, 2
    x = torch.zeros(T * H, device="cuda")
    idx = torch.zeros(T * k, dtype=torch.int32, device="cuda")
    w = torch.zeros(T * k, device="cuda")
    out = torch.zeros(T * H, device="cuda")
    table = torch.zeros(E * synth.expert_layout(H, EFF, 14)[0], dtype=torch.uint8, device="cuda")
    lay = synth.expert_layout(H, EFF, 14)
    small = torch.zeros(64, dtype=torch.uint8, device="cuda")
    with pytest.raises(gpu.MnemoError, match="workspace"):
        gpu.ops.moe_prefill(table, *lay, 14, x, idx, w, T, H, EFF, E, k, small, out)
    ws = torch.zeros(gpu.ops.moe_prefill_workspace_bytes(T, H, EFF, E, k), dtype=torch.uint8, device="cuda")
    with pytest.raises(gpu.MnemoError, match="down type"):
        gpu.ops.moe_prefill(table, *lay, 3, x, idx, w, T, H, EFF, E, k, ws, out)
    # weight blocks are copied by DMA from 4-byte aligned addresses
    big = torch.zeros(table.numel() + 16, dtype=torch.uint8, device="cuda")
    with pytest.raises(gpu.MnemoError, match="4-byte aligned"):
        gpu.ops.moe_prefill(big[2:], *lay, 14, x, idx, w, T, H, EFF, E, k, ws, out)
    stride, g_off, u_off, d_off = lay
    with pytest.raises(gpu.MnemoError, match="4-byte aligned"):
        gpu.ops.moe_prefill(big, stride, g_off, u_off, d_off + 2, 14, x, idx, w, T, H, EFF, E, k, ws, out)


def test_moe_prefill_baseline_shape(gpu):
    """512 tokens, hidden 4096, eff 1536, 128 experts, top-8 Zipf(1.1), Q6_K down."""
    T, H, EFF, E, k, DT = 512, 4096, 1536, 128, 8, 14
    rng = np.random.default_rng(5)
    idx, w = synth.zipf_routing(rng, T, E, k)
    gen = torch.Generator(device="cuda").manual_seed(5)
    case("moe_prefill baseline shape: building expert table")
    table = synth.expert_table_torch(gen, E, H, EFF, DT, "cuda")
    lay = synth.expert_layout(H, EFF, DT)
    stride, g_off, u_off, d_off = lay
    x = torch.randn(T, H, device="cuda", generator=gen)
    out0 = torch.randn(T, H, device="cuda", generator=gen)
    idx_d, w_d = dev(idx), dev(w)
    case("moe_prefill baseline shape: grouped run x2")
    out = _run(gpu, table, lay, DT, x, idx_d, w_d, T, H, EFF, E, k, out0)
    out_b = _run(gpu, table, lay, DT, x, idx_d, w_d, T, H, EFF, E, k, out0)
    assert torch.equal(out, out_b), "grouped prefill is not deterministic"

    case("moe_prefill baseline shape: fp64 per-token chain (torch restatement of the oracle)")

    def quantize(a):
        q = torch.empty(a.shape[0] * (a.shape[1] // 128) * 144, dtype=torch.uint8, device="cuda")
        gpu.ops.quantize_q8_1(a, q, a.shape[1], a.shape[0])
        return q.view(a.shape[0], -1)

    ref = torch_ref.moe_prefill(table, *lay, DT, x, idx, w, H, EFF, quantize=quantize)
    got = host(out).astype(np.float64) - host(out0).astype(np.float64)
    err_o = rel_l2(got, host(ref))
    case("moe_prefill baseline shape: per-expert composition of the plain GEMMs")
    comp = _compose_plain(gpu, table, lay, DT, x, idx, w, T, H, EFF, out0)
    err_c = rel_l2(got, host(comp) - host(out0))
    print(f"rel_l2 vs fp64 chain={err_o:.2e} vs plain composition={err_c:.2e}")
    assert err_o < TOL_ORACLE
    assert err_c < TOL


# ------------------------------------------------------------------ decode (one token)
def _decode_ref(oracle, table, lay, DT, router, x, H, EFF, E, k):
    """fp64 oracle chain: router -> top-k -> sum_slot w * down(silu(gate x) * up x)."""
    stride, g_off, u_off, d_off = lay
    logits = oracle.matvec_f32(router, x, E, H)
    idx, w = oracle.topk_softmax(logits.astype(np.float32), k)
    delta = np.zeros(H)
    for e, wt in zip(idx, w):
        base = int(e) * stride
        g = oracle.gemv(12, table[base + g_off: base + u_off], x, EFF, H)
        u = oracle.gemv(12, table[base + u_off: base + d_off], x, EFF, H)
        act = oracle.swiglu(g.astype(np.float32), u.astype(np.float32))
        delta += float(wt) * oracle.gemv(DT, table[base + d_off: base + stride], act, H, EFF)
    return logits, idx, w, delta


def _routable(rng, E, H, k):
    """router weights and x whose top-k has a clear margin (so the id set is exact in fp32)"""
    while True:
        router = (rng.standard_normal((E, H)) / np.sqrt(H)).astype(np.float32)
        x = rng.standard_normal(H).astype(np.float32)
        z = np.sort(router.astype(np.float64) @ x)[::-1]
        if k == E or z[k - 1] - z[k] > 1e-3:
            return router, x


@pytest.mark.parametrize("H,EFF,E,k,DT", [(512, 256, 16, 4, 14), (1024, 512, 8, 8, 12), (4096, 1536, 24, 8, 14),
                                        (1024, 768, 24, 12, 14), (2048, 2560, 16, 6, 12), (4608, 512, 8, 4, 14),
                                        (256, 256, 1024, 16, 14), (256, 256, 1, 1, 12),
                                        (1024, 512, 128, 8, 14), (512, 256, 64, 6, 12), (512, 256, 256, 8, 14),
                                        (512, 256, 40, 8, 14),
                                        # the staged Q6_K down kernel (1536-value rows): 3 of
                                        # 8 slot waves live; the SwiGLU formed in the down
                                        # launch (gate/up rows past 4096 values)
                                        (2048, 1536, 16, 3, 14), (4608, 1536, 8, 4, 14),
                                        # the staged gate/up kernel (4096-value rows) with 3 slots
                                        (4096, 512, 16, 3, 12)])
def test_moe_decode_vs_oracle(gpu, oracle, H, EFF, E, k, DT):
    rng = np.random.default_rng(H + E * k)
    table = synth.expert_table(rng, E, H, EFF, DT)
    lay = synth.expert_layout(H, EFF, DT)
    router, x = _routable(rng, E, H, k)
    out0 = rng.standard_normal(H).astype(np.float32)
    ws = torch.zeros(gpu.ops.moe_decode_workspace_bytes(H, EFF, E, k), dtype=torch.uint8, device="cuda")
    out = dev(out0)
    idx = torch.full((k,), -1, dtype=torch.int32, device="cuda")
    w = torch.zeros(k, device="cuda")
    case(f"moe_decode H={H} EFF={EFF} E={E} k={k} down={DT}")
    gpu.ops.moe_decode(dev(router), dev(table), *lay, DT, dev(x), H, EFF, E, k, ws, out, idx, w)
    _, ridx, rw, delta = _decode_ref(oracle, table, lay, DT, router, x, H, EFF, E, k)
    assert sorted(host(idx).tolist()) == sorted(ridx.tolist())
    assert np.allclose(host(w)[np.argsort(host(idx))], rw[np.argsort(ridx)], rtol=1e-5, atol=1e-6)
    err = rel_l2(host(out).astype(np.float64) - out0, delta)
    print(f"rel_l2={err:.2e}")
    assert err < TOL
    # a second call on the same workspace (tile counters must have been reset) adds again
    gpu.ops.moe_decode(dev(router), dev(table), *lay, DT, dev(x), H, EFF, E, k, ws, out, idx, w)
    assert rel_l2(host(out).astype(np.float64) - out0, 2 * delta) < TOL


def test_moe_decode_router_ties(gpu, oracle):
    """Router logits with exact ties (x one-hot, so each logit is one router weight): equal
    logits rank by lower expert index, also across the k-th place, as the oracle's top-k."""
    H, EFF, E, k, DT = 256, 256, 64, 8, 14
    rng = np.random.default_rng(5)
    table = synth.expert_table(rng, E, H, EFF, DT)
    lay = synth.expert_layout(H, EFF, DT)
    router = np.zeros((E, H), dtype=np.float32)
    col = -np.abs(rng.standard_normal(E)).astype(np.float32) - 4.0  # all below the winners
    col[[50, 3, 33, 12]] = [2.0, 2.0, 1.5, 1.5]  # ties inside the top k
    col[[7, 9, 60]] = [1.0, 0.5, 0.25]
    col[[44, 21, 30]] = 0.125  # three-way tie for the 8th place: 21 wins
    router[:, 0] = col
    x = np.zeros(H, dtype=np.float32)
    x[0] = 1.0
    out0 = rng.standard_normal(H).astype(np.float32)
    ws = torch.zeros(gpu.ops.moe_decode_workspace_bytes(H, EFF, E, k), dtype=torch.uint8, device="cuda")
    out = dev(out0)
    idx = torch.full((k,), -1, dtype=torch.int32, device="cuda")
    w = torch.zeros(k, device="cuda")
    case("moe_decode router ties")
    gpu.ops.moe_decode(dev(router), dev(table), *lay, DT, dev(x), H, EFF, E, k, ws, out, idx, w)
    _, ridx, rw, delta = _decode_ref(oracle, table, lay, DT, router, x, H, EFF, E, k)
    assert host(idx).tolist() == [3, 50, 12, 33, 7, 9, 60, 21]
    assert sorted(ridx.tolist()) == sorted(host(idx).tolist())
    assert np.allclose(host(w)[np.argsort(host(idx))], rw[np.argsort(ridx)], rtol=1e-5, atol=1e-6)
    assert rel_l2(host(out).astype(np.float64) - out0, delta) < TOL


def test_moe_decode_graph_replays(gpu):
    """Captured once, replayed several times with eager work in between: every replay
    matches the eager result bit for bit (deterministic combine, counters reset)."""
    H, EFF, E, k, DT = 1024, 512, 16, 8, 14
    rng = np.random.default_rng(3)
    table = dev(synth.expert_table(rng, E, H, EFF, DT))
    lay = synth.expert_layout(H, EFF, DT)
    router = dev((rng.standard_normal((E, H)) / 32).astype(np.float32))
    x = dev(rng.standard_normal(H).astype(np.float32))
    ws = torch.zeros(gpu.ops.moe_decode_workspace_bytes(H, EFF, E, k), dtype=torch.uint8, device="cuda")
    out = torch.zeros(H, device="cuda")
    case("moe_decode eager")
    gpu.ops.moe_decode(router, table, *lay, DT, x, H, EFF, E, k, ws, out)
    ref = host(out).copy()
    case("moe_decode graph capture + replays")
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=s):
            gpu.ops.moe_decode(router, table, *lay, DT, x, H, EFF, E, k, ws, out)
    for _ in range(3):
        out.zero_()
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert np.array_equal(host(out), ref)
        junk = torch.randn(1 << 20, device="cuda").sum()  # eager work between replays
        torch.cuda.synchronize()
        del junk


def test_moe_decode_workspace_shared_across_shapes(gpu):
    """One workspace (sized for the largest call) shared by calls of different shapes and
    expert counts, in an order where each call's layout overlaps data the previous call left:
    every call matches the same call on a fresh zero-filled workspace bit for bit (the router's
    arrival counter and tagged logit slots stay valid whatever came before)."""
    # (2048, 2560, 16, 10): the down launch combines through the tagged partial slots
    shapes = [(4096, 1536, 128, 8, 14), (1024, 512, 16, 4, 12), (2048, 2560, 16, 10, 14),
              (1024, 512, 16, 4, 12), (2048, 2560, 16, 10, 14), (4096, 1536, 128, 8, 14)]
    big = max(gpu.ops.moe_decode_workspace_bytes(H, EFF, E, k) for H, EFF, E, k, _ in shapes)
    shared = torch.zeros(big, dtype=torch.uint8, device="cuda")
    for i, (H, EFF, E, k, DT) in enumerate(shapes):
        rng = np.random.default_rng(100 + i)
        table = dev(synth.expert_table(rng, E, H, EFF, DT))
        lay = synth.expert_layout(H, EFF, DT)
        router = dev((rng.standard_normal((E, H)) / np.sqrt(H)).astype(np.float32))
        x = dev(rng.standard_normal(H).astype(np.float32))
        outs = []
        for ws in (torch.zeros(gpu.ops.moe_decode_workspace_bytes(H, EFF, E, k), dtype=torch.uint8,
                               device="cuda"), shared):
            out = torch.zeros(H, device="cuda")
            idx = torch.full((k,), -1, dtype=torch.int32, device="cuda")
            w = torch.zeros(k, device="cuda")
            case(f"moe_decode shared workspace call {i}: H={H} EFF={EFF} E={E} k={k} fresh={ws is not shared}")
            gpu.ops.moe_decode(router, table, *lay, DT, x, H, EFF, E, k, ws, out, idx, w)
            outs.append((host(out).copy(), host(idx).copy(), host(w).copy()))
        (o0, i0, w0), (o1, i1, w1) = outs
        assert (i0 >= 0).all() and np.array_equal(i0, i1) and np.array_equal(w0, w1)
        assert np.array_equal(o0, o1)


@pytest.mark.parametrize("H,EFF,E,k,DT,alias", [(512, 256, 16, 4, 14, False), (4096, 1536, 24, 8, 14, True),
                                                (1024, 512, 8, 8, 12, True)])
def test_moe_decode_rmsnorm_vs_oracle(gpu, oracle, H, EFF, E, k, DT, alias):
    """The norm folded into the router and gate/up launches: the same routing and delta as the
    oracle chain on rms_norm(x) * norm_w (forward.c:800-806 then :808-895), also with x == out."""
    rng = np.random.default_rng(7 * H + E + k)
    table = synth.expert_table(rng, E, H, EFF, DT)
    lay = synth.expert_layout(H, EFF, DT)
    eps = 1e-6
    while True:
        router = (rng.standard_normal((E, H)) / np.sqrt(H)).astype(np.float32)
        x = (3.0 * rng.standard_normal(H)).astype(np.float32)
        nw = (1.0 + 0.25 * rng.standard_normal(H)).astype(np.float32)
        xn = oracle.rms_norm(x, nw, eps)
        z = np.sort(router.astype(np.float64) @ xn)[::-1]
        if k == E or z[k - 1] - z[k] > 1e-3:
            break
    ws = torch.zeros(gpu.ops.moe_decode_workspace_bytes(H, EFF, E, k), dtype=torch.uint8, device="cuda")
    idx = torch.full((k,), -1, dtype=torch.int32, device="cuda")
    w = torch.zeros(k, device="cuda")
    _, ridx, rw, delta = _decode_ref(oracle, table, lay, DT, router, xn, H, EFF, E, k)
    case(f"moe_decode_rmsnorm H={H} EFF={EFF} E={E} k={k} down={DT} alias={alias}")
    if alias:  # the residual stream updated in place: out = x + moe(norm(x))
        out = dev(x)
        gpu.ops.moe_decode_rmsnorm(dev(router), dev(table), *lay, DT, out, dev(nw), eps, H, EFF, E, k, ws, out, idx, w)
        base = x.astype(np.float64)
    else:
        out0 = rng.standard_normal(H).astype(np.float32)
        out = dev(out0)
        gpu.ops.moe_decode_rmsnorm(dev(router), dev(table), *lay, DT, dev(x), dev(nw), eps, H, EFF, E, k, ws, out,
                                   idx, w)
        base = out0.astype(np.float64)
    assert sorted(host(idx).tolist()) == sorted(ridx.tolist())
    assert np.allclose(host(w)[np.argsort(host(idx))], rw[np.argsort(ridx)], rtol=1e-5, atol=1e-6)
    err = rel_l2(host(out).astype(np.float64) - base, delta)
    print(f"rel_l2={err:.2e}")
    assert err < TOL


def test_moe_decode_rmsnorm_rejects_ragged_hidden(gpu):
    H, EFF, E, k, DT = 514, 256, 4, 2, 14
    ws = torch.zeros(1 << 20, dtype=torch.uint8, device="cuda")
    table = torch.zeros(E * 4 << 20, dtype=torch.uint8, device="cuda")
    case("moe_decode_rmsnorm hidden % 4 != 0 rejected")
    with pytest.raises(gpu.MnemoError):
        gpu.ops.moe_decode_rmsnorm(torch.zeros(E * H, device="cuda"), table, 1 << 20, 0, 1 << 18, 1 << 19, DT,
                                   torch.zeros(H, device="cuda"), torch.ones(H, device="cuda"), 1e-6, H, EFF, E, k,
                                   ws, torch.zeros(H, device="cuda"))


@pytest.mark.parametrize("k", [8, 12])
def test_moe_decode_rmsnorm_in_place_graph(gpu, k):
    """The residual stream updated in place (x == out) by a captured graph, replayed as a
    token sequence: replay t reads the residual replay t-1 wrote.  Every replay equals the
    eager call on the same state, bit for bit (k = 8: the slot-parallel down launch; k = 12:
    the partial-buffer one with its counters)."""
    H, EFF, E, DT = 2048, 768, 32, 14
    rng = np.random.default_rng(k)
    table = dev(synth.expert_table(rng, E, H, EFF, DT))
    lay = synth.expert_layout(H, EFF, DT)
    router = dev((rng.standard_normal((E, H)) / 32).astype(np.float32))
    nw = dev((1 + 0.2 * rng.standard_normal(H)).astype(np.float32))
    x0 = rng.standard_normal(H).astype(np.float32)
    ws = torch.zeros(gpu.ops.moe_decode_workspace_bytes(H, EFF, E, k), dtype=torch.uint8, device="cuda")
    res = dev(x0)
    case(f"moe_decode_rmsnorm in place, eager sequence k={k}")
    eager = []
    for _ in range(4):
        gpu.ops.moe_decode_rmsnorm(router, table, *lay, DT, res, nw, 1e-6, H, EFF, E, k, ws, res)
        eager.append(host(res).copy())
    case(f"moe_decode_rmsnorm in place, graph replays k={k}")
    res.copy_(dev(x0))
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=s):
            gpu.ops.moe_decode_rmsnorm(router, table, *lay, DT, res, nw, 1e-6, H, EFF, E, k, ws, res)
    res.copy_(dev(x0))
    torch.cuda.synchronize()
    for t in range(4):
        g.replay()
        torch.cuda.synchronize()
        assert np.array_equal(host(res), eager[t]), t
        junk = torch.randn(1 << 18, device="cuda").sum()  # eager work between replays
        torch.cuda.synchronize()
        del junk


def test_moe_decode_staged_adversarial_x(gpu, oracle):
    """The staged gate/up (4096-value rows) and down (Q6_K 1536-value rows) launches on an
    input with one 1e3-times value in every 32-value block, a run of zero blocks and
    Student-t(2) tails: the two-byte x digits of each launch's image against the fp64 chain."""
    H, EFF, E, k, DT = 4096, 1536, 16, 8, 14
    rng = np.random.default_rng(77)
    table = synth.expert_table(rng, E, H, EFF, DT)
    lay = synth.expert_layout(H, EFF, DT)
    while True:
        x = rng.standard_t(2, H).astype(np.float32)
        x[rng.integers(0, 32, H // 32) + 32 * np.arange(H // 32)] *= 1e3
        x[512:768] = 0.0
        router = (rng.standard_normal((E, H)) / np.sqrt(H) / 1e3).astype(np.float32)
        z = np.sort(router.astype(np.float64) @ x)[::-1]
        if z[k - 1] - z[k] > 1e-3 * max(1.0, abs(z[0])):
            break
    out0 = rng.standard_normal(H).astype(np.float32)
    ws = torch.zeros(gpu.ops.moe_decode_workspace_bytes(H, EFF, E, k), dtype=torch.uint8, device="cuda")
    out = dev(out0)
    idx = torch.full((k,), -1, dtype=torch.int32, device="cuda")
    w = torch.zeros(k, device="cuda")
    case("moe_decode staged launches, adversarial x")
    gpu.ops.moe_decode(dev(router), dev(table), *lay, DT, dev(x), H, EFF, E, k, ws, out, idx, w)
    _, ridx, rw, delta = _decode_ref(oracle, table, lay, DT, router, x, H, EFF, E, k)
    assert sorted(host(idx).tolist()) == sorted(ridx.tolist())
    err = rel_l2(host(out).astype(np.float64) - out0, delta)
    print(f"rel_l2={err:.2e}")
    assert err < TOL


def test_moe_decode_unaligned_table(gpu, oracle):
    """The Qwen3 expert shape with the expert table 4 bytes past a 16-byte boundary: the
    staged gate/up and down launches (aligned 16-byte loads) decline it and the whole-row /
    slot-parallel kernels give the oracle chain's result."""
    H, EFF, E, k, DT = 4096, 1536, 16, 8, 14
    rng = np.random.default_rng(78)
    table = synth.expert_table(rng, E, H, EFF, DT)
    lay = synth.expert_layout(H, EFF, DT)
    while True:
        x = rng.standard_normal(H).astype(np.float32)
        router = (rng.standard_normal((E, H)) / np.sqrt(H)).astype(np.float32)
        z = np.sort(router.astype(np.float64) @ x)[::-1]
        if z[k - 1] - z[k] > 1e-3 * max(1.0, abs(z[0])):
            break
    buf = torch.zeros(table.size + 4, dtype=torch.uint8, device="cuda")
    buf[4:] = dev(table)
    td = buf[4:]
    assert td.data_ptr() % 16 == 4
    out0 = rng.standard_normal(H).astype(np.float32)
    ws = torch.zeros(gpu.ops.moe_decode_workspace_bytes(H, EFF, E, k), dtype=torch.uint8, device="cuda")
    out = dev(out0)
    idx = torch.full((k,), -1, dtype=torch.int32, device="cuda")
    w = torch.zeros(k, device="cuda")
    case("moe_decode, expert table at a 4-byte-aligned address")
    gpu.ops.moe_decode(dev(router), td, *lay, DT, dev(x), H, EFF, E, k, ws, out, idx, w)
    _, ridx, rw, delta = _decode_ref(oracle, table, lay, DT, router, x, H, EFF, E, k)
    assert sorted(host(idx).tolist()) == sorted(ridx.tolist())
    err = rel_l2(host(out).astype(np.float64) - out0, delta)
    print(f"rel_l2={err:.2e}")
    assert err < TOL


def test_moe_prefill_q4k_down_rounding(gpu):
    """The Q4_K down projection's roundings, in tiles of 128 and 72 tokens.  Its sum starts as the min term, M, and takes the products
    P_s of the 24 sub-blocks one by one, two roundings each, so the error's square is the sum of
    2 (2^-24 / sqrt(3))^2 S_s^2 at most, S_s = M + P_1 + .. + P_s; over mantissas in [1, 2) the mean is
    0.54 of that (0.74 in the error), and 15 % more is left for the last few roundings and the draw.
    (With the min term added at the end it is 1.06.)  The median over the tokens leaves out those where a SwiGLU
    value lies so close to a quantization step that fp32 takes the other side."""
    T, H, EFF = 200, 1024, 768
    rng = np.random.default_rng(77)
    lay = synth.expert_layout(H, EFF, 12)
    stride, g_off, u_off, d_off = lay
    blocks = rng.integers(0, 256, (stride // 144, 144), dtype=np.uint8)
    d = ((0.5 + rng.random((stride // 144, 2))) * np.array([1.2e-4, 9e-4])).astype(np.float16)
    blocks[:, :4] = d.view(np.uint8)
    table = dev(blocks.reshape(-1))
    x = dev((3 * rng.standard_normal((T, H))).astype(np.float32))
    idx, w = np.zeros((T, 1), np.int32), np.ones((T, 1), np.float32)
    case(f"moe_prefill down rounding T={T} H={H} EFF={EFF}")
    got = _run(gpu, table, lay, 12, x, dev(idx), dev(w), T, H, EFF, 1, 1, torch.zeros((T, H), device="cuda"))
    xq = torch_ref.quantize_q8_1(x).reshape(T, -1)
    g = torch_ref.gemm(12, table[g_off:u_off], xq, EFF, H, T).float()
    u = torch_ref.gemm(12, table[u_off:d_off], xq, EFF, H, T).float()
    a, ds = torch_ref.q8_1_parts(torch_ref.quantize_q8_1((g / (1 + torch.exp(-g)) * u).contiguous()), T, EFF)
    main, mins = torch_ref.q4k_split(table[d_off:stride], H, EFF)
    s = -(ds @ mins.T)
    sq = torch.zeros(T, dtype=torch.float64, device="cuda")
    for i in range(EFF // 32):
        s = s + a[:, 32 * i:32 * i + 32] @ main[:, 32 * i:32 * i + 32].T
        sq += 2 * (s * s).sum(1)
    assert torch.isfinite(s).all()
    ratio = (got.view(T, H).double() - s).norm(dim=1) / (2.0**-24 * (sq / 3).sqrt())
    print(f"median error / bound {float(ratio.median()):.3f}")
    assert float(ratio.median()) < 0.74 * 1.15
