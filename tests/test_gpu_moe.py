"""GPU parity for the MoE block through the C-ABI: router indices and slot
order bit-exact against tb_route_experts semantics, MoE outputs within
rel-L2 1e-5 of the oracle on the output and on the MoE delta (out - resid),
at the reference's golden layer, at the Qwen3-30B-A3B shapes of
BASELINE.json (batch 1 and 16), with a Zipf-skewed router bias, on tied, nearly tied and
underflowing logits, and through the C11 host block."""
import ctypes as C

import numpy as np
import pytest

import trailblaze_amd as tb
from conftest import bits_equal, load_golden, rel_l2
from gpu_util import dev, empty, host
from trailblaze_amd import formats as fm
from trailblaze_amd import synth

pytestmark = pytest.mark.gpu
TOL = 1e-5
COUNTER_BYTES = 256 * 1024   # counter area at the start of the MoE workspace


@pytest.fixture(scope="module", autouse=True)
def _init():
    print("device:", tb.init(), flush=True)


def gpu_route(xn, router, bias, k):
    import torch
    T, H = xn.shape
    E = router.shape[0]
    idx = empty(T * 8, torch.int32)
    w = empty(T * 8, torch.float32)
    tb.route(dev(xn), dev(router), None if bias is None else dev(bias), T, H, E, k, idx, w)
    return host(idx).reshape(T, 8), host(w).reshape(T, 8)


def gpu_moe(xn, resid, router, gate, up, down, F, k, qt, bias=None, mode=tb.TBQ_MOE_FP32):
    import torch
    T, H = xn.shape
    E = router.shape[0]
    L = tb.moe_layer(H, F, E, k, qt, dev(router), dev(gate), dev(up), dev(down),
                     None if bias is None else dev(bias))
    out = empty(T * H, torch.float32)
    idx = empty(T * 8, torch.int32)
    w = empty(T * 8, torch.float32)
    ws = torch.zeros(tb.moe_workspace_size(L, T, mode), dtype=torch.uint8, device="cuda")
    tb.moe_forward(L, T, dev(xn), dev(resid), out, idx, w, workspace=ws, mode=mode)
    assert_counters_zero(ws)
    return host(out).reshape(T, H), host(idx).reshape(T, 8), host(w).reshape(T, 8)


def assert_counters_zero(ws):
    """The workspace's counter words (the router's per-token arrival
    counters) are zero after every call."""
    c = host(ws[:COUNTER_BYTES])
    assert not c.any(), np.flatnonzero(c.view(np.uint32))[:8]


def test_route_golden_logit_vectors(oracle):
    # identity router: logits = xn exactly, so the reference's own routing
    # vectors (route.npz) drive the device softmax/top-k directly
    g = load_golden("route.npz")
    off_l = off_s = 0
    for E, k in zip(g["E"], g["k"]):
        lg = g["logits"][off_l:off_l + E]
        Hp = ((E + 7) // 8) * 8
        xn = np.zeros((1, Hp), np.float32)
        xn[0, :E] = lg
        router = np.zeros((E, Hp), np.float32)
        router[np.arange(E), np.arange(E)] = 1.0
        kk = min(int(k), 8)
        idx, w = gpu_route(xn, router, None, int(k))
        ref_i, ref_w = g["idx"][off_s:off_s + kk], g["w"][off_s:off_s + kk]
        assert np.array_equal(idx[0, :kk], ref_i), (E, k, lg)
        assert bits_equal(w[0, :kk], ref_w)
        off_l += E
        off_s += kk


def tie_case_logits(case):
    """64 logits that exercise the slot scan's tie rule (first slot holding
    the minimum; strictly larger enters) or underflowing probabilities."""
    rng = np.random.default_rng(7)
    E = 64
    lg = rng.standard_normal(E).astype(np.float32)
    if case == "tie4":
        lg[:8] = 1.0          # the fill leaves equal minima; the next entry picks among them
        lg[20] = 3.0
    elif case == "tie_boundary":
        lg[:] = np.float32(-2.0)
        lg[::5] = np.float32(1.5)  # 13 equal leaders for 8 slots
    elif case == "near_tie":
        top = np.argsort(-lg)
        lg[top[8]] = np.nextafter(lg[top[7]], np.float32(-np.inf))   # 8th and 9th one ulp apart
    else:
        lg[:] = np.float32(-200.0)  # probabilities of the tail underflow to zero
        lg[3] = 0.0
        lg[40] = np.float32(-199.0)
    return lg


@pytest.mark.parametrize("case", ["tie4", "tie_boundary", "near_tie", "underflow"])
def test_route_ties_and_underflow(oracle, case):
    """The slot scan's tie rule and probabilities that underflow to zero."""
    lg = tie_case_logits(case)
    E, k = lg.size, 8
    H = 512
    xn = np.zeros((1, H), np.float32)
    xn[0, :E] = lg
    router = np.zeros((E, H), np.float32)
    router[np.arange(E), np.arange(E)] = 1.0
    idx, w = gpu_route(xn, router, None, k)
    ri, rw = oracle.route(lg, k)
    assert np.array_equal(idx[0], ri)
    assert bits_equal(w[0], rw)


@pytest.mark.parametrize("T", [1, 16, 512])
def test_route_config_bit_exact(oracle, T):
    rng = np.random.default_rng(T)
    H, E, k = 2048, 128, 8
    router = synth.router_weights(E, H, rng)
    xn = synth.activations((T, H), rng)
    bias = synth.zipf_router_bias(E, 1.1, 1.0, rng) if T == 512 else None
    idx, w = gpu_route(xn, router, bias, k)
    lg = oracle.router_logits(xn, router, bias)
    for t in range(T):
        ri, rw = oracle.route(lg[t], k)
        assert np.array_equal(idx[t], ri), t
        assert bits_equal(w[t], rw), t


def test_moe_golden_layer():
    g = load_golden("moe.npz")
    out, idx, w = gpu_moe(g["xn"], g["resid"], g["router"], g["gate"], g["up"], g["down"], int(g["F"]),
                          int(g["k"]), int(g["qtype"]), bias=g["bias"])
    k = int(g["k"])
    assert np.array_equal(idx[:, :k], g["idx"][:, :k])
    assert bits_equal(w[:, :k], g["w"][:, :k])
    assert rel_l2(out, g["out"]) <= TOL
    assert rel_l2(out - g["resid"], g["out"] - g["resid"]) <= TOL


@pytest.fixture(scope="module")
def qwen_layer():
    H, F, E = 2048, 768, 128
    router, gate, up, down = synth.moe_layer(H, F, E, fm.Q4_K, seed=30)
    return H, F, E, router, gate, up, down


@pytest.mark.parametrize("T", [1, 16])
def test_moe_decode_config(oracle, qwen_layer, T):
    H, F, E, router, gate, up, down = qwen_layer
    rng = np.random.default_rng(100 + T)
    xn = synth.activations((T, H), rng)
    resid = synth.activations((T, H), rng)
    print("moe decode T=", T, flush=True)
    out, idx, w = gpu_moe(xn, resid, router, gate, up, down, F, 8, fm.Q4_K)
    ref, ridx, rw = oracle.moe(xn, resid, router, gate, up, down, F=F, top_k=8, qtype=fm.Q4_K)
    assert np.array_equal(idx, ridx)
    assert bits_equal(w, rw)
    assert rel_l2(out, ref) <= TOL
    assert rel_l2(out - resid, ref - resid) <= TOL


@pytest.mark.parametrize("T,H,F,E,k,qt,skew", [
    (8, 2048, 768, 128, 8, fm.Q4_K, False),
    (24, 1024, 512, 64, 6, fm.Q4_K, True),
    (32, 2048, 768, 128, 8, fm.Q4_K, True),
    (12, 4096, 1536, 256, 8, fm.Q4_K, False),
    (16, 2048, 768, 128, 8, fm.GGML | fm.Q4_K, True),
])
def test_moe_decode_expert_order(oracle, T, H, F, E, k, qt, skew):
    """Decode batches of 8..32 tokens run their expert kernels in expert
    order (a sorted pair list, down per pair, slot-ordered combine).  With a
    skewed router bias many tokens share an expert; every index and weight
    equals the reference's and the output is within tolerance."""
    router, gate, up, down = synth.moe_layer(H, F, E, qt, seed=T + E)
    rng = np.random.default_rng(T * 7 + k)
    bias = synth.zipf_router_bias(E, 1.1, 2.0, rng) if skew else None
    xn = synth.activations((T, H), rng)
    resid = synth.activations((T, H), rng)
    print("moe expert order T=", T, "H=", H, "E=", E, "k=", k, "qt=", qt, flush=True)
    out, idx, w = gpu_moe(xn, resid, router, gate, up, down, F, k, qt, bias=bias)
    ref, ridx, rw = oracle.moe(xn, resid, router, gate, up, down, F=F, top_k=k, qtype=qt, bias=bias)
    assert np.array_equal(idx, ridx)
    assert bits_equal(w, rw)
    if skew:   # the bias concentrates the selections: some expert has several tokens
        assert np.bincount(idx[:, :k].ravel(), minlength=E).max() >= 3
    assert rel_l2(out - resid, ref - resid) <= TOL


def test_moe_decode_router_many_tokens(oracle):
    """Routing inside tbq_moe_forward over 512 decode tokens (32 batches of
    16): every index, slot and weight equal to the reference's."""
    H, F, E, k = 2048, 256, 128, 8
    router, gate, up, down = synth.moe_layer(H, F, E, fm.Q4_K, seed=41)
    import torch
    L = tb.moe_layer(H, F, E, k, fm.Q4_K, dev(router), dev(gate), dev(up), dev(down))
    rng = np.random.default_rng(41)
    T = 16
    ws = torch.zeros(tb.moe_workspace_size(L, T), dtype=torch.uint8, device="cuda")
    out = empty(T * H, torch.float32)
    for b in range(32):
        xn = synth.activations((T, H), rng)
        resid = np.zeros((T, H), np.float32)
        idx = empty(T * 8, torch.int32)
        w = empty(T * 8, torch.float32)
        tb.moe_forward(L, T, dev(xn), dev(resid), out, idx, w, workspace=ws)
        idx, w = host(idx).reshape(T, 8), host(w).reshape(T, 8)
        lg = oracle.router_logits(xn, router, None)
        for t in range(T):
            ri, rw = oracle.route(lg[t], k)
            assert np.array_equal(idx[t], ri), (b, t)
            assert bits_equal(w[t], rw), (b, t)


def test_moe_decode_repeated_calls(oracle):
    """One workspace across calls of different batch sizes (1, 16, 3, 1):
    outputs in tolerance every time and the counter words back at zero
    after each call."""
    import torch
    H, F, E, k = 2048, 256, 128, 8
    router, gate, up, down = synth.moe_layer(H, F, E, fm.Q4_K, seed=52)
    L = tb.moe_layer(H, F, E, k, fm.Q4_K, dev(router), dev(gate), dev(up), dev(down))
    ws = torch.zeros(tb.moe_workspace_size(L, 16), dtype=torch.uint8, device="cuda")
    rng = np.random.default_rng(52)
    for T in (1, 16, 3, 1):
        print("moe repeated call T=", T, flush=True)
        xn = synth.activations((T, H), rng)
        resid = synth.activations((T, H), rng)
        out = empty(T * H, torch.float32)
        idx = empty(T * 8, torch.int32)
        w = empty(T * 8, torch.float32)
        tb.moe_forward(L, T, dev(xn), dev(resid), out, idx, w, workspace=ws)
        ref, ridx, _ = oracle.moe(xn, resid, router, gate, up, down, F=F, top_k=k, qtype=fm.Q4_K)
        assert np.array_equal(host(idx).reshape(T, 8), ridx), T
        assert rel_l2(host(out).reshape(T, H) - resid, ref - resid) <= TOL, T
        assert_counters_zero(ws)


@pytest.mark.parametrize("case", ["tie4", "tie_boundary", "near_tie", "underflow"])
def test_moe_decode_router_ties(oracle, case):
    """Tied, nearly tied and underflowing logits through tbq_moe_forward:
    the reference's indices, slot order and weights bit for bit."""
    lg = tie_case_logits(case)
    E, k, H, F = lg.size, 8, 512, 256
    router = np.zeros((E, H), np.float32)
    router[np.arange(E), np.arange(E)] = 1.0
    _, gate, up, down = synth.moe_layer(H, F, E, fm.Q4_K, seed=13)
    xn = np.zeros((1, H), np.float32)
    xn[0, :E] = lg
    resid = synth.activations((1, H), np.random.default_rng(13))
    out, idx, w = gpu_moe(xn, resid, router, gate, up, down, F, k, fm.Q4_K)
    ref, ridx, rw = oracle.moe(xn, resid, router, gate, up, down, F=F, top_k=k, qtype=fm.Q4_K)
    assert np.array_equal(idx, ridx)
    assert bits_equal(w, rw)
    assert rel_l2(out - resid, ref - resid) <= TOL


@pytest.mark.parametrize("qt", [fm.Q2_K, fm.Q3_K, fm.Q5_K, fm.Q6_K, fm.Q8_0])
def test_moe_other_formats(oracle, qt):
    H, F, E, k, T = 512, 256, 16, 4, 3
    router, gate, up, down = synth.moe_layer(H, F, E, qt, seed=qt)
    rng = np.random.default_rng(qt)
    xn = synth.activations((T, H), rng)
    resid = synth.activations((T, H), rng)
    out, idx, w = gpu_moe(xn, resid, router, gate, up, down, F, k, qt)
    ref, ridx, rw = oracle.moe(xn, resid, router, gate, up, down, F=F, top_k=k, qtype=qt)
    assert np.array_equal(idx, ridx)
    assert rel_l2(out - resid, ref - resid) <= TOL


def test_moe_host_block(oracle):
    """The C11 host substitution for tb_layer_forward's MoE branch."""
    g = load_golden("moe.npz")
    H, F, E, k = int(g["H"]), int(g["F"]), int(g["E"]), int(g["k"])
    T = g["xn"].shape[0]
    tensors = [dev(g[n]) for n in ("router", "gate", "up", "down", "bias")]
    L = tb.moe_layer(H, F, E, k, int(g["qtype"]), *tensors[:4], bias=tensors[4])
    import torch
    torch.cuda.synchronize()
    out = np.zeros((T, H), np.float32)
    idx = np.zeros((T, 8), np.int32)
    w = np.zeros((T, 8), np.float32)
    ok = tb.lib().tbq_moe_block_host(C.byref(L), T, g["xn"].ctypes.data, g["resid"].ctypes.data,
                                     out.ctypes.data, idx.ctypes.data, w.ctypes.data, tb.TBQ_MOE_FP32)
    assert ok == 1, tb.lib().tbq_last_error()
    assert np.array_equal(idx[:, :k], g["idx"][:, :k])
    assert rel_l2(out, g["out"]) <= TOL


@pytest.mark.parametrize("H", [512, 2048])
def test_moe_host_block_varying_batches(oracle, H):
    """tbq_moe_block_host over a sequence of calls whose T and mode change,
    so its cached buffer is reused at a smaller T and regrown at a larger
    one: every call routes exactly and stays within tolerance.  H = 512 and
    2048 take the router whose per-token arrival counters live in the
    workspace (T < 32), the path a misplaced or unzeroed counter area
    breaks."""
    F, E, k = 256, 16, 4
    router, gate, up, down = synth.moe_layer(H, F, E, fm.Q4_K, seed=H + 7)
    L = tb.moe_layer(H, F, E, k, fm.Q4_K, dev(router), dev(gate), dev(up), dev(down))
    import torch
    torch.cuda.synchronize()
    for i, (T, mode) in enumerate([(5, tb.TBQ_MOE_FP32), (1, tb.TBQ_MOE_FP32), (16, tb.TBQ_MOE_FP32),
                                   (1, tb.TBQ_MOE_FP32), (40, tb.TBQ_MOE_BF16), (1, tb.TBQ_MOE_FP32),
                                   (3, tb.TBQ_MOE_BF16), (2, tb.TBQ_MOE_FP32), (24, tb.TBQ_MOE_I8),
                                   (1, tb.TBQ_MOE_FP32)]):
        print(f"host block H={H} call {i}: T={T} mode={mode}", flush=True)
        rng = np.random.default_rng(1000 * H + i)
        xn = synth.activations((T, H), rng)
        resid = synth.activations((T, H), rng)
        out = np.zeros((T, H), np.float32)
        idx = np.full((T, 8), 77, np.int32)
        w = np.zeros((T, 8), np.float32)
        ok = tb.lib().tbq_moe_block_host(C.byref(L), T, xn.ctypes.data, resid.ctypes.data, out.ctypes.data,
                                         idx.ctypes.data, w.ctypes.data, mode)
        assert ok == 1, tb.lib().tbq_last_error()
        ref, ridx, rw = oracle.moe(xn, resid, router, gate, up, down, F=F, top_k=k, qtype=fm.Q4_K)
        assert np.array_equal(idx, ridx), (T, mode)
        assert bits_equal(w, rw), (T, mode)
        tol = TOL if mode == tb.TBQ_MOE_FP32 else 1e-2
        assert rel_l2(out - resid, ref - resid) <= tol, (T, mode)


# ---------------------------------------------------------------------------
# Prefill: grouped fp16 MFMA experts (tolerance 1e-2 rel-L2, routing exact)
# ---------------------------------------------------------------------------
PREFILL_TOL = 1e-2


def test_moe_prefill_mfma_golden_layer():
    g = load_golden("moe.npz")
    out, idx, w = gpu_moe(g["xn"], g["resid"], g["router"], g["gate"], g["up"], g["down"], int(g["F"]),
                          int(g["k"]), int(g["qtype"]), bias=g["bias"], mode=tb.TBQ_MOE_BF16)
    k = int(g["k"])
    assert np.array_equal(idx[:, :k], g["idx"][:, :k])
    assert rel_l2(out - g["resid"], g["out"] - g["resid"]) <= PREFILL_TOL


def test_moe_prefill_mfma_config(oracle, qwen_layer):
    """512 tokens, Zipf(1.1)-skewed router bias."""
    H, F, E, router, gate, up, down = qwen_layer
    T = 512
    rng = np.random.default_rng(512)
    bias = synth.zipf_router_bias(E, 1.1, 1.0, rng)
    xn = synth.activations((T, H), rng)
    resid = synth.activations((T, H), rng)
    out, idx, w = gpu_moe(xn, resid, router, gate, up, down, F, 8, fm.Q4_K, bias=bias, mode=tb.TBQ_MOE_BF16)
    # routing: every token bit-exact
    lg = oracle.router_logits(xn, router, bias)
    for t in range(T):
        ri, rw = oracle.route(lg[t], 8)
        assert np.array_equal(idx[t], ri), t
        assert bits_equal(w[t], rw), t
    counts = np.bincount(idx.reshape(-1), minlength=E)
    assert counts.max() > 4 * counts.mean()      # the bias really skews the load
    # outputs: tokens are independent, so a sample checks the whole layer
    sample = np.sort(rng.choice(T, 32, replace=False))
    ref, _, _ = oracle.moe(xn[sample], resid[sample], router, gate, up, down, F=F, top_k=8, qtype=fm.Q4_K, bias=bias)
    assert rel_l2(out[sample] - resid[sample], ref - resid[sample]) <= PREFILL_TOL
    assert rel_l2(out[sample], ref) <= PREFILL_TOL


def test_moe_prefill_mfma_small_batches(oracle):
    """Tiles with 1..64 pairs, experts with zero tokens, several tiles per expert."""
    H, F, E, k = 512, 256, 8, 4
    router, gate, up, down = synth.moe_layer(H, F, E, fm.Q4_K, seed=91)
    for T in (1, 3, 17, 70):
        rng = np.random.default_rng(T)
        xn = synth.activations((T, H), rng)
        resid = synth.activations((T, H), rng)
        out, idx, w = gpu_moe(xn, resid, router, gate, up, down, F, k, fm.Q4_K, mode=tb.TBQ_MOE_BF16)
        ref, ridx, rw = oracle.moe(xn, resid, router, gate, up, down, F=F, top_k=k, qtype=fm.Q4_K)
        assert np.array_equal(idx, ridx)
        assert rel_l2(out - resid, ref - resid) <= PREFILL_TOL


@pytest.mark.parametrize("mode", ["BF16", "I8"])
def test_moe_prefill_many_pairs(oracle, mode):
    """More (token, slot) pairs than the dispatch keeps in LDS (8400 > 8192):
    the permutation goes through global memory.  Routing exact for every
    token; outputs checked on a sample (tokens are independent)."""
    H, F, E, k, T = 512, 256, 8, 4, 2100
    router, gate, up, down = synth.moe_layer(H, F, E, fm.Q4_K, seed=93)
    rng = np.random.default_rng(94)
    xn = synth.activations((T, H), rng)
    resid = synth.activations((T, H), rng)
    out, idx, w = gpu_moe(xn, resid, router, gate, up, down, F, k, fm.Q4_K, mode=getattr(tb, "TBQ_MOE_" + mode))
    sample = np.sort(rng.choice(T, 48, replace=False))
    ref, ridx, rw = oracle.moe(xn[sample], resid[sample], router, gate, up, down, F=F, top_k=k, qtype=fm.Q4_K)
    assert np.array_equal(idx[sample], ridx)
    assert rel_l2(out[sample] - resid[sample], ref - resid[sample]) <= PREFILL_TOL


# ---------------------------------------------------------------------------
# Prefill on int8 MFMA with Q8_K activations (TBQ_MOE_I8): routing exact,
# outputs within 1e-2 rel-L2 (8-bit activations)
# ---------------------------------------------------------------------------
def test_quantize_q8k_device_matches_oracle(oracle):
    """tbq_quantize_q8k writes the Q8_K blocks the pinned oracle quantiser
    writes (d, every int8 quant, every 16-element sum), byte for byte, on
    N(0,1) blocks, tiny and huge scales, 1000x outliers, an all-zero block,
    a constant block and exact rounding ties."""
    import torch
    rng = np.random.default_rng(81)
    parts = [rng.standard_normal(4096).astype(np.float32),
             (rng.standard_normal(512) * 1e-30).astype(np.float32),
             (rng.standard_normal(512) * 1e30).astype(np.float32),
             np.zeros(256, np.float32), np.full(256, -3.25, np.float32)]
    o = rng.standard_normal(1024).astype(np.float32)
    o[rng.choice(1024, 9, replace=False)] *= 1000.0
    ties = np.zeros(256, np.float32)
    ties[0], ties[1], ties[2] = 127.0, 2.5, -3.5
    x = np.concatenate(parts + [o, ties])
    blocks = empty(x.size // 256 * 292, torch.uint8)
    assert tb.lib().tbq_quantize_q8k(dev(x).data_ptr(), x.size, blocks.data_ptr(), None) == 1
    got = host(blocks)
    want = oracle.quantize_q8k(x)
    assert np.array_equal(got, want), np.flatnonzero(got != want)[:10]


def test_moe_prefill_i8_config(oracle, qwen_layer):
    """BASELINE configs[4] on the int8 path: 512 tokens, Zipf(1.1)-skewed
    router bias."""
    H, F, E, router, gate, up, down = qwen_layer
    T = 512
    rng = np.random.default_rng(512)
    bias = synth.zipf_router_bias(E, 1.1, 1.0, rng)
    xn = synth.activations((T, H), rng)
    resid = synth.activations((T, H), rng)
    out, idx, w = gpu_moe(xn, resid, router, gate, up, down, F, 8, fm.Q4_K, bias=bias, mode=tb.TBQ_MOE_I8)
    lg = oracle.router_logits(xn, router, bias)
    for t in range(T):
        ri, rw = oracle.route(lg[t], 8)
        assert np.array_equal(idx[t], ri), t
        assert bits_equal(w[t], rw), t
    sample = np.sort(rng.choice(T, 32, replace=False))
    ref, _, _ = oracle.moe(xn[sample], resid[sample], router, gate, up, down, F=F, top_k=8, qtype=fm.Q4_K, bias=bias)
    e = rel_l2(out[sample] - resid[sample], ref - resid[sample])
    print("int8 prefill delta rel-L2", e, flush=True)
    assert e <= PREFILL_TOL
    assert rel_l2(out[sample], ref) <= PREFILL_TOL


@pytest.mark.parametrize("H,F,E,k", [(512, 256, 8, 4), (2048, 768, 16, 8), (1024, 512, 6, 2)])
def test_moe_prefill_i8_small_batches(oracle, H, F, E, k):
    """Tiles of 1..70 pairs (one and two 64-pair halves), experts with no
    tokens, several tiles per expert, K of 2..16 chunks."""
    router, gate, up, down = synth.moe_layer(H, F, E, fm.Q4_K, seed=H + E)
    for T in (1, 3, 17, 70):
        print(f"int8 prefill H={H} F={F} E={E} k={k} T={T}", flush=True)
        rng = np.random.default_rng(T + H)
        xn = synth.activations((T, H), rng)
        resid = synth.activations((T, H), rng)
        out, idx, w = gpu_moe(xn, resid, router, gate, up, down, F, k, fm.Q4_K, mode=tb.TBQ_MOE_I8)
        ref, ridx, rw = oracle.moe(xn, resid, router, gate, up, down, F=F, top_k=k, qtype=fm.Q4_K)
        assert np.array_equal(idx, ridx)
        assert rel_l2(out - resid, ref - resid) <= PREFILL_TOL


# Every token takes the same k experts (a zero router under distinct biases), so
# each expert's tile holds exactly T pairs: both sides of the 32-pair sub-tiles
# and of the 128-pair tile, one super-block rows (the shortest ring), and the
# shapes whose items take one and two row blocks per wave in either GEMM.
@pytest.mark.parametrize("qt", [fm.Q4_K, fm.GGML | fm.Q4_K])
@pytest.mark.parametrize("T,H,F,E,k", [
    (1, 256, 512, 2, 1), (31, 512, 256, 3, 2), (33, 256, 256, 4, 2), (64, 768, 512, 2, 2), (65, 256, 768, 4, 1),
    (97, 512, 256, 2, 1), (128, 256, 256, 3, 1), (129, 512, 256, 2, 2),
    (33, 256, 4096, 64, 8), (129, 256, 4096, 64, 8), (97, 4096, 256, 128, 8),
    # two row blocks per wave on 256 CUs, 16 tiles (128 pairs, and 1 to 128): gate/up, then down
    (161, 256, 4096, 8, 8), (193, 256, 4096, 8, 8), (256, 256, 4096, 8, 8),
    (129, 4096, 256, 8, 8), (161, 4096, 256, 8, 8), (193, 4096, 256, 8, 8), (256, 4096, 256, 8, 8),
])
def test_moe_prefill_tile_edges(oracle, qt, T, H, F, E, k):
    import torch
    _, gate, up, down = synth.moe_layer(H, F, E, qt, seed=T + H)
    router = np.zeros((E, H), np.float32)
    rng = np.random.default_rng(T * 3 + F)
    bias = rng.permutation(E).astype(np.float32) * np.float32(0.25)
    xn = synth.activations((T, H), rng)
    resid = synth.activations((T, H), rng)
    L = tb.moe_layer(H, F, E, k, qt, dev(router), dev(gate), dev(up), dev(down), dev(bias))
    out, idx, w = empty((T + 1) * H, torch.float32), empty(T * 8, torch.int32), empty(T * 8, torch.float32)
    out.fill_(7.0)
    ws = torch.zeros(tb.moe_workspace_size(L, T, tb.TBQ_MOE_BF16), dtype=torch.uint8, device="cuda")
    print("moe prefill tile edges", T, H, F, E, k, qt, flush=True)
    for _ in range(2):   # the second call on the first one's workspace
        tb.moe_forward(L, T, dev(xn), dev(resid), out, idx, w, workspace=ws, mode=tb.TBQ_MOE_BF16)
    # the oracle on every fifth token of the largest shapes (tokens do not mix)
    t = np.arange(0, T, 5 if T * k * H * F > 5e8 else 1)
    ref, ridx, rw = oracle.moe(xn[t], resid[t], router, gate, up, down, F=F, top_k=k, qtype=qt, bias=bias)
    assert np.array_equal(host(idx).reshape(T, 8)[t], ridx)
    assert bits_equal(host(w).reshape(T, 8)[t], rw)
    got = host(out).reshape(T + 1, H)
    resid = resid[t]
    assert np.all(got[T] == 7.0)
    # The mode's bound over the layer, and the same per token against the tokens'
    # typical size: fp16 operands err by 2^-11 of the sum of |w||x|, which tokens
    # share, and these weights' nonzero mean makes some tokens' sums cancel to a
    # fraction of it.  A token in a wrong slot would be off by its whole size.
    d, r = got[t] - ref, ref - resid
    assert np.all(np.isfinite(got)) and np.linalg.norm(d) <= 1e-2 * np.linalg.norm(r)
    assert np.linalg.norm(d, axis=1).max() <= 3e-2 * np.sqrt(np.mean(np.sum(r * r, axis=1)))


# Experts of very different loads, so the int8 items of one launch come from
# tiles of all four sub-tile counts: full tiles, remainders on both sides of a
# sub-tile, and experts with no pair at all.
@pytest.mark.parametrize("T,H,F,E,k,spread", [(37, 256, 256, 16, 2, 4.0), (150, 512, 256, 24, 3, 3.0),
                                              (400, 256, 512, 16, 2, 3.0)])
def test_moe_prefill_int8_mixed_tiles(oracle, T, H, F, E, k, spread):
    import torch
    router, gate, up, down = synth.moe_layer(H, F, E, fm.Q4_K, seed=T + E)
    rng = np.random.default_rng(T + 5 * E)
    xn, resid = synth.activations((T, H), rng), synth.activations((T, H), rng)
    bias = (np.linspace(-spread, spread, E) * np.std(xn @ router.T)).astype(np.float32)
    ref, ridx, rw = oracle.moe(xn, resid, router, gate, up, down, F=F, top_k=k, qtype=fm.Q4_K, bias=bias)
    n = np.bincount(ridx[:, :k].ravel(), minlength=E)
    classes = {(int(c) % 128 + 31) // 32 for c in n if c % 128} | {4 for c in n if c >= 128}
    assert n.min() == 0 and len(classes) >= min(T // 50, 4)
    L = tb.moe_layer(H, F, E, k, fm.Q4_K, dev(router), dev(gate), dev(up), dev(down), dev(bias))
    out, idx, w = empty(T * H, torch.float32), empty(T * 8, torch.int32), empty(T * 8, torch.float32)
    ws = torch.zeros(tb.moe_workspace_size(L, T, tb.TBQ_MOE_I8), dtype=torch.uint8, device="cuda")
    print("moe int8 mixed tiles", T, H, F, E, k, sorted(n), flush=True)
    for _ in range(2):
        tb.moe_forward(L, T, dev(xn), dev(resid), out, idx, w, workspace=ws, mode=tb.TBQ_MOE_I8)
    assert np.array_equal(host(idx).reshape(T, 8)[:, :k], ridx[:, :k])
    assert rel_l2(host(out).reshape(T, H) - resid, ref - resid) <= PREFILL_TOL


# Scale fields at and below fp16's smallest normal number.  The reference's
# layout reads a subnormal half as m * 2^-136 (zero beside anything else),
# ggml's as IEEE does; here they carry about half of the weights' size, so a
# decoder of the other kind is off by tens of percent.
@pytest.mark.parametrize("qt,mode", [(fm.Q4_K, tb.TBQ_MOE_BF16), (fm.GGML | fm.Q4_K, tb.TBQ_MOE_BF16),
                                     (fm.Q4_K, tb.TBQ_MOE_I8)])
@pytest.mark.parametrize("T", [40, 150])   # one row block per wave at both; one and two 32-pair sub-tiles
def test_moe_prefill_subnormal_scales(oracle, qt, mode, T):
    H, F, E, k = 512, 256, 4, 2
    router, gate, up, down = synth.moe_layer(H, F, E, qt, seed=77)
    rng = np.random.default_rng(T)
    for W in (gate, up, down):
        b = W.reshape(-1, 144)
        for off in (0, 2):
            h = np.where(rng.random(len(b)) < 0.5, rng.integers(0x0200, 0x0400, len(b)), rng.integers(0x0400, 0x0600, len(b)))
            b[:, off:off + 2] = h.astype(np.uint16).view(np.uint8).reshape(-1, 2)
    xn, resid = synth.activations((T, H), rng) * np.float32(32), np.zeros((T, H), np.float32)
    print("moe prefill subnormal scales", qt, mode, T, flush=True)
    out, idx, _ = gpu_moe(xn, resid, router, gate, up, down, F, k, qt, mode=mode)
    ref, ridx, _ = oracle.moe(xn, resid, router, gate, up, down, F=F, top_k=k, qtype=qt)
    assert np.array_equal(idx, ridx)
    assert rel_l2(out, ref) <= 1e-2


# Both sides of the pair counts at which the dispatch goes to its next instance
# (4, 8 and 16 pairs a thread, then the permutation in global memory).
@pytest.mark.parametrize("T", [512, 513, 1024, 1025, 2048, 2049])
def test_moe_prefill_dispatch_instances(oracle, T):
    H, F, E, k = 256, 256, 200, 8
    router, gate, up, down = synth.moe_layer(H, F, E, fm.Q4_K, seed=91)
    rng = np.random.default_rng(T)
    xn, resid = synth.activations((T, H), rng), synth.activations((T, H), rng)
    print("moe dispatch instances", T, flush=True)
    out, idx, w = gpu_moe(xn, resid, router, gate, up, down, F, k, fm.Q4_K, mode=tb.TBQ_MOE_BF16)
    t = np.r_[0:T:11, T - 2, T - 1]   # tokens do not mix: the oracle on some of them
    ref, ridx, rw = oracle.moe(xn[t], resid[t], router, gate, up, down, F=F, top_k=k, qtype=fm.Q4_K)
    assert np.array_equal(idx[t], ridx) and bits_equal(w[t], rw) and np.all(np.isfinite(out))
    d, r = out[t] - ref, ref - resid[t]
    assert np.linalg.norm(d) <= PREFILL_TOL * np.linalg.norm(r)
    assert np.linalg.norm(d, axis=1).max() <= 3 * PREFILL_TOL * np.sqrt(np.mean(np.sum(r * r, axis=1)))
