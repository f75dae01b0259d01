"""The framework's main path as a user's program runs it: decode matvecs over
quantised rows, the MoE block at decode and at prefill, and a dense
Qwen3-style model's decode step and prompt prefill, each through the package's
public entry points (trailblaze_amd.matvec, moe_forward and the tbq_dense_*
calls of include/tbq.h).

Weights are random K-quant blocks whose fp16 scales are chosen so that a
dequantised weight has mean ~0 and a standard deviation near 1/sqrt(K), as
trained matrices have (and never an fp16 subnormal); activations, KV rows and
router weights follow the repository's own synthetic recipe (N(0, 1), N(0, 1),
N(0, 0.02)).
"""
from __future__ import annotations

import ctypes as C
import math

import torch

import trailblaze_amd as tb
from trailblaze_amd import dense as td
from trailblaze_amd import formats as fm

Q4_0, Q8_0, Q2_K, Q3_K, Q4_K, Q5_K, Q6_K = fm.Q4_0, fm.Q8_0, fm.Q2_K, fm.Q3_K, fm.Q4_K, fm.Q5_K, fm.Q6_K
GGML = fm.GGML
ROUTER_STD = 0.02   # standard deviation of the router's weights
NORM_EPS, ROPE_THETA = 1e-6, 1e6


# ---- the cases ---------------------------------------------------------------
def listed():
    moe = dict(H=2048, F=768, E=128, k=8)                       # Qwen3-30B-A3B's layer
    qwen4b = dict(hidden=2560, heads=32, kv=8, dim=128, ffn=9728)  # Qwen3-4B's widths
    return [
        # one square projection at batch 1: the smallest call, launch and latency
        dict(name="matvec-q4k-4096x4096", kind="matvec", qt=Q4_K, M=4096, K=4096),
        # an 8B model's down projection in the 3-bit format
        dict(name="matvec-q3k-4096x12288", kind="matvec", qt=Q3_K, M=4096, K=12288),
        # the lm_head: the largest matrix of a decode step, in llama.cpp's layout
        dict(name="matvec-ggml-q6k-151936x4096", kind="matvec", qt=GGML | Q6_K, M=151936, K=4096),
        # one token through a MoE layer
        dict(name="moe-decode-1", kind="moe", T=1, qg=Q4_K, qd=Q4_K, mode=tb.TBQ_MOE_FP32, zipf=False, **moe),
        # a serving batch of 16, with the wider down projection that Q4_K_M files have
        dict(name="moe-decode-16-q6k-down", kind="moe", T=16, qg=Q4_K, qd=Q6_K, mode=tb.TBQ_MOE_FP32, zipf=False, **moe),
        # a 512-token prompt, expert load Zipf-skewed
        dict(name="moe-prefill-512-zipf", kind="moe", T=512, qg=Q4_K, qd=Q4_K, mode=tb.TBQ_MOE_BF16, zipf=True, **moe),
        # a longer ragged prompt on llama.cpp's layout
        dict(name="moe-prefill-1999-ggml", kind="moe", T=1999, qg=GGML | Q4_K, qd=GGML | Q4_K, mode=tb.TBQ_MOE_BF16,
             zipf=False, **moe),
        # the int8 option, for programs that want its smaller error
        dict(name="moe-prefill-512-int8", kind="moe", T=512, qg=Q4_K, qd=Q4_K, mode=tb.TBQ_MOE_I8, zipf=True, **moe),
        # one decode step of a small model early in a conversation: launches and latency
        dict(name="dense-decode-small", kind="decode", layers=8, hidden=1024, heads=16, kv=8, dim=64, ffn=3072,
             vocab=32000, pos=200, ql=Q8_0, qd=Q8_0, qe=Q8_0),
        # one decode step of the whole 36-layer model at context 4096
        dict(name="dense-decode-4b-ctx4096", kind="decode", layers=36, vocab=151936, pos=4095, ql=Q4_K, qd=Q4_K,
             qe=Q6_K, **qwen4b),
        # two layers of the same model over a 512-token prompt (a small
        # vocabulary: the layers are what is measured)
        dict(name="dense-prefill-512", kind="prefill", layers=2, vocab=8192, T=512, pos0=0, ql=Q4_K, qd=Q4_K, qe=Q6_K,
             **qwen4b),
        # the second, ragged chunk of a longer prompt, on a Q4_K_M file's
        # layers in llama.cpp's layout (Q6_K down projections)
        dict(name="dense-prefill-1999-ggml-mix", kind="prefill", layers=2, vocab=8192, T=1999, pos0=1024,
             ql=GGML | Q4_K, qd=GGML | Q6_K, qe=GGML | Q6_K, **qwen4b),
    ]


def _log(rng, lo, hi, step=1):
    """A size spread evenly over the logarithm of lo .. hi, a multiple of step."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi))) / step)) * step))


FORMATS = (Q4_0, Q8_0, Q2_K, Q3_K, Q4_K, Q5_K, Q6_K)


def draw(rng):
    kind = rng.choice(["matvec", "matvec", "moe-decode", "moe-prefill", "moe-prefill", "decode", "prefill", "prefill"])
    layout = rng.choice([0, GGML])
    if kind == "matvec":
        K = _log(rng, 512, 16384, 256)
        return dict(kind="matvec", qt=layout | rng.choice(FORMATS), M=_log(rng, 256, min(151936, 600_000_000 // K)), K=K)
    if kind.startswith("moe"):
        c = dict(kind="moe", H=rng.choice([1024, 1536, 2048, 3072]), F=rng.choice([512, 768, 1024, 1536]),
                 E=rng.choice([32, 64, 128]), k=rng.choice([2, 4, 8]), zipf=rng.random() < 0.5)
        if kind == "moe-decode":
            q = rng.choice([(Q4_K, Q4_K), (Q4_K, Q6_K), (Q5_K, Q5_K), (Q8_0, Q8_0), (Q3_K, Q4_K)])
            return dict(c, T=_log(rng, 1, 32), qg=layout | q[0], qd=layout | q[1], mode=tb.TBQ_MOE_FP32)
        mode = tb.TBQ_MOE_I8 if not layout and rng.random() < 0.25 else tb.TBQ_MOE_BF16
        return dict(c, T=_log(rng, 33, 2048), qg=layout | Q4_K, qd=layout | Q4_K, mode=mode)
    shape = rng.choice([dict(hidden=1024, heads=16, kv=8, dim=64, ffn=3072), dict(hidden=2048, heads=16, kv=8, dim=128, ffn=6144),
                        dict(hidden=2560, heads=32, kv=8, dim=128, ffn=9728), dict(hidden=4096, heads=32, kv=4, dim=128, ffn=12288)])
    q = rng.choice([(Q4_K, Q4_K), (Q4_K, Q4_K), (Q4_K, Q6_K), (Q5_K, Q5_K), (Q8_0, Q8_0)])
    c = dict(vocab=8192, ql=layout | q[0], qd=layout | q[1], qe=layout | Q6_K, **shape)
    if kind == "decode":
        return dict(c, kind="decode", layers=rng.randint(2, 8), pos=_log(rng, 1, 4095))
    return dict(c, kind="prefill", layers=2, T=_log(rng, 16, 2048), pos0=rng.choice([0, 0, _log(rng, 16, 1024)]))


# ---- inputs ------------------------------------------------------------------
# per unit of the fp16 scale d: dmin (chosen so that the weights' mean is 0)
# and the standard deviation of a weight whose integer fields are uniform
DMIN = {Q2_K: 1.5, Q4_K: 7.5, Q5_K: 15.5}
UNIT = {Q4_0: 4.6, Q8_0: 74.0, Q2_K: 14.0, Q3_K: 43.0, Q4_K: 258.0, Q5_K: 525.0, Q6_K: 1366.0}


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _kquant(qt, M, K, g):
    """[M][row bytes] of random blocks on the GPU."""
    bw, bb = fm.GEOMETRY[qt]
    q = fm.base(qt)
    nb = M * (K // bw)
    w = torch.randint(0, 256, (nb, bb), dtype=torch.uint8, device="cuda", generator=g)
    d0 = max(6.5e-5 / 0.7, 1 / math.sqrt(K) / UNIT[q])     # at least fp16's smallest normal number
    d = torch.empty(nb, device="cuda").uniform_(0.7 * d0, 1.3 * d0, generator=g)
    for off, f in zip(fm.SCALE_FIELDS[q], (1.0, DMIN.get(q))):
        w[:, off:off + 2] = (d * f).half().view(torch.uint8).view(nb, 2)
    return w.view(M, (K // bw) * bb)


def _randn(shape, g, scale=1.0):
    return torch.randn(shape, device="cuda", generator=g) * scale


class _State:
    pass


def prepare(case, seed):
    g, c, s = _gen(seed), case, _State()
    s.case = c
    if c["kind"] == "matvec":
        s.W, s.x = _kquant(c["qt"], c["M"], c["K"], g), _randn(c["K"], g)
        s.y = torch.empty(c["M"], device="cuda")
    elif c["kind"] == "moe":
        _moe_state(s, c, g)
    else:
        _dense_state(s, c, g)
    return s


def _moe_state(s, c, g):
    H, F, E, T = c["H"], c["F"], c["E"], c["T"]
    s.router = _randn((E, H), g, ROUTER_STD)
    s.gate, s.up = _kquant(c["qg"], E * F, H, g), _kquant(c["qg"], E * F, H, g)
    s.down = _kquant(c["qd"], E * H, F, g)
    s.bias = None
    if c["zipf"]:   # log of a Zipf(1.1) expert popularity over a random ranking
        rank = torch.randperm(E, device="cuda", generator=g).double() + 1
        p = rank ** -1.1
        s.bias = (p / p.sum()).log().float()
    s.xn, s.resid = _randn((T, H), g), _randn((T, H), g)
    s.layer = tb.moe_layer(H, F, E, c["k"], c["qg"], s.router, s.gate, s.up, s.down, bias=s.bias, qt_down=c["qd"])
    s.ws = torch.zeros(tb.moe_workspace_size(s.layer, T, c["mode"]), dtype=torch.uint8, device="cuda")
    s.out = torch.empty((T, H), device="cuda")
    s.idx = torch.empty((T, 8), dtype=torch.int32, device="cuda")
    s.w = torch.empty((T, 8), device="cuda")


def _max_ctx(c):
    return (c["pos"] if c["kind"] == "decode" else c["pos0"] + c["T"]) // 128 * 128 + 128


def _dense_state(s, c, g):
    NL, H, F, D, NQ, NKV = c["layers"], c["hidden"], c["ffn"], c["dim"], c["heads"], c["kv"]
    norm = lambda n: 1 + _randn(n, g, 0.1)   # noqa: E731
    s.weights = []
    s.layers = (td.DenseLayer * NL)()
    for L in s.layers:
        t = dict(attn_norm=norm(H), q_norm=norm(D), k_norm=norm(D), ffn_norm=norm(H),
                 wqkv=_kquant(c["ql"], (NQ + 2 * NKV) * D, H, g), wo=_kquant(c["ql"], H, NQ * D, g),
                 wgu=_kquant(c["ql"], 2 * F, H, g), wdown=_kquant(c["qd"], H, F, g))
        s.weights.append(t)
        for k, v in t.items():
            setattr(L, k, v.data_ptr())
        L.qt_down = c["qd"]
    s.embd, s.out_norm = _kquant(c["qe"], c["vocab"], H, g), norm(H)
    ctx = _max_ctx(c)
    past = c["pos"] if c["kind"] == "decode" else c["pos0"]
    s.kc, s.vc = (torch.zeros((NL, NKV, ctx, D), device="cuda") for _ in range(2))
    for cache in (s.kc, s.vc):     # the rows of the positions before this call
        for l in range(NL):
            cache[l, :, :past] = _randn((NKV, past, D), g)
    s.model = td.DenseModel(NL, H, NQ, NKV, D, F, c["vocab"], ctx, NORM_EPS, ROPE_THETA, c["ql"], c["qe"],
                            s.embd.data_ptr(), s.embd.data_ptr(), s.out_norm.data_ptr(), s.layers, s.kc.data_ptr(),
                            s.vc.data_ptr())
    n = 1 if c["kind"] == "decode" else c["T"]
    s.tokens = torch.randint(0, c["vocab"], (n,), device="cuda", generator=g).to(torch.int32).cpu().numpy()
    lib = tb.lib()
    size = lib.tbq_dense_workspace_size(C.byref(s.model)) if c["kind"] == "decode" else \
        lib.tbq_dense_prefill_workspace_size(C.byref(s.model), n)
    s.ws = torch.empty(size, dtype=torch.uint8, device="cuda")
    s.logits = torch.empty(c["vocab"], device="cuda")


# ---- one pass ----------------------------------------------------------------
def run(s):
    c = s.case
    if c["kind"] == "matvec":
        return tb.matvec(s.W, c["qt"], c["M"], c["K"], s.x, s.y)
    if c["kind"] == "moe":
        tb.moe_forward(s.layer, c["T"], s.xn, s.resid, s.out, s.idx, s.w, s.ws, c["mode"])
        return {"out": s.out, "experts": s.idx, "weights": s.w}
    stream = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    args = (s.logits.data_ptr(), s.ws.data_ptr(), s.ws.numel(), stream)
    if c["kind"] == "decode":
        ok = tb.lib().tbq_dense_decode(C.byref(s.model), int(s.tokens[0]), c["pos"], *args)
    else:
        ok = tb.lib().tbq_dense_prefill(C.byref(s.model), s.tokens.ctypes.data, c["T"], c["pos0"], *args)
    if not ok:
        raise tb.TbqError(tb.lib().tbq_last_error().decode())
    return {"logits": s.logits, "k": s.kc, "v": s.vc}


# ---- what a pass cannot do without --------------------------------------------
def work(case):
    c = case
    if c["kind"] == "matvec":
        return {"bytes": fm.weight_bytes(c["qt"], c["M"], c["K"]) + 4 * (c["M"] + c["K"]), "flops": 2 * c["M"] * c["K"]}
    if c["kind"] == "moe":
        H, F, E, k, T = c["H"], c["F"], c["E"], c["k"], c["T"]
        used = E * (1 - (1 - k / E) ** T)    # experts that T tokens reach when the routing is even
        expert = 2 * fm.weight_bytes(c["qg"], F, H) + fm.weight_bytes(c["qd"], H, F)
        return {"bytes": used * expert + 4 * E * H + 12 * T * H + 64 * T, "flops": 2 * T * (k * 3 * H * F + E * H)}
    H, F, D, NQ, NKV, NL = c["hidden"], c["ffn"], c["dim"], c["heads"], c["kv"], c["layers"]
    QR = (NQ + 2 * NKV) * D
    T, past = (1, c["pos"]) if c["kind"] == "decode" else (c["T"], c["pos0"])
    layer = fm.weight_bytes(c["ql"], QR + 2 * F, H) + fm.weight_bytes(c["ql"], H, NQ * D) + fm.weight_bytes(c["qd"], H, F)
    kv = 2 * 4 * NKV * D * (past + T)
    seen = T * past + T * (T + 1) // 2       # (query, cached position) pairs of a causal prompt
    head = fm.weight_bytes(c["qe"], c["vocab"], H) + 4 * c["vocab"]
    flops = NL * (2 * T * (H * (QR + 2 * F) + NQ * D * H + F * H) + 4 * seen * NQ * D) + 2 * c["vocab"] * H
    return {"bytes": NL * (layer + kv) + head + T * fm.weight_bytes(c["qe"], 1, H), "flops": flops}


def tolerance(case):
    """About four times the distance from 64 bits that was measured: 5e-7 for a
    matvec, 8e-7 for a decode MoE layer, 5e-4 with fp16 and 3e-5 with two-level
    int8 operands in its prefill, 1e-5 for a decode step of 36 layers, 3e-3
    for the fp16 prefill of two.  Experts are the same ones.  "max" is wider
    where the new KV rows are few among the cached ones."""
    if case["kind"] == "matvec":
        return {"rel": 2e-6, "max": 4e-5}
    if case["kind"] == "moe":
        return {tb.TBQ_MOE_FP32: {"rel": 3e-6, "max": 6e-5}, tb.TBQ_MOE_BF16: {"rel": 2e-3, "max": 5e-2},
                tb.TBQ_MOE_I8: {"rel": 1e-4, "max": 4e-3}}[case["mode"]]
    return {"rel": 5e-5, "max": 2e-3} if case["kind"] == "decode" else {"rel": 1e-2, "max": 0.2}


# ---- the same in 64 bits -------------------------------------------------------
def _f16(b, off, qt):
    """The fp16 field at byte `off` of each block, in 64 bits (never subnormal here)."""
    return b[:, off:off + 2].contiguous().view(torch.float16).double()


def _bits(b, width):
    """Little-endian fields of `width` bits of each byte, in order: [n][bytes * 8 / width]."""
    n = 8 // width
    sh = torch.arange(n, device=b.device) * width
    return ((b.long().unsqueeze(-1) >> sh) & ((1 << width) - 1)).flatten(1)


def _planes(b, width, run):
    """Fields of `width` bits stored as planes: for every `run` bytes first
    their lowest fields, then their next ones, ..."""
    n = 8 // width
    v = b.long().view(b.shape[0], -1, 1, run) >> (torch.arange(n, device=b.device) * width).view(1, 1, n, 1)
    return (v & ((1 << width) - 1)).flatten(1)


def _scales45(b, qt):
    """The 8 scales and mins of Q4_K / Q5_K blocks, as each layout reads them."""
    s = b[:, 4:20].long()
    if qt & GGML:
        hi_s = (s[:, 8:12] & 15) | (s[:, 0:4] >> 6 << 4)
        hi_m = (s[:, 8:12] >> 4) | (s[:, 4:8] >> 6 << 4)
    elif fm.base(qt) == Q4_K:
        hi_s, hi_m = s[:, 8:12] & 63, s[:, 12:16] & 63
    else:
        hi_s = (s[:, 0:4] >> 6) | ((s[:, 8:12] & 15) << 2)
        hi_m = (s[:, 4:8] >> 6) | ((s[:, 12:16] & 15) << 2)
    return torch.cat([s[:, 0:4] & 63, hi_s], 1).double(), torch.cat([s[:, 4:8] & 63, hi_m], 1).double()


def _blocks64(b, qt):
    """Dequantised blocks [n][weights per block] in 64 bits, in the layout qt says."""
    q, gg = fm.base(qt), bool(qt & GGML)
    if q == Q8_0:
        return _f16(b, 0, qt) * b[:, 2:34].contiguous().view(torch.int8).double()
    if q == Q4_0:
        return _f16(b, 0, qt) * ((_planes(b[:, 2:18], 4, 16) if gg else _bits(b[:, 2:18], 4)) - 8).double()
    if q in (Q4_K, Q5_K):
        S, M = _scales45(b, qt)
        quants = b[:, 16:144] if q == Q4_K else b[:, 48:176]
        v = _planes(quants, 4, 32) if gg else _bits(quants, 4)
        if q == Q5_K:
            v = v + 16 * (_planes(b[:, 16:48], 1, 32) if gg else _bits(b[:, 16:48], 1))
        S, M = _f16(b, 0, qt) * S, _f16(b, 2, qt) * M
        return (S.unsqueeze(-1) * v.view(-1, 8, 32).double() - M.unsqueeze(-1)).flatten(1)
    if q == Q6_K:
        lo = _planes(b[:, 0:128], 4, 64) if gg else _bits(b[:, 0:128], 4)
        hi = _planes(b[:, 128:192], 2, 32) if gg else _bits(b[:, 128:192], 2)
        sc = b[:, 192:208].contiguous().view(torch.int8).double() * _f16(b, 208, qt)
        return (sc.unsqueeze(-1) * ((lo | hi << 4) - 32).view(-1, 16, 16).double()).flatten(1)
    if q == Q2_K:
        v = _planes(b[:, 16:80], 2, 32) if gg else _bits(b[:, 16:80], 2)
        S, M = _f16(b, 80, qt) * (b[:, :16] & 15).double(), _f16(b, 82, qt) * (b[:, :16] >> 4).double()
        return (S.unsqueeze(-1) * v.view(-1, 16, 16).double() - M.unsqueeze(-1)).flatten(1)
    if q == Q3_K:
        s = b[:, 96:108].long()
        if gg:
            lo = torch.cat([s[:, :8] & 15, s[:, :8] >> 4], 1)
            hi = torch.cat([(s[:, 8:12] >> sh) & 3 for sh in (0, 2, 4, 6)], 1)
            v = _planes(b[:, 32:96], 2, 32) + 4 * _planes(b[:, :32], 1, 32)
        else:   # 8 scales, used twice
            lo = _bits(b[:, 96:100], 4).repeat(1, 2)
            hi = _bits(b[:, 104:106], 2).repeat(1, 2)
            v = _bits(b[:, 32:96], 2) + 4 * _bits(b[:, :32], 1)
        S = _f16(b, 108, qt) * ((lo | hi << 4) - 32).double()
        return (S.unsqueeze(-1) * (v - 4).view(-1, 16, 16).double()).flatten(1)
    raise ValueError(qt)


def _rows64(W, qt, K):
    bw, bb = fm.GEOMETRY[qt]
    return _blocks64(W.view(-1, bb), qt).view(-1, K)


def _mul64(W, qt, K, x):
    """x [n][K] . W^T in 64 bits, some rows of W at a time."""
    step = max(1, (1 << 26) // K)
    return torch.cat([x @ _rows64(W[i:i + step], qt, K).t().contiguous() for i in range(0, W.shape[0], step)], 1)


def _silu(g):
    return g * torch.sigmoid(g)


def exact(case, seed):
    s, c = prepare(case, seed), case
    if c["kind"] == "matvec":
        return _mul64(s.W, c["qt"], c["K"], s.x.double()[None])[0]
    return _moe64(s, c) if c["kind"] == "moe" else _dense64(s, c)


def _moe64(s, c):
    H, F, E, k, T = c["H"], c["F"], c["E"], c["k"], c["T"]
    # the router's sums are defined as 32-bit ones in element order, so the
    # experts are theirs; everything after the selection is in 64 bits
    acc = torch.zeros((T, E), device="cuda")
    rt, xt = s.router.t().contiguous(), s.xn.t().contiguous()
    for h in range(H):
        acc += xt[h][:, None] * rt[h][None]
    if s.bias is not None:
        acc += s.bias
    p32 = torch.softmax(acc, 1)
    top = torch.topk(p32, k, 1).indices
    # slot order: a slot holds the expert that replaced the smallest so far
    idx = torch.full((T, 8), -1, dtype=torch.int32)
    rows, tops = p32.cpu().tolist(), top.cpu().tolist()
    for t in range(T):
        w, e8 = [-1e30] * k, [0] * k
        for e, v in enumerate(rows[t]):
            lo = min(range(k), key=w.__getitem__)
            if v > w[lo]:
                w[lo], e8[lo] = v, e
        assert set(e8) == set(tops[t]) or len(set(w)) < k
        idx[t, :k] = torch.tensor(e8, dtype=torch.int32)
    idx = idx.cuda()
    sel = idx[:, :k].long()
    p = torch.softmax(acc.double(), 1).gather(1, sel)
    wts = torch.zeros((T, 8), dtype=torch.float64, device="cuda")
    wts[:, :k] = p / p.sum(1, keepdim=True)
    out, x = s.resid.double().clone(), s.xn.double()
    gate, up, down = s.gate.view(E, F, -1), s.up.view(E, F, -1), s.down.view(E, H, -1)
    for e in range(E):
        t, slot = (sel == e).nonzero(as_tuple=True)
        if t.numel():
            a = _silu(_mul64(gate[e], c["qg"], H, x[t])) * _mul64(up[e], c["qg"], H, x[t])
            out.index_add_(0, t, _mul64(down[e], c["qd"], F, a) * wts[t, slot][:, None])
    return {"out": out, "experts": idx, "weights": wts}


def _dense64(s, c):
    H, F, D, NQ, NKV = c["hidden"], c["ffn"], c["dim"], c["heads"], c["kv"]
    n, past = (1, c["pos"]) if c["kind"] == "decode" else (c["T"], c["pos0"])
    rms = lambda v, w: v * torch.rsqrt((v * v).mean(-1, keepdim=True) + NORM_EPS) * w.double()   # noqa: E731
    pos = torch.arange(past, past + n, device="cuda", dtype=torch.float64)
    j = torch.arange(D // 2, device="cuda", dtype=torch.float64)
    ang = pos[:, None] * ROPE_THETA ** (-2 * j / D)
    cos, sin = ang.cos()[:, None], ang.sin()[:, None]

    def rope(v):   # [n][heads][D], rotated by halves
        a, b = v[..., :D // 2], v[..., D // 2:]
        return torch.cat([a * cos - b * sin, a * sin + b * cos], -1)

    toks = torch.from_numpy(s.tokens).long().cuda()
    x = _rows64(s.embd[toks].contiguous(), c["qe"], H)
    kc, vc = s.kc.double(), s.vc.double()
    hidden_keys = torch.arange(past + n, device="cuda")[None] > pos[:, None]
    for l, t in enumerate(s.weights):
        qkv = _mul64(t["wqkv"], c["ql"], H, rms(x, t["attn_norm"])).view(n, NQ + 2 * NKV, D)
        q = rope(rms(qkv[:, :NQ], t["q_norm"]))
        kc[l, :, past:past + n] = rope(rms(qkv[:, NQ:NQ + NKV], t["k_norm"])).transpose(0, 1)
        vc[l, :, past:past + n] = qkv[:, NQ + NKV:].transpose(0, 1)
        att = torch.empty((n, NQ, D), dtype=torch.float64, device="cuda")
        for h in range(NQ):
            g = h // (NQ // NKV)
            sc = q[:, h].contiguous() @ kc[l, g, :past + n].t().contiguous() / math.sqrt(D)
            att[:, h] = torch.softmax(sc.masked_fill(hidden_keys, -math.inf), -1) @ vc[l, g, :past + n].contiguous()
        x = x + _mul64(t["wo"], c["ql"], NQ * D, att.view(n, NQ * D))
        gu = _mul64(t["wgu"], c["ql"], H, rms(x, t["ffn_norm"]))
        x = x + _mul64(t["wdown"], c["qd"], F, _silu(gu[:, :F]) * gu[:, F:])
    logits = _mul64(s.embd, c["qe"], H, rms(x[-1:], s.out_norm))[0]
    return {"logits": logits, "k": kc, "v": vc}
