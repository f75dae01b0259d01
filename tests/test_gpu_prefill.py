"""GPU parity of tbq_dense_prefill, the batched prefill of a dense
Qwen3-style model (T prompt tokens per layer pass; the reference prefills
token by token, layer4/tb_infer.c:1068-1075), through the C-ABI:
  * batched path (any format or layout; fused or separate matrices): the
    last token's logits and the K/V cache
    rows of every prompt position within PREFILL_TOL of the float64 oracle
    run token by token, and of libtbq's own decode steps; prompts of 1, 7,
    130 and 300 tokens, from an empty cache and after decoded tokens, head_dim
    64 and 128, GQA 2, 4, 8 (the GEMMs' tiles: test_gemm_tiles.py);
  * a one-token prefill is the decode step itself (bit-identical);
  * argument checks."""
import numpy as np
import pytest

import trailblaze_amd as tb
from conftest import bits_equal, rel_l2
from gpu_util import host
from trailblaze_amd import formats as fm

pytestmark = pytest.mark.gpu
# fp16-operand MFMA GEMMs (fp32 accumulate) against float64
PREFILL_TOL = 1e-2


@pytest.fixture(scope="module", autouse=True)
def _init():
    print("device:", tb.init(), flush=True)


def _cfg(**kw):
    from trailblaze_amd.dense import DenseConfig
    base = dict(n_layers=2, hidden=256, n_heads=4, n_kv_heads=2, head_dim=64, ffn=512, vocab=512, max_ctx=512)
    base.update(kw)
    return DenseConfig(**base)


def _check_prefill(oracle, cfg, seed, tokens, pre=()):
    """Decode `pre` token by token, then prefill `tokens`; compare with the
    oracle over pre + tokens and with libtbq's decode steps."""
    import torch
    from oracle.dense import DenseOracle
    from trailblaze_amd.dense import SyntheticDense
    m = SyntheticDense(cfg, seed, keep_host=True)
    seq = SyntheticDense(cfg, seed)
    assert m.prefill_batched()
    ref = DenseOracle(oracle, cfg, m.host)
    logits = torch.empty(cfg.vocab, dtype=torch.float32, device="cuda")
    for pos, tok in enumerate(pre):
        m.decode(tok, pos, logits)
    print("prefill T=", len(tokens), "pos0=", len(pre), flush=True)
    m.prefill(tokens, len(pre), logits)
    got = host(logits)
    want = None
    for pos, tok in enumerate(list(pre) + list(tokens)):
        want = ref.decode(tok, pos)
    for pos, tok in enumerate(list(pre) + list(tokens)):
        seq.decode(tok, pos, logits)
    assert rel_l2(got, want) <= PREFILL_TOL
    assert rel_l2(got, host(logits)) <= PREFILL_TOL
    n = len(pre) + len(tokens)
    kc = host(m.k_cache).reshape(ref.kc.shape)
    vc = host(m.v_cache).reshape(ref.vc.shape)
    assert rel_l2(kc[:, :, :n], ref.kc[:, :, :n]) <= PREFILL_TOL
    assert rel_l2(vc[:, :, :n], ref.vc[:, :, :n]) <= PREFILL_TOL
    assert not np.any(kc[:, :, n:])


@pytest.mark.parametrize("T", [1, 7, 130])
def test_prefill_from_empty_cache(oracle, T):
    rng = np.random.default_rng(T)
    _check_prefill(oracle, _cfg(), 41, rng.integers(0, 512, T))


def test_prefill_after_decoded_tokens(oracle):
    rng = np.random.default_rng(9)
    _check_prefill(oracle, _cfg(), 42, rng.integers(0, 512, 40), pre=[3, 99, 511, 0, 17])


@pytest.mark.parametrize("G", [4, 8])
def test_prefill_head_dim_128(oracle, G):
    rng = np.random.default_rng(G)
    cfg = _cfg(n_layers=1, hidden=512, n_heads=8, n_kv_heads=8 // G, head_dim=128, ffn=768, vocab=256)
    _check_prefill(oracle, cfg, 43, rng.integers(0, 256, 300))


@pytest.mark.parametrize("G", [1, 2])
def test_prefill_long_context_many_splits(oracle, G):
    """A 100-token prompt after 1100 cached positions (N(0,1) K/V in the
    cache and in the oracle): the attention runs over 8 position splits of
    more than 128 positions each, then merges them."""
    import torch
    from oracle.dense import DenseOracle
    from trailblaze_amd.dense import SyntheticDense
    cfg = _cfg(n_layers=1, n_heads=4, n_kv_heads=4 // G, max_ctx=1536, vocab=256)
    m = SyntheticDense(cfg, 46, keep_host=True)
    ref = DenseOracle(oracle, cfg, m.host)
    rng = np.random.default_rng(12)
    P = 1100
    kc = np.zeros(ref.kc.shape, np.float32)
    vc = np.zeros(ref.vc.shape, np.float32)
    kc[:, :, :P] = rng.standard_normal(kc[:, :, :P].shape)
    vc[:, :, :P] = rng.standard_normal(vc[:, :, :P].shape)
    m.k_cache.copy_(torch.from_numpy(kc))
    m.v_cache.copy_(torch.from_numpy(vc))
    ref.kc[:] = kc
    ref.vc[:] = vc
    toks = rng.integers(0, 256, 100)
    logits = torch.empty(cfg.vocab, dtype=torch.float32, device="cuda")
    print("prefill long context G=", G, flush=True)
    m.prefill(toks, P, logits)
    for i, tok in enumerate(toks):
        want = ref.decode(tok, P + i)
    assert rel_l2(host(logits), want) <= PREFILL_TOL
    kcg = host(m.k_cache).reshape(ref.kc.shape)
    assert rel_l2(kcg[:, :, P:P + 100], ref.kc[:, :, P:P + 100]) <= PREFILL_TOL


@pytest.mark.parametrize("D,G,P,T", [(64, 1, 0, 64), (64, 2, 63, 2), (64, 8, 64, 65), (128, 4, 127, 33), (128, 1, 1, 63),
                                     (128, 8, 200, 17), (128, 2, 690, 131)])
def test_prefill_attention_edges(oracle, D, G, P, T):
    """Query blocks and position chunks on either side of their 64-position
    edges, one and several splits, after P cached N(0,1) K/V rows: the second
    layer's K/V rows of every prompt position depend on its own attention."""
    import torch
    from oracle.dense import DenseOracle
    from trailblaze_amd.dense import SyntheticDense
    cfg = _cfg(n_layers=2, n_heads=8, n_kv_heads=8 // G, head_dim=D, max_ctx=P + T + 5, vocab=256)
    m = SyntheticDense(cfg, 50, keep_host=True)
    ref = DenseOracle(oracle, cfg, m.host)
    rng = np.random.default_rng(P + T)
    for dev, cache in ((m.k_cache, ref.kc), (m.v_cache, ref.vc)):
        cache[:, :, :P] = rng.standard_normal(cache[:, :, :P].shape).astype(np.float32)
        dev.copy_(torch.from_numpy(cache.astype(np.float32)))
    toks = rng.integers(0, 256, T)
    logits = torch.empty(cfg.vocab, dtype=torch.float32, device="cuda")
    print("prefill attention edges", D, G, P, T, flush=True)
    m.prefill(toks, P, logits)
    for i, tok in enumerate(toks):
        want = ref.decode(tok, P + i)
    assert rel_l2(host(logits), want) <= PREFILL_TOL
    for dev, cache in ((m.k_cache, ref.kc), (m.v_cache, ref.vc)):
        got = host(dev).reshape(cache.shape)
        for p in range(P, P + T):
            assert rel_l2(got[1, :, p], cache[1, :, p]) <= PREFILL_TOL, p
        assert np.array_equal(got[:, :, :P], cache[:, :, :P].astype(np.float32)) and not np.any(got[:, :, P + T:])


@pytest.mark.parametrize("D,G,P", [(64, 4, 0), (128, 4, 10), (128, 8, 0), (64, 2, 5)])
def test_prefill_nan_token_stays_in_its_block(D, G, P):
    """A token whose embedding holds a NaN leaves the tokens of earlier query
    blocks (128 / G tokens each) as they are, bit for bit, though it shares a
    chunk of 64 positions with them."""
    import torch
    from trailblaze_amd.dense import SyntheticDense
    QB = 128 // G
    bad, T = QB + 3, QB + 20
    cfg = _cfg(n_heads=8, n_kv_heads=8 // G, head_dim=D, vocab=256, qtype_embd=fm.F32)
    rng = np.random.default_rng(D + G)
    toks = rng.integers(0, 255, P + T)
    logits = torch.empty(cfg.vocab, dtype=torch.float32, device="cuda")
    rows = []
    for nan in (False, True):
        m = SyntheticDense(cfg, 60)
        if nan:
            m.lm_head.view(torch.float32).view(256, -1)[255, 7] = float("nan")
        t = toks.copy()
        t[P + bad] = 255
        for pos in range(P):
            m.decode(int(t[pos]), pos, logits)
        print("prefill nan token", D, G, P, nan, flush=True)
        m.prefill(t[P:], P, logits)
        rows.append([host(c).reshape(2, 8 // G, cfg.max_ctx, D)[:, :, :P + T] for c in (m.k_cache, m.v_cache)])
    for a, b in zip(*rows):
        assert np.all(np.isnan(b[0, :, P + bad])) and np.all(np.isfinite(a))
        assert bits_equal(a[:, :, :P + QB], b[:, :, :P + QB])


@pytest.mark.parametrize("seed", [1, 2, 3])
def test_prefill_attention_heaviest_weight_is_exact(oracle, seed):
    """The softmax's running max is the exact one, so a position that holds
    most of a query's weight has probability 1 and no fp16 rounding.  Position
    90 scores 5 above position 20, the highest of the first chunk (N(0,1)
    scores otherwise): 0.993 of the weight.  The relative error of that weight
    is read per head off the next layer's V row: the row's error projected on
    its derivatives by the heads' cached V vectors (fp16 weights and no FFN
    output, so little else rounds).  A running max that may stay behind by up
    to 2^8 leaves the position some probability in [1, 256), whose fp16
    rounding has an RMS of 2.1e-4; the roundings of the other operands (each
    2^-11 / sqrt(12) an element, projected on 128 dimensions a head) leave 7e-5
    to 1e-4."""
    import torch
    from oracle.dense import DenseOracle, rmsnorm, rope
    from trailblaze_amd.dense import SyntheticDense
    NH, D, P, A, B = 8, 128, 100, 20, 90
    cfg = _cfg(hidden=1024, n_heads=NH, n_kv_heads=NH, head_dim=D, max_ctx=128, vocab=256, qtype_layers=fm.F16,
               qtype_embd=fm.F16)
    m = SyntheticDense(cfg, seed, keep_host=True)
    for name, by in (("wdown", 0), ("wo", 2.0 ** -9)):   # the attention's output as large as the embedding beside it
        for w in (m._keep[0][name].view(torch.float16), m.host["layers"][0][name].view(np.float16)):
            w *= by
    ref = DenseOracle(oracle, cfg, m.host)
    rng = np.random.default_rng(seed)
    toks = rng.integers(0, 256, 2)
    L = ref.layers[0]
    q = (L["wqkv"][:NH * D] @ rmsnorm(ref.lm[toks[1]], L["attn_norm"], cfg.norm_eps)).reshape(NH, D)
    q = np.stack([rope(rmsnorm(v, L["q_norm"], cfg.norm_eps), P + 1, cfg.rope_theta) for v in q])
    for cache, dev in ((ref.kc, m.k_cache), (ref.vc, m.v_cache)):
        cache[:, :, :P] = rng.standard_normal(cache[:, :, :P].shape)
        if cache is ref.kc:
            for at, score in ((A, 12), (B, 17)):
                cache[0, :, at] = q * (score * np.sqrt(D) / np.sum(q * q, axis=1))[:, None]
        else:
            cache[0, :, B] *= 16
        cache[:] = cache.astype(np.float32)
        dev.copy_(torch.from_numpy(cache.astype(np.float32)))
    logits = torch.empty(cfg.vocab, dtype=torch.float32, device="cuda")
    print("prefill heaviest weight", seed, flush=True)
    m.prefill(toks, P, logits)
    ref.decode(toks[0], P)

    def v_row(h=None, by=0.0):
        if h is not None:
            ref.vc[0, h, B] *= 1 + by
        ref.decode(toks[1], P + 1)
        if h is not None:
            ref.vc[0, h, B] /= 1 + by
        return ref.vc[1, :, P + 1].flatten().copy()

    want = v_row()
    by = 1e-4
    U = np.stack([(v_row(h, by) - want) / by for h in range(NH)], 1)
    e = host(m.v_cache).reshape(ref.vc.shape)[1, :, P + 1].flatten() - want
    c = np.linalg.lstsq(U, e, rcond=None)[0]
    print(c, flush=True)
    assert np.sqrt(np.mean(c * c)) <= 1.4e-4


@pytest.mark.parametrize("ql,qe", [(fm.Q8_0, fm.Q6_K), (fm.Q5_K, fm.Q8_0), (fm.GGML | fm.Q4_K, fm.GGML | fm.Q6_K),
                                   (fm.GGML | fm.Q3_K, fm.Q4_K)])
def test_prefill_other_formats(oracle, ql, qe):
    """Layer matrices of every format and either layout take the batched
    path (each matrix dequantised to fp16 before its GEMM)."""
    rng = np.random.default_rng(ql)
    _check_prefill(oracle, _cfg(qtype_layers=ql, qtype_embd=qe, vocab=256), 47, rng.integers(0, 256, 70))


def test_prefill_separate_matrices(oracle):
    """A mixed-quant layer (separate q, k, v and gate, up matrices of
    different formats, as a GGUF file assembles them) on the batched path."""
    import torch
    from gguf_write import dense_gguf_tensors, write_gguf
    from oracle.dense import DenseOracle
    from trailblaze_amd import synth
    from trailblaze_amd.gguf import GgufFile, dense_prefill
    cfg = _cfg(n_layers=1, vocab=256, max_ctx=128)
    r = np.random.default_rng(48)
    norm = lambda n: (1.0 + 0.1 * r.standard_normal(n)).astype(np.float32)
    mat = lambda qt, M, K: synth.kquant_matrix(qt, M, K, r)
    l0 = {"attn_norm": norm(256), "q_norm": norm(64), "k_norm": norm(64), "ffn_norm": norm(256),
          "wq": mat(fm.Q4_K, 256, 256), "wk": mat(fm.Q4_K, 128, 256), "wv": mat(fm.Q6_K, 128, 256),
          "qt_wq": fm.Q4_K, "qt_wk": fm.Q4_K, "qt_wv": fm.Q6_K, "wo": mat(fm.Q5_K, 256, 256), "qt_wo": fm.Q5_K,
          "wgate": mat(fm.Q4_K, 512, 256), "wup": mat(fm.Q8_0, 512, 256), "qt_wgate": fm.Q4_K, "qt_wup": fm.Q8_0,
          "wdown": mat(fm.Q6_K, 256, 512), "qt_wdown": fm.Q6_K}
    hostd = {"layers": [l0], "lm_head": mat(fm.Q6_K, 256, 256), "output_norm": norm(256)}
    kv, ts = dense_gguf_tensors(cfg, hostd)
    import tempfile, os
    with tempfile.TemporaryDirectory() as d:
        path = os.path.join(d, "mixed.gguf")
        write_gguf(path, kv, ts)
        ref = DenseOracle(oracle, cfg, hostd)
        with GgufFile(path) as g:
            m, ws = g.dense_model(cfg.max_ctx)
            assert not m.layers[0].wqkv and not m.layers[0].wgu
            toks = r.integers(0, 256, 50)
            logits = torch.empty(cfg.vocab, dtype=torch.float32, device="cuda")
            print("prefill separate matrices", flush=True)
            dense_prefill(m, toks, 0, logits)
            for pos, tok in enumerate(toks):
                want = ref.decode(tok, pos)
            assert rel_l2(host(logits), want) <= PREFILL_TOL


@pytest.mark.parametrize("short_by", [0, 1, 1 << 20])
def test_prefill_workspace_of_a_longer_prompt(short_by):
    """A buffer for 512 tokens serves 480 of them bit for bit as their own
    does; one with less room for split-K partial sums takes fewer slices."""
    import ctypes as C
    import torch
    from trailblaze_amd.dense import SyntheticDense
    m = SyntheticDense(_cfg(n_layers=1, hidden=1024, n_heads=8, n_kv_heads=4, head_dim=128, ffn=2048), 71)
    lib, T = tb.lib(), 480
    toks = np.random.default_rng(4).integers(0, 512, T).astype(np.int32)
    logits = torch.empty((2, 512), dtype=torch.float32, device="cuda")
    own = int(lib.tbq_dense_prefill_workspace_size(C.byref(m.model), T))
    for i, n in enumerate((own, own - short_by if short_by else
                           int(lib.tbq_dense_prefill_workspace_size(C.byref(m.model), 512)))):
        print("prefill workspace", short_by, n, flush=True)
        ws = torch.empty(n, dtype=torch.uint8, device="cuda")
        assert lib.tbq_dense_prefill(C.byref(m.model), toks.ctypes.data, T, 0, logits[i].data_ptr(), ws.data_ptr(), n,
                                     C.c_void_p(torch.cuda.current_stream().cuda_stream))
        torch.cuda.synchronize()
    a, b = host(logits).reshape(2, 512)
    if short_by:
        assert rel_l2(b, a) <= 2e-3   # the same fp16 operands, other fp32 sums rounded to fp16 again
    else:
        assert bits_equal(a, b)


def test_prefill_one_token_is_the_decode_step():
    """T = 1 runs the decode step itself: the same logits and cache bits."""
    import torch
    from trailblaze_amd.dense import SyntheticDense
    cfg = _cfg(max_ctx=64)
    a, b = SyntheticDense(cfg, 44), SyntheticDense(cfg, 44)
    la = torch.empty(cfg.vocab, dtype=torch.float32, device="cuda")
    lb = torch.empty(cfg.vocab, dtype=torch.float32, device="cuda")
    a.decode(7, 0, la)
    b.decode(7, 0, lb)
    a.prefill([500], 1, la)
    b.decode(500, 1, lb)
    assert bits_equal(host(la), host(lb))
    assert bits_equal(host(a.k_cache), host(b.k_cache)) and bits_equal(host(a.v_cache), host(b.v_cache))


def test_prefill_rejects_bad_arguments():
    import torch
    from trailblaze_amd.dense import SyntheticDense
    m = SyntheticDense(_cfg(max_ctx=32), 45)
    logits = torch.empty(512, dtype=torch.float32, device="cuda")
    for toks, pos0, what in (([], 0, "T="), ([1] * 30, 3, "positions"), ([1, 512], 0, "out of range"),
                             ([1, -1], 0, "out of range")):
        with pytest.raises(tb.TbqError, match=what):
            m.prefill(toks, pos0, logits)
