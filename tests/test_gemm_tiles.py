"""Every tile of the batched prefill's GEMM (csrc/tbq_gemm.hip), with and
without split K and with SwiGLU in the epilogue: the launch chooses the tile
by a cost rule, so each shape here is first checked to take the tile that it
is listed for (tbq_gemm_plan, on the CPU for 256 compute units)."""
import ctypes as C

import numpy as np
import pytest

import trailblaze_amd as tb
from conftest import rel_l2
from trailblaze_amd import formats as fm, synth

F16_TILES = {(256, 256), (128, 128), (128, 64)}
Q4K_TILES = {(256, 128), (128, 128), (256, 64), (128, 64), (128, 32)}

# (tile rows, tile tokens, split K?, T, N, K): T and N off the tile's multiples,
# on both sides of them, down to one super-block of columns
GEMM = {
    fm.F16: [(256, 256, False, 513, 20484, 256), (256, 256, False, 1999, 4100, 768), (256, 256, True, 1000, 4100, 2560),
             (256, 256, True, 1025, 4092, 4096), (128, 128, False, 200, 8196, 512), (128, 128, False, 513, 8196, 256),
             (128, 128, True, 65, 8196, 1024), (128, 64, False, 17, 132, 256), (128, 64, True, 63, 124, 512)],
    fm.Q4_K: [(256, 128, False, 1999, 8188, 256), (256, 128, False, 1999, 2052, 512), (256, 128, False, 255, 16388, 512),
              (256, 128, True, 200, 4100, 2560), (128, 128, False, 1500, 2052, 2048), (128, 128, True, 1500, 1028, 2560),
              (256, 64, False, 17, 132, 256), (256, 64, True, 65, 260, 512), (128, 64, False, 1999, 516, 768),
              (128, 64, True, 513, 1300, 2560), (128, 32, False, 767, 2564, 1024), (128, 32, True, 700, 1300, 2560)],
}
# (tile rows, tile tokens, T, F, H): the product of 2 F rows with SwiGLU
GLU = {
    fm.F16: [(256, 256, 1500, 2816, 768), (128, 128, 383, 2816, 768), (128, 64, 17, 256, 256), (128, 64, 65, 512, 256)],
    fm.Q4_K: [(256, 128, 1025, 2048, 512), (256, 128, 129, 11264, 768), (128, 128, 1025, 1024, 2560), (256, 64, 17, 256, 256),
              (128, 64, 17, 256, 768), (128, 32, 17, 256, 1024)],
}


def _plan(qt, T, N, K, glu=0):
    p = (C.c_int * 3)()
    assert tb.lib().tbq_gemm_plan(qt, T, N, K, glu, p) == 1
    return p[0], p[1], p[2]


def test_shapes_take_the_tiles_they_are_listed_for():
    for qt, tiles in ((fm.F16, F16_TILES), (fm.Q4_K, Q4K_TILES)):
        for rows, tok, split, T, N, K in GEMM[qt]:
            r, t, s = _plan(qt, T, N, K)
            assert (r, t, s > 1) == (rows, tok, split), (qt, T, N, K, r, t, s)
        assert {c[:3] for c in GEMM[qt]} == {(*t, s) for t in tiles for s in (False, True)}
        for rows, tok, T, F, H in GLU[qt]:
            assert _plan(qt, T, 2 * F, H, 1) == (rows, tok, 1), (qt, T, F, H)
        assert {c[:2] for c in GLU[qt]} == tiles
    assert tb.lib().tbq_gemm_plan(fm.Q4_K, 16, 64, 100, 0, (C.c_int * 3)()) == 0


def _dev(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


@pytest.mark.gpu
@pytest.mark.parametrize("qt,case", [(qt, c) for qt in GEMM for c in GEMM[qt]])
def test_gemm_tile(oracle, qt, case):
    """Against the 64-bit product: fp32 sums for fp16 rows, the decode's fp16
    roundings of 16 S, C and the weight besides for Q4_K; no row, column or
    token off by more than that, and nothing written past the last token."""
    import torch
    rows, tok, split, T, N, K = case
    r, t, s = _plan(qt, T, N, K)
    assert (r, t, s > 1) == (rows, tok, split)
    rng = np.random.default_rng(T + N + K)
    if qt == fm.Q4_K:
        W = synth.kquant_matrix(qt, N, K, rng)
        w = oracle.dequant_rows(W, qt, N, K)
    else:
        W = w = (rng.standard_normal((N, K)) * 0.05).astype(np.float16)
    X = (rng.standard_normal((T, K)) * 4).astype(np.float16)
    print("gemm tile", fm.NAMES[qt], case, s, flush=True)
    ldc = N + 4 * (T % 2) * (not split)   # a row stride above N too
    out = torch.full((T + 1, ldc), 7.0, dtype=torch.float32, device="cuda")
    tb.gemm(_dev(W), qt, _dev(X), T, N, K, out, ldc=ldc)
    ref = _dev(X).double() @ _dev(w).double().t().contiguous()
    assert bool((out[T] == 7.0).all()) and bool((out[:T, N:] == 7.0).all())
    d = out[:T, :N].double() - ref
    tol, rms = (1e-6 if qt == fm.F16 else 1e-3), float(ref.square().mean().sqrt())
    assert float(d.norm() / ref.norm()) <= tol
    assert float(d.abs().max()) <= 20 * tol * rms
    for axis in (0, 1):
        assert float(d.square().mean(axis).sqrt().max()) <= 8 * tol * rms


@pytest.mark.gpu
@pytest.mark.parametrize("qt,case", [(qt, c) for qt in GLU for c in GLU[qt]])
def test_glu_tile(qt, case):
    """A prefill whose gate|up matrix is fused (SwiGLU in the epilogue, on the
    listed tile) against the same weights given as two matrices (two products,
    pinned above, and a SwiGLU kernel): the second layer's K and V rows of
    every token.  Other fp32 sums only, so a few fp16 operands round the other
    way; a wrong pairing of gate and up rows is off by the rows' own size."""
    import torch
    from gpu_util import host
    from trailblaze_amd.dense import DenseConfig, SyntheticDense
    rows, tok, T, F, H = case
    assert _plan(qt, T, 2 * F, H, 1)[:2] == (rows, tok)
    ql = fm.Q4_K if qt == fm.Q4_K else fm.Q8_0
    cfg = DenseConfig(n_layers=2, hidden=H, n_heads=4, n_kv_heads=4, head_dim=64, ffn=F, vocab=256, max_ctx=T,
                      qtype_layers=ql, qtype_embd=fm.Q8_0)
    toks = np.random.default_rng(T).integers(0, 256, T)
    m = SyntheticDense(cfg, 80)
    logits = torch.empty((2, 256), dtype=torch.float32, device="cuda")
    got = []
    for fused in (True, False):
        if not fused:
            for L in m.layers:
                L.wgate, L.wup, L.wgu = L.wgu, L.wgu + F * fm.row_bytes(ql, H), None
        m.k_cache.zero_()
        m.v_cache.zero_()
        print("glu tile", fm.NAMES[qt], case, fused, flush=True)
        m.prefill(toks, 0, logits[int(fused)])
        got.append([host(c).reshape(2, 4, T, 64).copy() for c in (m.k_cache, m.v_cache)])
    for a, b in zip(*got):
        assert np.all(np.isfinite(a)) and rel_l2(a[0], b[0]) == 0
        d = np.linalg.norm(a[1] - b[1], axis=(0, 2)) / np.linalg.norm(b[1], axis=(0, 2))
        assert d.max() <= 1e-3
    assert rel_l2(host(logits[1]), host(logits[0])) <= 1e-3
