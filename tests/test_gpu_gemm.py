"""The batched prefill's GEMM (tbq_gemm, csrc/tbq_gemm.hip): a hand-written
fp16 MFMA kernel with fp32 accumulation, for W as fp16 halves or as Q4_K
rows dequantised inside the kernel.

* fp16 W: against a torch fp32 product of the same fp16 values (only the
  summation order differs), over tile edges (T and N not multiples of a
  tile), a row stride ldc > N and the split-K shapes (partial sums added in
  slice order).
* Q4_K W: close to the fp16 path on the fp16 values of the oracle's
  dequantised weights (the kernel's packed fp16 decode rounds 16 S, M and
  S q - M to fp16, about one fp16 ulp per weight), and to the fp64 product
  of the exact weights.
"""
import numpy as np
import pytest

import trailblaze_amd as tb
from trailblaze_amd import formats as fm, synth

from conftest import rel_l2

pytestmark = pytest.mark.gpu


def _dev(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def _x16(T, K, rng):
    return (rng.standard_normal((T, K)) * 4).astype(np.float16)


@pytest.mark.parametrize("T,N,K,ldc", [
    (2, 128, 256, 0),
    (37, 200, 512, 0),          # partial tiles in t and n
    (300, 640, 2560, 0),
    (512, 2560, 4096, 0),       # split K (80 tiles)
    (512, 2560, 9728, 2688),    # split K, row stride above N
    (130, 6144, 2560, 0),
])
def test_gemm_f16_matches_torch(T, N, K, ldc):
    import torch
    rng = np.random.default_rng(T + N + K)
    X = _x16(T, K, rng)
    W = (rng.standard_normal((N, K)) * 0.05).astype(np.float16)
    print("gemm f16", T, N, K, ldc, flush=True)
    ld = ldc or N
    C = torch.full((T, ld), 7.0, dtype=torch.float32, device="cuda")
    tb.gemm(_dev(W), 1, _dev(X), T, N, K, C, ldc=ld)
    got = C.cpu().numpy()
    ref = (torch.from_numpy(X.astype(np.float32)).double() @ torch.from_numpy(W.astype(np.float32)).double().T).numpy()
    assert rel_l2(got[:, :N], ref) <= 1e-6
    if ld > N:   # columns past N untouched
        assert np.all(got[:, N:] == 7.0)


@pytest.mark.parametrize("T,N,K", [(3, 256, 512), (512, 2560, 2560), (200, 768, 4096)])
def test_gemm_q4k_fused_matches_f16_path(oracle, T, N, K):
    import torch
    rng = np.random.default_rng(N + K)
    Wq = synth.kquant_matrix(fm.Q4_K, N, K, rng)
    X = _x16(T, K, rng)
    wf = oracle.dequant_rows(Wq, fm.Q4_K, N, K)              # the reference's fp32 weights
    w16 = wf.astype(np.float16)                              # rounded once, as the prefill's fp16 weights
    print("gemm q4k", T, N, K, flush=True)
    Cq = torch.empty((T, N), dtype=torch.float32, device="cuda")
    Cf = torch.empty((T, N), dtype=torch.float32, device="cuda")
    tb.gemm(_dev(Wq), fm.Q4_K, _dev(X), T, N, K, Cq)
    tb.gemm(_dev(w16), 1, _dev(X), T, N, K, Cf)
    a, b = Cq.cpu().numpy(), Cf.cpu().numpy()
    assert rel_l2(a, b) <= 1e-3
    ref = X.astype(np.float64) @ wf.astype(np.float64).T
    assert rel_l2(a, ref) <= 1e-3   # fp16 rounding of the weights
    assert rel_l2(b, ref) <= 1e-3


# Ragged T and N around 32 to 256, one super-block, uneven slices.  The launch's
# cost rule takes small tiles for nearly all of these; test_gemm_tiles.py goes
# through every tile.
@pytest.mark.parametrize("T,N,K", [
    (1, 4, 256), (31, 124, 512), (33, 132, 256), (64, 260, 8192), (65, 1028, 2304), (127, 256, 5120),
    (129, 6148, 768), (257, 516, 1792), (513, 3076, 256), (1030, 5124, 512),
])
def test_gemm_tile_edges(oracle, T, N, K):
    import torch
    rng = np.random.default_rng(T * 7 + N + K)
    Wq = synth.kquant_matrix(fm.Q4_K, N, K, rng)
    wf = oracle.dequant_rows(Wq, fm.Q4_K, N, K)
    w16 = wf.astype(np.float16)
    X = _x16(T, K, rng)
    x64 = torch.from_numpy(X).cuda().double()
    prod = lambda w: (x64 @ _dev(w).double().t().contiguous()).cpu().numpy()   # noqa: E731
    for qt, W, ref, tol in ((fm.F16, w16, prod(w16), 1e-6), (fm.Q4_K, Wq, prod(wf), 1e-3)):
        print("gemm edges", T, N, K, fm.NAMES[qt], flush=True)
        C = torch.full((T + 1, N), 7.0, dtype=torch.float32, device="cuda")
        tb.gemm(_dev(W), qt, _dev(X), T, N, K, C)
        got = C.cpu().numpy()
        assert rel_l2(got[:T], ref) <= tol            # fp32 sums; fp16 rounding of the decoded weights
        assert np.abs(got[:T] - ref).max() <= 20 * tol * np.sqrt(np.mean(ref ** 2)) # no single row or column off
        assert np.all(got[T] == 7.0)                  # nothing past the last row


def test_gemm_rejects_bad_shapes():
    import torch
    X = torch.zeros((4, 256), dtype=torch.float16, device="cuda")
    W = torch.zeros((8, 256), dtype=torch.float16, device="cuda")
    C = torch.zeros((4, 8), dtype=torch.float32, device="cuda")
    with pytest.raises(tb.TbqError):
        tb.gemm(W, 1, X, 4, 6, 256, C)      # N not a multiple of 4
    with pytest.raises(tb.TbqError):
        tb.gemm(W, 1, X, 4, 8, 200, C)      # K not a multiple of 256
    with pytest.raises(tb.TbqError):
        tb.gemm(W, 10, X, 4, 8, 256, C)     # Q2_K weights: not this kernel's
