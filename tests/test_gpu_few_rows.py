"""Projections of two to eight rows, on both sides of the limits that choose their kernel (kh_gemm_ex)."""
import numpy as np
import pytest

from kandle_amd import Tensor, synthetic as syn
from kandle_amd import functional as F

pytestmark = pytest.mark.gpu


# A single step of k and less, a k that is not a multiple of 8 (no tiles), columns around a tile; 64 KiB of
# fp32 rows (8 x 2048, 2 x 8192) and the next k, a row that is longer than that by itself, and one past the
# one-row kernel's limit of 32768.
@pytest.mark.parametrize("N,K", [(37, 8), (130, 40), (33, 20), (65, 520), (300, 2048), (300, 2056), (64, 8192),
                                 (100, 8200), (40, 16392), (24, 32776)])
@pytest.mark.parametrize("M", [2, 3, 7, 8])
@pytest.mark.parametrize("act,out", [("bfloat16", "bfloat16"), ("bfloat16", "float32"), ("float32", "float32")])
def test_few_rows_match_float64(hip, act, out, M, N, K):
    """With bias and, for fp32 results, the C term.  The K products are summed in fp32: at most K 2^-24
    sum |a w|; 2^-22 of the epilogue's terms; a bf16 result is rounded by at most 2^-8 of itself."""
    x = syn.normal(1, (M, K))
    if act == "bfloat16":
        bits, x = syn.bf16(x)
        xt = Tensor(bits, dtype=act)
    else:
        xt = Tensor(x, dtype=act)
    wbits, w = syn.bf16(syn.normal(2, (N, K), 0.05))
    bbits, b = syn.bf16(syn.normal(4, (N,)))
    c = syn.normal(3, (M, N))
    wt = Tensor(wbits, dtype="bfloat16")
    x64, w64 = x.astype(np.float64), w.astype(np.float64)
    ref, mag = x64 @ w64.T + b, np.abs(x64) @ np.abs(w64).T
    if out == "float32":
        y = F.dispatch_matmul(xt, wt, c=Tensor(c), beta=0.5, alpha=2.0, bias=Tensor(b.astype(np.float32)),
                              transpose_b=True, out_dtype=out).numpy()
        ref, mag = 2.0 * (ref - b) + 0.5 * c + b, 2.0 * mag
    else:
        y = F.dispatch_matmul(xt, wt, bias=Tensor(bbits, dtype=out), transpose_b=True, out_dtype=out).numpy()
    y = y.astype(np.float64)
    bar = K * 2.0 ** -24 * mag + 2.0 ** -22 * (np.abs(ref) + np.abs(c) + np.abs(b) + 1.0)
    if out == "bfloat16":
        bar = bar + 2.0 ** -8 * (np.abs(ref) + bar)
    assert np.all(np.abs(y - ref) <= bar), np.max(np.abs(y - ref) - bar)


@pytest.mark.parametrize("M,N,K", [(8, 1024, 3072), (5, 256, 4104), (2, 64, 8200), (8, 1024, 1024), (9, 1024, 3072)])
def test_split_count_of_few_rows(hip, M, N, K):
    """The count is kh_gemm's with fp32 results also where two to eight bf16 rows are too long for the skinny
    kernel's LDS (M K > 16384) and take the tiles: kh_gemm's result is its partials added in split order, bit
    for bit.  fp32 rows are not split there."""
    from kandle_amd import kernels
    bits, _ = syn.bf16(syn.normal(1, (M, K)))
    wbits, _ = syn.bf16(syn.normal(2, (N, K), 0.05))
    xt, wt = Tensor(bits, dtype="bfloat16"), Tensor(wbits, dtype="bfloat16")
    n = kernels.gemm_split_count(M, N, K, "bfloat16")
    if M <= 8:
        assert (n > 1) == (M * K > 16384)
        assert kernels.gemm_split_count(M, N, K, "float32") == 1
    if n == 1:
        return
    y = F.dispatch_matmul(xt, wt, transpose_b=True, out_dtype="float32").numpy()
    part = F.zeros((n, M, N))
    kernels._lib.call("kh_gemm_splitk_partials", xt.handle.data_ptr(), K, wt.handle.data_ptr(), K,
                      part.handle.data_ptr(), M, N, K, n, 1)
    total = np.zeros((M, N), np.float32)
    for p in part.numpy():
        total += p
    assert np.array_equal(total, y)
