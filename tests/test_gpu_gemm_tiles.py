"""The MFMA tile kernel over its tiles and K splits (kh_gemm_ex): edges of rows, columns and k ranges."""
import numpy as np
import pytest

import oracle
from kandle_amd import Tensor, kernels, synthetic as syn
from kandle_amd import functional as F

pytestmark = pytest.mark.gpu


# Rows and columns one short of, on and past tiles of 64 to 256; k of one 16-wide step and less, not a
# multiple of the 32- and 64-wide stages, and long enough to split; the large ones reach the 128- and
# 256-wide tiles of each activation type.
@pytest.mark.parametrize("M,N,K", [
    (9, 64, 8), (17, 130, 40), (63, 65, 72), (65, 100, 136), (129, 257, 104), (200, 1000, 1016), (257, 300, 2056),
    (513, 1027, 264), (300, 6144, 520), (700, 6150, 328), (1000, 4100, 200), (2040, 5000, 96)])
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_tiles_match_oracle(hip, dtype, M, N, K):
    """fp32 outputs with the C and bias terms.  fp32 activations are multiplied as a bf16 pair, 2^-16 of
    each product off at most; the K products are summed in fp32: at most (2^-16 + K 2^-24) sum |a w|
    (bf16 activations: only the sums), plus 2^-22 of the epilogue's terms."""
    x = syn.normal(1, (M, K))
    if dtype == "bfloat16":
        bits, x = syn.bf16(x)
        xt = Tensor(bits, dtype=dtype)
    else:
        xt = Tensor(x, dtype=dtype)
    wbits, w = syn.bf16(syn.normal(2, (N, K), 0.05))
    c, b = syn.normal(3, (M, N)), syn.normal(4, (N,))
    y = F.dispatch_matmul(xt, Tensor(wbits, dtype="bfloat16"), c=Tensor(c), beta=0.5, alpha=2.0, bias=Tensor(b),
                          transpose_b=True, out_dtype="float32").numpy()
    x64, w64 = x.astype(np.float64), w.astype(np.float64)
    ref = 2.0 * (x64 @ w64.T) + 0.5 * c + b
    each = (2.0 ** -16 if dtype == "float32" else 0.0) + K * 2.0 ** -24
    bar = 2.0 * each * (np.abs(x64) @ np.abs(w64).T) + 2.0 ** -22 * (np.abs(ref) + np.abs(c) + np.abs(b) + 1.0)
    assert np.all(np.abs(y - ref) <= bar), np.max(np.abs(y - ref) - bar)


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("M,I,K", [(70, 40, 72), (300, 1504, 136), (512, 3072, 64), (1000, 3080, 40)])
def test_swiglu_tiles_match_plain_tiles(hip, dtype, M, I, K):
    """The SwiGLU epilogue, whatever tile runs it, equals silu * mul of the same projection's columns from
    the plain product, whose sums have the same bits."""
    def act(seed, shape, std):
        v = syn.normal(seed, shape, std)
        return Tensor(syn.bf16(v)[0], dtype=dtype) if dtype == "bfloat16" else Tensor(v, dtype=dtype)
    x = act(1, (M, K), 1.0)
    g, u = (syn.bf16(syn.normal(s, (I, K), 0.2))[0] for s in (2, 3))
    gu = kernels.interleave_gate_up(g, u)
    got = F.linear_swiglu(x, Tensor(gu, dtype="bfloat16")).numpy()
    gate, up = (F.linear(x, Tensor(w, dtype="bfloat16")) for w in (g, u))
    assert kernels.gemm_split_count(M, I, K, dtype) == 1
    assert np.array_equal(got, F.silu_mul(gate, up).numpy())


def test_split_counts_follow_the_activation_type(hip):
    """kh_gemm_split_count (bf16) and the typed count; partials accept the other type's count."""
    assert kernels.gemm_split_count(1000, 1024, 3072) == 1
    n = kernels.gemm_split_count(1000, 1024, 3072, "float32")
    assert n > 1
    M, N, K = 1000, 1024, 3072
    bits, x = syn.bf16(syn.normal(1, (M, K)))
    wbits, w = syn.bf16(syn.normal(2, (N, K), 0.05))
    xt, wt = Tensor(bits, dtype="bfloat16"), Tensor(wbits, dtype="bfloat16")
    part = F.zeros((n, M, N))
    kernels._lib.call("kh_gemm_splitk_partials", xt.handle.data_ptr(), K, wt.handle.data_ptr(), K, part.handle.data_ptr(),
                      M, N, K, n, 1)
    x64, w64 = x.astype(np.float64), w.astype(np.float64)
    bar = K * 2.0 ** -24 * (np.abs(x64) @ np.abs(w64).T)
    assert np.all(np.abs(part.numpy().astype(np.float64).sum(0) - x64 @ w64.T) <= bar)


@pytest.mark.parametrize("M,N,K", [(640, 1024, 2048), (128, 4096, 1024), (960, 1024, 3072), (200, 2560, 4096),
                                   (100, 6144, 2560), (9, 2560, 4096), (256, 2560, 9728), (900, 1004, 1024)])
def test_bf16_products_sum_fp32_results_in_short_chains(hip, M, N, K):
    """fp32 results of bf16 products of few tiles.  A chain of n 16-wide steps of like products has a
    rounding error of about 2^-24 sqrt(n / 6) of the result (step i adds half a unit, uniformly, of a sum of
    i of the n steps); n = K / 16 split over the workgroups that put two 64 x 64 tiles on a CU, at most
    eight, is the longest chain.  One chain of twice that is sqrt(2) off the bar, and the whole K more."""
    parts = min(8, 512 // (-(-M // 64) * -(-N // 64)))
    bits, x = syn.bf16(syn.normal(1, (M, K)))
    wbits, w = syn.bf16(syn.normal(2, (N, K), 0.02))
    y = F.dispatch_matmul(Tensor(bits, dtype="bfloat16"), Tensor(wbits, dtype="bfloat16"), transpose_b=True,
                          out_dtype="float32").numpy().astype(np.float64)
    ref = x.astype(np.float64) @ w.astype(np.float64).T
    err = np.linalg.norm(y - ref) / np.linalg.norm(ref)
    assert err <= 1.1 * 2.0 ** -24 * np.sqrt(K / (16.0 * max(2, parts) * 6.0)), err


@pytest.mark.parametrize("act", ["bfloat16", "float32"])
@pytest.mark.parametrize("M,N,K", [(512, 1024, 640), (256, 1024, 640), (640, 512, 512), (200, 2048, 1016)])
def test_short_sums_are_not_split(hip, act, M, N, K):
    """Sums shorter than 1024 of more than a few tiles: one launch, and fp32 results of bf16 products still in short chains (a chain of
    n steps is about 2^-24 sqrt(n / 6) of the result off; four of them, added at the end, half of one)."""
    assert kernels.gemm_split_count(M, N, K, act) == 1
    if act == "float32":
        return
    bits, x = syn.bf16(syn.normal(1, (M, K)))
    wbits, w = syn.bf16(syn.normal(2, (N, K), 0.02))
    y = F.dispatch_matmul(Tensor(bits, dtype="bfloat16"), Tensor(wbits, dtype="bfloat16"), transpose_b=True,
                          out_dtype="float32").numpy().astype(np.float64)
    ref = x.astype(np.float64) @ w.astype(np.float64).T
    err = np.linalg.norm(y - ref) / np.linalg.norm(ref)
    assert err <= 0.7 * 2.0 ** -24 * np.sqrt(K / (16.0 * 6.0)), err


@pytest.mark.parametrize("M,N,K,n", [(256, 2560, 9728, 3), (150, 5120, 6152, 2), (250, 2500, 6144, 3), (256, 2560, 4096, 1)])
def test_long_bf16_sums_are_split(hip, M, N, K, n):
    """bf16 products of five eighths to all of the CUs' 64 x 64 tiles: split from 6144 columns on.  The K
    products are summed in fp32 (K 2^-24 sum |a w| at most), the bf16 result rounded (2^-8 of itself)."""
    assert kernels.gemm_split_count(M, N, K) == n
    assert kernels.gemm_split_count(M, 0, K) == 1
    bits, x = syn.bf16(syn.normal(1, (M, K)))
    wbits, w = syn.bf16(syn.normal(2, (N, K), 0.02))
    x64, w64 = x.astype(np.float64), w.astype(np.float64)
    ref, bar = x64 @ w64.T, K * 2.0 ** -24 * (np.abs(x64) @ np.abs(w64).T)
    for out in ("float32", "bfloat16"):
        y = F.dispatch_matmul(Tensor(bits, dtype="bfloat16"), Tensor(wbits, dtype="bfloat16"), transpose_b=True,
                              out_dtype=out).numpy().astype(np.float64)
        most = bar if out == "float32" else bar + 2.0 ** -8 * (np.abs(ref) + bar)
        assert np.all(np.abs(y - ref) <= most)


@pytest.mark.parametrize("M,N,K,n", [(9, 2560, 4096, 8), (32, 2560, 9728, 8), (9, 6144, 2568, 5), (9, 5120, 2048, 6),
                                     (17, 100, 2056, 6)])
def test_few_fp32_rows_are_split_widely(hip, M, N, K, n):
    """Up to 32 fp32 rows, which stream weights: 512 / tiles parts of K, at most eight and of whole 128 columns.
    Each product is 2^-16 off at most (the bf16 pair), the K of them are summed in fp32."""
    assert kernels.gemm_split_count(M, N, K, "float32") == n
    x = syn.normal(1, (M, K))
    wbits, w = syn.bf16(syn.normal(2, (N, K), 0.02))
    y = F.dispatch_matmul(Tensor(x), Tensor(wbits, dtype="bfloat16"), transpose_b=True).numpy().astype(np.float64)
    x64, w64 = x.astype(np.float64), w.astype(np.float64)
    bar = (2.0 ** -16 + K * 2.0 ** -24) * (np.abs(x64) @ np.abs(w64).T)
    assert np.all(np.abs(y - x64 @ w64.T) <= bar)


@pytest.mark.parametrize("M", [9, 4194305])
def test_no_columns(hip, M):
    """K = 0: the C and bias terms alone, also for more rows than the generic kernel's grid holds."""
    n = 8
    c, b = Tensor(np.full((M, n), 3.0, np.float32)), Tensor(np.arange(n, dtype=np.float32))
    a = Tensor(np.zeros((1, 8), np.uint16), dtype="bfloat16")
    out = F.zeros((M, n))
    kernels._lib.call("kh_gemm_ex", a.handle.data_ptr(), 0, 1, a.handle.data_ptr(), 0, 1, out.handle.data_ptr(), n,
                      c.handle.data_ptr(), n, b.handle.data_ptr(), M, n, 0, 1.0, 0.5, 1, 0)
    assert np.array_equal(out.numpy(), np.broadcast_to(1.5 + np.arange(n, dtype=np.float32), (M, n)))
