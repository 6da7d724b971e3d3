"""The fused QKV projection (kh_gemm_qk_norm_rope) on every tile that real sizes choose, and the K-split
products of fp32 activations on theirs."""
import numpy as np
import pytest

import oracle
from kandle_amd import Tensor, kernels, synthetic as syn
from kandle_amd import functional as F
from kandle_amd.tensor import HipTensorHandle

pytestmark = pytest.mark.gpu


# 64 x 128 tiles, 128 x 128, 128 x 256 (fp32 activations) or 256 x 128 (bf16), 256 x 256: whole heads and an odd
# number of them, which leaves the 256-wide tiles' last half past the last head.
@pytest.mark.parametrize("S,Hq,Hkv", [(300, 5, 1), (1000, 16, 8), (1100, 15, 5), (1531, 15, 5), (1100, 21, 7),
                                      (1531, 32, 8), (2048, 21, 7), (1531, 16, 8), (2048, 16, 8)])
@pytest.mark.parametrize("act", ["float32", "bfloat16"])
def test_fused_projection_equals_separate_launches(hip, act, S, Hq, Hkv):
    """Bit for bit projection, then qk-norm + RoPE and the cache write; the last rows lie past the cache."""
    D, H, L, pos0 = 128, 136, S + 5, 10
    N = (Hq + 2 * Hkv) * D
    assert kernels.gemm_split_count(S, N, H, act) == 1
    x = syn.normal(1, (S, H))
    x = Tensor(syn.bf16(x)[0], dtype=act) if act == "bfloat16" else Tensor(x)
    w = Tensor(syn.bf16(syn.normal(2, (N, H), 0.05))[0], dtype="bfloat16")
    norm = []
    for seed in (3, 4):
        bits, vals = syn.bf16(syn.uniform(seed, (D,), 0.5, 1.5))
        b = Tensor(bits, dtype="bfloat16")
        norm.append((b, b if act == "bfloat16" else Tensor(vals)))
    inv = Tensor(oracle.rope_inv_freq(D, 1e6))
    pos = Tensor(np.arange(pos0, pos0 + S, dtype=np.int32), dtype="int32")
    params = {"inv_freq": inv.handle, "positions": pos.handle, "eps": 1e-6}

    def outputs():
        return [HipTensorHandle.create_new((1, Hq, S, D), act)] + [F.zeros((1, Hkv, L, D), act).handle for _ in range(2)]

    qkv = F.linear(x, w)
    assert qkv.dtype == act

    def heads(col, n):
        return HipTensorHandle.create_view(qkv.handle.storage, (1, S, n, D), act, (S * N, N, D, 1), col)

    q1, k1, v1 = outputs()
    kernels.rms_norm_rope(heads(0, Hq), heads(Hq * D, Hkv), dict(
        params, q_weight=norm[0][1].handle, k_weight=norm[1][1].handle, q_out=q1, k_out=k1, v=heads((Hq + Hkv) * D, Hkv),
        v_out=v1, cache_positions=True))
    q2, k2, v2 = outputs()
    kernels.linear_qk_norm_rope(x.handle, w.handle, dict(
        params, q_weight=norm[0][0].handle, k_weight=norm[1][0].handle, q_out=q2, k_out=k2, v_out=v2))
    for a, b in ((q1, q2), (k1, k2), (v1, v2)):
        assert np.array_equal(Tensor(handle=a).numpy(), Tensor(handle=b).numpy())
    assert not Tensor(handle=k2).numpy()[:, :, :pos0].any()


# Split on 128 x 128, 128 x 256, 256 x 256, 64 x 192 and 128 x 192 tiles, rows and columns ragged, the last part
# shorter than the others.
@pytest.mark.parametrize("M,N,K", [(700, 1000, 2056), (1001, 1028, 2056), (2040, 1028, 2056), (1300, 1000, 4104),
                                   (1001, 2564, 9736), (2040, 300, 2056), (700, 1028, 3080), (1001, 1028, 3080)])
def test_split_products_of_large_tiles(hip, M, N, K):
    """fp32 activations as a bf16 pair (2^-16 of each product off at most) and K sums in fp32, with the C term."""
    assert kernels.gemm_split_count(M, N, K, "float32") > 1
    x, c = syn.normal(1, (M, K)), syn.normal(3, (M, N))
    wbits, w = syn.bf16(syn.normal(2, (N, K), 0.05))
    y = F.dispatch_matmul(Tensor(x), Tensor(wbits, dtype="bfloat16"), c=Tensor(c), beta=1.0, transpose_b=True).numpy()
    x64, w64 = x.astype(np.float64), w.astype(np.float64)
    ref = x64 @ w64.T + c
    bar = (2.0 ** -16 + K * 2.0 ** -24) * (np.abs(x64) @ np.abs(w64).T) + 2.0 ** -22 * (np.abs(ref) + np.abs(c))
    assert np.all(np.abs(y - ref) <= bar), np.max(np.abs(y - ref) - bar)
