"""Decode attention's two chunk sizes (kh_decode_attention): full chunks and, where those would leave
CUs idle, chunks of a quarter."""
import numpy as np
import pytest

import oracle
from kandle_amd import Tensor, synthetic as syn
from kandle_amd import functional as F

pytestmark = pytest.mark.gpu


def _case(seed, shape, dtype):
    x = syn.normal(seed, shape)
    if dtype == "float32":
        return Tensor(x, dtype=dtype), x
    bits, vals = syn.bf16(x)
    return Tensor(bits, dtype=dtype), vals


@pytest.mark.parametrize("dtype,d,hq", [("float32", 128, 4), ("bfloat16", 128, 4), ("float32", 64, 6), ("bfloat16", 64, 2)])
def test_quarter_chunks_match_full_chunks_and_oracle(hip, dtype, d, hq):
    """Lengths on and beside the edges of the small (32 to 128 keys) and full chunks.  The same rows in a
    cache long enough for two full chunks per CU take full chunks: both against the oracle, and each
    against the other (fp32: sums of a few hundred products in two groupings, 1e-5 of the largest
    value; bf16: one output rounding, 2^-8 of it)."""
    hkv, lens = 2, np.array([0, 1, 31, 32, 33, 127, 128, 129, 300], np.int32)
    B, short = len(lens), 300
    full = {("float32", 128): 128, ("bfloat16", 128): 256, ("float32", 64): 256, ("bfloat16", 64): 512}[(dtype, d)]
    q, qh = _case(1, (B, hq, d), dtype)
    k, kh = _case(2, (B, hkv, short, d), dtype)
    v, vh = _case(3, (B, hkv, short, d), dtype)
    sl = Tensor(lens, dtype="int32")
    scale = 1.0 / np.sqrt(d)
    assert (short + full - 1) // full * hkv * B < 400      # quarter chunks
    got = F.decode_attention(q, k, v, sl, scale).numpy()
    long = full * (512 // (hkv * B) + 1)                    # at least 512 full chunks, more than 17 a sequence
    assert long // full * hkv * B >= 512 and long // full > 17
    kl, vl = (F.zeros((B, hkv, long, d), dtype) for _ in range(2))
    for dst, src in ((kl, k), (vl, v)):
        F.copy_(F.narrow(dst, 2, 0, short), src)
    got_full = F.decode_attention(q, kl, vl, sl, scale).numpy()
    for b, n in enumerate(lens):
        if n == 0:
            assert not got[b].any() and not got_full[b].any()
            continue
        ref = oracle.sdpa(qh[b][None, :, None], kh[b][None, :, :n], vh[b][None, :, :n], scale=scale)[0, :, 0]
        bar = np.abs(ref).max() * (1e-4 if dtype == "float32" else 2.0 ** -7)
        assert np.abs(got[b] - ref).max() <= bar
        assert np.abs(got_full[b] - ref).max() <= bar
        assert np.abs(got[b] - got_full[b]).max() <= np.abs(ref).max() * (1e-5 if dtype == "float32" else 2.0 ** -7)


@pytest.mark.parametrize("hq,hkv,L", [(16, 8, 8000), (32, 8, 8000), (12, 2, 8000)])
def test_quarter_chunks_are_as_exact_as_full_chunks(hip, hq, hkv, L):
    """One long fp32 sequence: four times the partials, merged without longer chains of fp32 sums.  The mean
    error of four inputs against float64 (some 2e-7; the means of two such sets of outputs differ by about a
    percent) is compared with that of full chunks, which the same rows take in a cache of more keys."""
    d, scale = 128, 1.0 / np.sqrt(128)
    groups = hq // (hq // hkv)
    long = 128 * (-(-512 // groups)) + 1
    sl = Tensor(np.array([L], np.int32), dtype="int32")
    err = np.zeros(2)
    for seed in range(4):
        q, k, v = (syn.normal(10 * seed + i, s) for i, s in enumerate(((1, hq, d), (1, hkv, L, d), (1, hkv, L, d))))
        ref = np.empty((hq, d))
        for h in range(hq):
            s = k[0, h // (hq // hkv)].astype(np.float64) @ q[0, h].astype(np.float64) * scale
            p = np.exp(s - s.max())
            ref[h] = p @ v[0, h // (hq // hkv)].astype(np.float64) / p.sum()
        for i, n in enumerate((L, long)):
            kc, vc = (Tensor(np.concatenate([x, np.zeros((1, hkv, n - L, d), np.float32)], 2)) for x in (k, v))
            got = F.decode_attention(Tensor(q), kc, vc, sl, scale).numpy()[0].astype(np.float64)
            err[i] += np.linalg.norm(got - ref) / np.linalg.norm(ref)
    assert err[0] <= 1.01 * err[1], err / 4


@pytest.mark.parametrize("dtype,B,hq,hkv,L,d", [
    ("bfloat16", 16, 16, 16, 512, 128), ("bfloat16", 16, 16, 16, 440, 128), ("float32", 16, 16, 8, 256, 128),
    ("bfloat16", 8, 64, 8, 1000, 128), ("bfloat16", 1, 64, 8, 8000, 128), ("float32", 1, 64, 8, 6000, 128)])
def test_both_sides_of_whole_rounds(hip, dtype, B, hq, hkv, L, d):
    """Caches whose full chunks fill the CUs a whole number of times, which keep full chunks for more than
    eight sequences and for groups of eight heads, and those beside them: against the oracle."""
    q, qh = _case(1, (B, hq, d), dtype)
    k, kh = _case(2, (B, hkv, L, d), dtype)
    v, vh = _case(3, (B, hkv, L, d), dtype)
    lens = np.linspace(L // 4, L, B).astype(np.int32)
    scale = 1.0 / np.sqrt(d)
    got = F.decode_attention(q, k, v, Tensor(lens, dtype="int32"), scale).numpy()
    for b in {0, B // 2, B - 1}:
        n = lens[b]
        ref = oracle.sdpa(qh[b][None, :, None], kh[b][None, :, :n], vh[b][None, :, :n], scale=scale)[0, :, 0]
        assert np.abs(got[b] - ref).max() <= np.abs(ref).max() * (1e-4 if dtype == "float32" else 2.0 ** -7)
