"""bf16 prefill attention of short calls: the kernel without shared tiles (flash_direct_kernel) and the
forms of the persistent kernel split over keys in four and, without the causal mask, in two."""
import numpy as np
import pytest

import oracle
from kandle_amd import Tensor, synthetic as syn
from kandle_amd import functional as F

pytestmark = pytest.mark.gpu


def _bf(seed, shape, std=1.0):
    bits, vals = syn.bf16(syn.normal(seed, shape, std))
    return Tensor(bits, dtype="bfloat16"), vals


def _check(B, hq, hkv, lq, lk, d, causal, std=1.0, rows=None):
    """Against the float oracle.  The weights P and the outputs are rounded to bf16 (2^-9 each) and l sums
    the rounded P, so an output is off by at most 2 * 2^-9 max|v| from the weights and 2^-9 max|v| from
    its own rounding; 1e-3 covers the fp32 scores and exponentials."""
    q, qh = _bf(1, (B, hq, lq, d), std)
    k, kh = _bf(2, (B, hkv, lk, d), std)
    v, vh = _bf(3, (B, hkv, lk, d))
    got = F.scaled_dot_product_attention(q, k, v, is_causal=causal).numpy()
    bar = 3 * 2.0 ** -9 * np.abs(vh).max() + 1e-3
    if rows is None:
        ref = oracle.sdpa(qh, kh, vh, causal=causal)
        assert np.abs(got - ref).max() <= bar
    else:   # chosen query rows of every head, each against the keys it sees
        for i in rows:
            end = min(i + 1, lk) if causal else lk
            ref = oracle.sdpa(qh[:, :, i:i + 1], kh[:, :, :end], vh[:, :, :end])
            assert np.abs(got[:, :, i:i + 1] - ref).max() <= bar, i


@pytest.mark.parametrize("B,hq,hkv,lq,lk,d,causal", [
    (1, 2, 1, 2, 2, 128, True), (1, 4, 2, 31, 31, 128, True), (2, 4, 1, 32, 32, 64, True), (1, 3, 3, 33, 33, 128, True),
    (1, 10, 2, 129, 129, 128, True), (1, 6, 2, 200, 200, 64, True), (1, 2, 2, 40, 150, 128, True),
    (1, 2, 2, 150, 40, 128, True), (2, 4, 2, 65, 97, 64, False), (1, 8, 8, 100, 33, 128, False),
    (1, 2, 1, 5, 300, 128, False)])
def test_direct_kernel_edges(hip, B, hq, hkv, lq, lk, d, causal):
    _check(B, hq, hkv, lq, lk, d, causal)


def test_direct_kernel_spread_scores(hip):
    """Scores spread over +-40 nats: the reference maximum is raised in the middle of the key loop."""
    _check(1, 4, 2, 190, 190, 128, True, std=2.0)


def test_direct_kernel_strided_views(hip):
    """q, k, v as heads-first views of [B, S, H, D] storage and an output view of [S, H D]."""
    B, S, hq, hkv, d = 1, 77, 4, 2, 128
    t, vals = [], []
    for seed, h in ((1, hq), (2, hkv), (3, hkv)):
        x, xv = _bf(seed, (B, S, h, d))
        t.append(F.permute(x, (0, 2, 1, 3)))
        vals.append(xv.transpose(0, 2, 1, 3))
    out = F.permute(F.zeros((B, S, hq, d), "bfloat16"), (0, 2, 1, 3))
    F.scaled_dot_product_attention(*t, is_causal=True, out=out)
    ref = oracle.sdpa(*vals, causal=True)
    assert np.abs(out.numpy() - ref).max() <= 3 * 2.0 ** -9 * np.abs(vals[2]).max() + 1e-3


# 32-row items on half to one and a half of the CUs: 16 / 8 heads from 32 x 33 rows; one head per kv head
# takes 64-row items; without the mask also the form split in two (four query heads per kv head).
@pytest.mark.parametrize("B,hq,hkv,lq,lk,d,causal", [
    (1, 16, 8, 1031, 1031, 128, True), (2, 16, 8, 740, 740, 64, True), (1, 16, 16, 1000, 1000, 128, True),
    (1, 16, 8, 1040, 900, 128, True), (1, 16, 8, 700, 700, 128, False), (1, 16, 8, 650, 1100, 64, False),
    (1, 32, 8, 700, 701, 128, False), (1, 40, 8, 500, 500, 128, False)])
def test_key_split_forms(hip, B, hq, hkv, lq, lk, d, causal):
    rows = [0, 1, 31, 32, 63, 64, 127, 128, lq // 2, lq - 33, lq - 2, lq - 1]
    _check(B, hq, hkv, lq, lk, d, causal, rows=rows)


# Both sides of the limits between the kernel without shared tiles, the forms split over keys and the small
# workgroups: 97 to 128 queries of more than one block per CU, and of exactly two; groups of eight and four heads
# of many short sequences; items split in four up to one per CU and beyond it with few and enough keys; groups
# of four without the mask.
@pytest.mark.parametrize("B,hq,hkv,S,d,causal", [
    (4, 16, 8, 128, 128, True), (5, 16, 8, 127, 128, True), (8, 16, 8, 128, 128, True), (9, 16, 8, 128, 128, True),
    (5, 16, 8, 126, 128, False), (16, 64, 8, 32, 128, True), (17, 64, 8, 31, 128, True), (64, 32, 8, 30, 128, True),
    (2, 16, 8, 512, 64, True), (4, 16, 8, 384, 128, True), (2, 16, 8, 600, 128, True), (3, 16, 8, 420, 64, True),
    (1, 40, 8, 480, 128, True), (2, 32, 8, 320, 128, False), (2, 32, 8, 321, 64, False)])
def test_forms_beside_their_limits(hip, B, hq, hkv, S, d, causal):
    _check(B, hq, hkv, S, S, d, causal, rows=sorted({0, 1, min(32, S - 1), S // 2, S - 2, S - 1}))


@pytest.mark.parametrize("B,hq,hkv,S,d,causal", [
    (1, 16, 8, 1531, 128, True), (1, 16, 8, 300, 128, True), (2, 16, 8, 600, 64, True), (1, 16, 8, 1000, 128, False),
    (1, 32, 8, 700, 128, False)])
def test_forms_repeat_themselves(hip, B, hq, hkv, S, d, causal):
    """The same call gives the same bits every time: the parts of the keys are merged in a fixed order."""
    q, k, v = (_bf(s, (B, h, S, d))[0] for s, h in ((1, hq), (2, hkv), (3, hkv)))
    first = F.scaled_dot_product_attention(q, k, v, is_causal=causal).numpy()
    for _ in range(4):
        assert np.array_equal(F.scaled_dot_product_attention(q, k, v, is_causal=causal).numpy(), first)
