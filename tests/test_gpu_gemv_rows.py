"""One-row projections over the row lengths at which the prologue changes how it reads its input."""
import numpy as np
import pytest

import oracle
from kandle_amd import Tensor, synthetic as syn
from kandle_amd import functional as F

pytestmark = pytest.mark.gpu


# One load and less, a 512-wide chunk's edges, the longest normalised row in registers (2048) and the next,
# the longest plain one (fp32 4096, bf16 8192) and the next.
@pytest.mark.parametrize("K", [8, 504, 512, 520, 2048, 2056, 4096, 4104, 8192, 8200])
@pytest.mark.parametrize("act", ["float32", "bfloat16"])
@pytest.mark.parametrize("prologue,skip", [("none", 0), ("none", 1), ("rms_norm", 0), ("rms_norm", 1)])
def test_row_lengths_match_oracle(hip, prologue, skip, act, K):
    """fp32 outputs; skip: the row starts one element past an aligned one.  The K products are summed in
    fp32: at most K 2^-24 sum |x' w|.  The RMSNorm's own sum and five roundings add at most (K / 2 + 5) 2^-24
    of each x'; where x' is then rounded to bf16, a value at a boundary may fall to the other side: 2^-8."""
    norm = prologue == "rms_norm"
    row = syn.normal(1, (1, K + skip), 2.0)
    if act == "bfloat16" and not norm:
        bits, row = syn.bf16(row)
        whole = Tensor(bits, dtype=act)
    else:
        whole = Tensor(row)
    x, row = F.narrow(whole, 1, skip, K), row[:, skip:].astype(np.float64)
    nbits, nw = syn.bf16(syn.uniform(2, (K,), 0.5, 1.5))
    wbits, w = syn.bf16(syn.normal(3, (37, K), 0.05))
    each = K * 2.0 ** -24
    if norm:
        row = row / np.sqrt(np.mean(row * row) + 1e-6) * nw
        each += (K / 2 + 5) * 2.0 ** -24
        if act == "bfloat16":
            row = oracle.bf16_round(row.astype(np.float32)).astype(np.float64)
            each += 2.0 ** -8
    y = F.linear_fused(prologue, x, Tensor(wbits, dtype="bfloat16"),
                       Tensor(nbits, dtype="bfloat16") if norm else None, 1e-6, out_dtype="float32",
                       act_dtype=act).numpy()
    w64 = w.astype(np.float64)
    bar = each * (np.abs(row) @ np.abs(w64).T)
    assert np.all(np.abs(y - row @ w64.T) <= bar + 1e-30), np.max(np.abs(y - row @ w64.T) / bar)
