"""Column counts that are no whole vectors: activations fetched as one flat span, at tile remainders
and at the end of x (what lies behind it is NaN and must not be multiplied)."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from deepfold_amd import nf4
from oracle import nf4_oracle as oc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2, 3, 7, 9, 15, 17, 31, 33, 47, 63])
@pytest.mark.parametrize("m,k", [(40, 1), (130, 65), (64, 256), (200, 1111), (256, 2049), (4096, 5120)])
def test_odd_columns(n, m, k):
    w = (np.random.default_rng(m + k).standard_normal((m, k)) * 0.05).astype(np.float32)
    p, s = oc.c_encode(w)
    dense = torch.from_numpy(oc.c_decode(p, s, m, k).copy()).cuda().to(torch.bfloat16).double()
    g = torch.Generator(device="cuda").manual_seed(n)
    room = torch.full((k * n + 64,), float("nan"), dtype=torch.bfloat16, device="cuda")
    x = room[:k * n].view(k, n)
    x.copy_(torch.randn(k, n, generator=g, device="cuda"))
    y = nf4.nf4_gemm(torch.from_numpy(p).cuda(), torch.from_numpy(np.ascontiguousarray(s).view(np.float16)).cuda(), x, m, k,
                     oc.k_pad(k), 64).double()
    want = dense @ x.double()
    assert bool(torch.isfinite(y).all())
    # one bf16 rounding of each result (2^-9) over fp32 sums of the bf16 weights these tiles multiply
    assert float((y - want).abs().max()) <= 2.0 ** -8 * float(want.abs().max())
    assert float((y - want).norm()) <= 2.5e-3 * float(want.norm())


# 33..63 columns are staged in an order of their own (512 pieces a wavefront): spans that end in each of its
# wavefronts, within a pair and within a piece
@pytest.mark.parametrize("n", [34, 39, 40, 48, 56, 61, 62])
@pytest.mark.parametrize("m,k", [(33, 63), (130, 150), (64, 256), (33, 257), (64, 2047)])
def test_columns_dealt_in_pairs(n, m, k):
    test_odd_columns(n, m, k)
