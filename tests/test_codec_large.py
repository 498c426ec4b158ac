"""More weights than one grid of the codec kernels has threads for, both ways, bit for bit against the CPU
codec at the rows where the launches meet and at the ends."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from deepfold_amd import nf4
from oracle import nf4_oracle as oc

pytestmark = pytest.mark.gpu


# 2^22 rows and a few: 2^24 workgroups of the quantiser, 2^23 (2^24 at the ragged width) of the decoder
@pytest.mark.parametrize("k", [8192, 8191])
def test_more_than_one_launch(k):
    m = (1 << 22) + 2053
    if torch.cuda.mem_get_info()[0] < 200 << 30:
        pytest.skip("needs 200 GiB of free device memory")
    rows = [0, 1, (1 << 20) - 1, 1 << 20, (1 << 21) - 1, 1 << 21, (1 << 21) + 1, (1 << 22) - 1, 1 << 22, m - 2, m - 1]
    some = (np.random.default_rng(k).standard_normal((len(rows), k)) * 0.03).astype(np.float32)
    try:
        w = torch.zeros((m, k), device="cuda")
        w[rows] = torch.from_numpy(some).cuda()
        packed, scale = nf4.nf4_quantize(w)
        del w
        torch.cuda.empty_cache()
        p, s = oc.c_encode(some)
        assert np.array_equal(packed[rows].cpu().numpy(), np.asarray(p).reshape(len(rows), -1))
        assert np.array_equal(scale[rows].cpu().numpy().view(np.uint16), np.asarray(s).view(np.uint16).reshape(len(rows), -1))
        others = torch.ones(m, dtype=torch.bool, device="cuda")
        others[rows] = False
        assert int((scale[:, 0] == 1).sum()) >= int(others.sum())        # a row of zeros: scale one, code seven
        assert bool((packed[others.nonzero()[::4096, 0]] == 0x77).all())
        out = nf4.nf4_dequant(packed, scale, m, k, oc.k_pad(k))
        assert np.array_equal(out[rows].cpu().numpy().view(np.uint32), oc.c_decode(p, s, len(rows), k).view(np.uint32))
        assert bool((out[others.nonzero()[::4096, 0]] == 0).all())
        del out
    finally:
        torch.cuda.empty_cache()
