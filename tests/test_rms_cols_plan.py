"""RMSNorm of ragged column tiles: where the squares are added in a launch of their own."""

from __future__ import annotations

import pytest
import torch

from deepfold_amd import nf4

LINES = [(17, 4096), (24, 4096), (31, 4096), (33, 2048), (48, 2048), (63, 2048)]


# one call after the other without a graph, 24 columns of 1024 to 3072 rows took 11.9 us in two launches, 7.4 to 9.2 in one
@pytest.mark.parametrize("n,rows", LINES)
def test_short_tiles_take_one_launch_and_no_workspace(n, rows):
    lib = nf4._load_ext()
    assert lib.chr_dv2_rms_cols_ws_for(rows - 1, n) == 0
    assert lib.chr_dv2_rms_cols_ws_for(rows, n) == lib.chr_dv2_rms_cols_ws_floats() > 0


def test_other_tiles_ask_for_none():
    lib = nf4._load_ext()
    assert [n for n in range(-1, 70) if lib.chr_dv2_rms_cols_ws_for(1 << 20, n) != 0] == [
        n for n in range(17, 64) if n != 32]


@pytest.mark.gpu
@pytest.mark.parametrize("n,rows", LINES)
@pytest.mark.parametrize("over", [-1, 0, 7])
def test_both_ways_give_the_same_bits(n, rows, over, monkeypatch):
    rows += over
    gen = torch.Generator(device="cuda").manual_seed(rows + n)
    x = torch.randn(rows, n, generator=gen, device="cuda").to(torch.bfloat16)
    w = torch.randn(rows, generator=gen, device="cuda").to(torch.bfloat16)
    allocated = []
    empty = torch.empty
    monkeypatch.setattr(torch, "empty", lambda *a, **k: allocated.append(a) or empty(*a, **k))
    out = nf4.dv2_rms_cols(x, w, 1e-6)
    assert len(allocated) == (over >= 0)
    one = torch.empty_like(x)
    assert nf4._load_ext().chr_dv2_rms_cols(x.data_ptr(), w.data_ptr(), one.data_ptr(), rows, n, 1e-6, nf4._stream()) == 0
    assert torch.equal(out, one)
