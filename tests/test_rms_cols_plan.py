"""RMSNorm of ragged column tiles: where the squares are added in a launch of their own."""

from __future__ import annotations

import pytest
import torch

from deepfold_amd import nf4

# columns, rows from which two launches are taken one by one, rows from which they are recorded into a graph
LINES = [(17, 4096, 1536), (24, 4096, 1536), (31, 4096, 1536), (33, 2048, 1024), (48, 2048, 1024), (63, 2048, 1024)]


# one call after the other without a graph, 24 columns of 1024 to 3072 rows took 11.9 us in two launches, 7.4 to 9.2 in one
@pytest.mark.parametrize("n,launched,recorded", LINES)
def test_short_tiles_take_one_launch_and_no_workspace(n, launched, recorded):
    lib = nf4._load_ext()
    for line, mode in ((launched, 0), (recorded, 1)):
        assert lib.chr_dv2_rms_cols_ws_for(line - 1, n, mode) == 0
        assert lib.chr_dv2_rms_cols_ws_for(line, n, mode) == lib.chr_dv2_rms_cols_ws_floats() > 0


def test_other_tiles_ask_for_none():
    lib = nf4._load_ext()
    for mode in (0, 1):
        assert [n for n in range(-1, 70) if lib.chr_dv2_rms_cols_ws_for(1 << 20, n, mode) != 0] == [
            n for n in range(17, 64) if n != 32]


@pytest.mark.gpu
@pytest.mark.parametrize("n,launched,recorded", LINES)
@pytest.mark.parametrize("over", [-1, 0, 7])
def test_both_ways_give_the_same_bits(n, launched, recorded, over, monkeypatch):
    allocated = []
    empty = torch.empty
    monkeypatch.setattr(torch, "empty", lambda *a, **k: allocated.append(a) or empty(*a, **k))
    for line, in_graph in ((launched, False), (recorded, True)):
        rows = line + over
        gen = torch.Generator(device="cuda").manual_seed(rows + n)
        x = torch.randn(rows, n, generator=gen, device="cuda").to(torch.bfloat16)
        w = torch.randn(rows, generator=gen, device="cuda").to(torch.bfloat16)
        one = torch.empty_like(x)

        def one_launch():
            rc = nf4._load_ext().chr_dv2_rms_cols(x.data_ptr(), w.data_ptr(), one.data_ptr(), rows, n, 1e-6, nf4._stream())
            assert rc == 0

        one_launch()
        allocated.clear()
        if not in_graph:
            out = nf4.dv2_rms_cols(x, w, 1e-6)
            assert len(allocated) == (over >= 0)
            assert torch.equal(out, one)
            continue
        graph = torch.cuda.CUDAGraph()
        torch.cuda.synchronize()
        with torch.cuda.graph(graph):
            out = nf4.dv2_rms_cols(x, w, 1e-6)
        assert len(allocated) == (over >= 0)
        for _ in range(3):
            x.copy_(torch.randn(rows, n, generator=gen, device="cuda"))
            one_launch()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, one)
