"""The token-major product of any number of tokens, against the decoded matrix in 64 bits, and
through the linear seat."""

from __future__ import annotations

import ctypes

import numpy as np
import pytest
import torch

from deepfold_amd import nf4
from deepfold_amd.chr0.loader import ChrMatrix
from deepfold_amd.host import CompressedLinear, k_pad
from oracle import nf4_oracle as oc

BF16 = torch.bfloat16


def test_arguments_are_refused_before_any_launch():
    lib = nf4._load_ext()
    p = 0x4000

    def rc(m=128, k=256, kp=256, n=65, stride=256, x=p, y=p, packed=0x1000, scale=0x2000):
        w = nf4._Dev(m, k, kp, packed, scale)
        return lib.chr_nf4_wide(ctypes.byref(w), x, stride, n, y, None, 0, None, None)

    assert lib.chr_nf4_wide(None, p, 256, 4, p, None, 0, None, None) == -1
    assert rc(x=None) == -1 and rc(y=None) == -1 and rc(n=0) == -2
    assert rc(m=0) == -3 and rc(packed=None) == -3 and rc(stride=248) == -3 and rc(stride=260) == -3
    assert rc(kp=320) == -4 and rc(packed=0x1008) == -5 and rc(scale=0x2001) == -5
    assert rc(x=p + 2) == -5 and rc(y=p + 2) == -5
    w = nf4._Dev(5120, 13824, 13824, 0x1000, 0x2000)
    need = lib.chr_nf4_wide_ws(ctypes.byref(w), 128)
    assert need > 0 and need % (128 * 5120) == 0       # few tokens, long K: split
    assert lib.chr_nf4_wide(ctypes.byref(w), p, 13824, 128, p, p, need - 1, None, None) == -7
    assert lib.chr_nf4_wide(ctypes.byref(w), p, 13824, 128, p, p + 4, need, None, None) == -5
    assert lib.chr_nf4_wide_ws(ctypes.byref(w), 0) == -1
    out = [ctypes.c_int32() for _ in range(3)]
    refs = [ctypes.byref(o) for o in out]
    assert lib.chr_nf4_wide_plan(ctypes.byref(w), 128, *refs) == 0 and out[2].value == need // (128 * 5120)
    assert lib.chr_nf4_wide_plan(None, 128, *refs) == -1 and lib.chr_nf4_wide_plan(ctypes.byref(w), 128, None, *refs[1:]) == -1
    assert lib.chr_nf4_wide_plan(ctypes.byref(w), 0, *refs) == -2

    def rows_rc(k=250, kp=256, x=p, stride=250, y=p):
        w = nf4._Dev(128, k, kp, 0x1000, 0x2000)
        return lib.chr_nf4_wide_rows(ctypes.byref(w), x, stride, 65, y, None, 0, None, None)

    assert rows_rc(x=None) == -1 and rows_rc(stride=249) == -3 and rows_rc(kp=320) == -4
    assert rows_rc(x=p + 1) == -5 and rows_rc(y=p + 2) == -5


# (tile, splits or not) -> shapes just past its edges: rows and tokens that end inside it, rows that are no whole
# vectors and some that are, odd group counts (a last half stage), a ragged K
TILES = [((512, 128), True, (513, 7169, 2050)), ((512, 128), False, (257, 22017, 200)), ((256, 128), True, (513, 257, 1990)),
         ((256, 128), True, (513, 260, 2112)), ((256, 128), False, (385, 5121, 320)), ((256, 128), False, (385, 5124, 300)),
         ((256, 64), True, (33, 11009, 2050)), ((256, 64), True, (33, 11012, 2112)), ((256, 64), False, (385, 5121, 576)),
         ((256, 64), False, (385, 5124, 570)), ((256, 32), True, (300, 257, 832)), ((256, 32), True, (385, 260, 1990)),
         ((256, 32), False, (513, 2049, 320)), ((256, 32), False, (513, 2052, 300)), ((256, 16), True, (2, 255, 2050)),
         ((256, 16), True, (16, 256, 2048)), ((256, 16), False, (2, 255, 320)), ((256, 16), False, (385, 1537, 1111))]


@pytest.mark.gpu
@pytest.mark.parametrize("tile,split,shape", TILES, ids=[f"{t[0]}x{t[1]}-{'split' if p else 'whole'}-{s}" for t, p, s in TILES])
@pytest.mark.parametrize("bias", [False, True])
def test_every_tile(tile, split, shape, bias):
    n, m, k = shape
    kp = k_pad(k)
    g = torch.Generator(device="cuda").manual_seed(m + k)
    packed, scale = nf4.nf4_quantize(torch.randn(m, k, generator=g, device="cuda") * 0.05)
    plan = [ctypes.c_int32() for _ in range(3)]
    w = nf4._Dev(m, k, kp, packed.data_ptr(), scale.data_ptr())
    assert nf4._load_ext().chr_nf4_wide_plan(ctypes.byref(w), n, *map(ctypes.byref, plan)) == 0
    rows, tokens, splits = (p.value for p in plan)
    assert ((rows, tokens), splits > 1) == (tile, split)      # a refit that moves a shape needs another one here
    x = rand(n, k, seed=n)
    b = rand(m, seed=5) if bias else None
    want = x.double() @ nf4.nf4_dequant(packed, scale, m, k, kp).double().t()
    want = want + b.double() if bias else want
    got = nf4.nf4_wide(packed, scale, x, m, k, kp, bias=b)
    close(got, want)
    # a row or a token left out or taken twice hides in the norm of a large result: no element is far off.  Its
    # error is the rounding of the result and a sum of k independent roundings of the levels, 1.15e-3 of the
    # norm: six of their deviations
    far = (got.double() - want).abs() - 2.0 ** -7 * want.abs()
    assert float(far.max()) <= 6 * 1.15e-3 * float(want.pow(2).mean().sqrt()) + (2.0 ** -7 * float(b.abs().max()) if bias else 0)
    # whole pieces and rows as they are: the same bits
    padded = nf4.nf4_wide(packed, scale, torch.nn.functional.pad(x, (0, kp - k)), m, kp, kp, bias=b)
    room = torch.full((n, k + 3), float("nan"), dtype=BF16, device="cuda")
    room[:, 1:1 + k] = x
    assert torch.equal(padded, got) and torch.equal(nf4.nf4_wide(packed, scale, room[:, 1:1 + k], m, k, kp, bias=b), got)


# the padded copy of a ragged K and the rows as they are: one result, and what lies behind a row is not multiplied
@pytest.mark.gpu
@pytest.mark.parametrize("n,m,k", [(2, 300, 1), (5, 64, 63), (33, 256, 65), (70, 1030, 200), (130, 512, 1111), (520, 5000, 1090)])
def test_rows_of_a_ragged_k(n, m, k):
    mat, w = matrix(m, k, seed=k)
    kp = k_pad(k)
    clean = rand(n, k, seed=n)
    want = nf4.nf4_wide(*mat[:2], torch.nn.functional.pad(clean, (0, kp - k)), m, kp, kp)
    close(want, clean.double() @ w.t())
    for before, behind in ((0, 1), (3, 6), (8, 8)):
        room = torch.full((n, before + k + behind), float("nan"), dtype=BF16, device="cuda")
        x = room[:, before:before + k]
        x.copy_(clean)
        assert torch.equal(nf4.nf4_wide(*mat[:2], x, m, k, kp), want)


def matrix(m, k, seed, sigma=0.05):
    w = np.random.default_rng(seed).standard_normal((m, k)).astype(np.float32) * sigma
    p, s = oc.c_encode(w)
    dense = torch.from_numpy(oc.c_decode(p, s, m, k).copy()).cuda().double()
    return (torch.from_numpy(p).cuda(), torch.from_numpy(np.ascontiguousarray(s).view(np.float16)).cuda(), m), dense


def rand(*shape, seed=0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randn(*shape, generator=g, device="cuda").to(BF16)


def close(got, want):
    # one bf16 rounding of the result (2^-9 of it at most, 1.7e-3 of its norm) and one of every level
    # (1.4e-3): 2.2e-3 of the norm; a bias rounds again
    got, want = got.double(), want.double()
    assert bool(torch.isfinite(got).all())
    assert float((got - want).norm()) <= 5e-3 * float(want.norm())
    assert float((got - want).abs().max()) <= 2e-2 * max(float(want.abs().max()), 1e-3)


# few tokens and many, odd group counts (a last half stage), ragged K, rows that are no whole vectors, few tokens
# over a long K (splits); all but one take the 256 x 16 tile: test_every_tile has the others
SHAPES = [(1, 64, 64), (2, 300, 128), (17, 5120, 1088), (33, 256, 576), (65, 256, 64), (63, 255, 192), (129, 513, 320), (70, 1030, 200), (128, 130, 2048),
          (257, 77, 1111), (66, 5120, 4160), (520, 512, 640)]


@pytest.mark.gpu
@pytest.mark.parametrize("n,m,k", SHAPES)
@pytest.mark.parametrize("bias", [False, True])
def test_product(n, m, k, bias):
    mat, w = matrix(m, k, seed=m + k)
    x = rand(n, k, seed=n)
    b = rand(m, seed=5) if bias else None
    want = x.double() @ w.t()
    got = nf4.nf4_wide(*mat[:2], x, m, k, k_pad(k), bias=b)
    close(got, want + b.double() if bias else want)
    # rows of a wider buffer, aligned or not, give the same bits
    for off in (8, 3):
        wide = torch.zeros((n, k + 16), dtype=BF16, device="cuda")
        wide[:, off:off + k] = x
        assert torch.equal(nf4.nf4_wide(*mat[:2], wide[:, off:off + k], m, k, k_pad(k), bias=b), got)


# activations whose sum does not vanish meet the average of the levels' roundings: it must not grow with K.
# Bound: the rounding of the result (2^-9 of it at most: 1.7e-3 of the norm) and of the levels (1.15e-3) make 2.1e-3
@pytest.mark.gpu
@pytest.mark.parametrize("m,k", [(512, 5120), (256, 27648)])
@pytest.mark.parametrize("weights", ["normal", "uniform"])
@pytest.mark.parametrize("acts", ["mean one", "relu", "zero mean"])
def test_roundings_of_the_levels_cancel(m, k, weights, acts):
    g = torch.Generator(device="cuda").manual_seed(m + len(weights))
    w = torch.randn(m, k, generator=g, device="cuda") if weights == "normal" else torch.rand(m, k, generator=g, device="cuda") * 2 - 1
    packed, scale = nf4.nf4_quantize(w * 0.02)
    x = torch.randn(40, k, generator=g, device="cuda")
    x = {"mean one": 1 + 0.3 * x, "relu": x.relu(), "zero mean": x}[acts].to(BF16)
    want = x.double() @ nf4.nf4_dequant(packed, scale, m, k, k).double().t()
    got = nf4.nf4_wide(packed, scale, x, m, k, k).double()
    assert float((got - want).norm()) <= 2.4e-3 * float(want.norm())


@pytest.mark.gpu
@pytest.mark.parametrize("n", [2, 16, 17, 32, 33, 64, 65, 257])
@pytest.mark.parametrize("dtype", [BF16, torch.float32])
def test_linear_seat_across_the_window(n, dtype):
    m, k = 640, 500
    (p, s, _), w = matrix(m, k, seed=9)
    lin = CompressedLinear(k, m, bias=True, device="cuda", dtype=dtype)
    lin.attach(ChrMatrix("t", m, k, k_pad(k), p, s))
    lin.set_bias(rand(m, seed=1).to(dtype))
    x = rand(n, k, seed=2)
    y = lin(x)
    assert y.dtype == dtype                        # a wider bias still widens the answer
    close(y, x.double() @ w.t() + lin.bias.double())
    assert torch.equal(lin(x.t().contiguous().t()), y)   # K not the fastest axis


@pytest.mark.gpu
@pytest.mark.parametrize("n", [128, 129, 700])
def test_many_tokens_through_a_small_seat(n):
    m, k = 96, 200
    (p, s, _), w = matrix(m, k, seed=4)
    lin = CompressedLinear(k, m, device="cuda")
    lin.attach(ChrMatrix("t", m, k, k_pad(k), p, s))
    x = rand(n, k, seed=2)
    close(lin(x), x.double() @ w.t())
    assert torch.equal(lin(x), nf4.nf4_wide(p, s, x, m, k, k_pad(k))) == (n > 128)


@pytest.mark.gpu
@pytest.mark.parametrize("n,m,k", [(17, 2048, 2048), (5, 300, 500), (129, 96, 200), (8, 40, 72)])
def test_the_seat_in_a_graph(n, m, k):
    """Split and not, whole and ragged, and a small seat's window: replays with eager calls between them."""
    (p, s, _), _ = matrix(m, k, seed=6)
    lin = CompressedLinear(k, m, bias=True, device="cuda")
    lin.attach(ChrMatrix("t", m, k, k_pad(k), p, s))
    lin.set_bias(rand(m, seed=1))
    x = rand(n, k, seed=2)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        lin(x)
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = lin(x)
    for i in range(4):
        x.copy_(rand(n, k, seed=10 + i))
        want = lin(x)
        y.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, want)
