"""Several windows of a prompt in one pass: the same bits as one 64-token window after the other,
product by product and for a whole prefill."""

from __future__ import annotations

import dataclasses

import numpy as np
import pytest
import torch

from deepfold_amd import decodev2 as dv2
from deepfold_amd import nf4

BF16 = torch.bfloat16


def test_arguments_are_refused_before_any_launch():
    lib = nf4._load_ext()
    p = 0x4000

    def mats(*ms, k=5120, kp=None, packed=0x1000, scale=0x2000):
        return (nf4._Dev * len(ms))(*[nf4._Dev(m, k, kp or k, packed, scale) for m in ms])

    def gemm(w, n_mats=1, swiglu=0, x=p, n=128, y=p, ws=None, floats=0):
        return lib.chr_dv2_prompt_gemm(w, n_mats, swiglu, x, n, y, ws, floats, None, None)

    big = mats(5120)
    assert gemm(big, x=None) == -1 and gemm(big, y=None) == -1 and gemm(None) == -1
    assert gemm(big, n=0) == -2 and gemm(big, n=100) == -2
    assert gemm(mats(5120, 1024), n_mats=2, swiglu=1) == -3 and gemm(big, n_mats=4) == -3
    assert gemm(mats(5120, k=5000, kp=5056)) == -3          # K in no whole chunks: not the 64-column tile
    assert gemm(mats(64, k=256)) == -3                      # too small for that tile
    assert gemm(mats(5120, scale=0x2004)) == -5 and gemm(big, x=p + 8) == -5
    need = lib.chr_dv2_prompt_ws(mats(5120, k=13824), 1, 0, 128)
    assert need > 0 and need % (128 * 5120) == 0
    assert gemm(mats(5120, k=13824), ws=p, floats=need - 1) == -7
    assert lib.chr_dv2_prompt_ws(big, 1, 2, 96) == -1 and lib.chr_dv2_prompt_ws(big, 1, 3, 128) == -1
    assert lib.chr_dv2_rope_kv_rows(p, p, 4, 8, 2, 128, 13, 16, p, p, p, p, None) == -3
    nf4.nf4_gemm_stream_policy(-1)                          # no launch runs that tile: nothing is served
    try:
        assert lib.chr_dv2_prompt_ws(big, 1, 0, 128) == -1
    finally:
        nf4.nf4_gemm_stream_policy(0)


def rand(*shape, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randn(*shape, generator=g, device="cuda")


def matrix(m, k, seed):
    return (*nf4.nf4_quantize(rand(m, k, seed=seed) * 0.02), m)


def windows(fn, n):
    """``fn`` on every window's slice, answers token-major."""
    return torch.cat([fn(slice(lo, lo + 64)).t() for lo in range(0, n, 64)]).contiguous()


def cols(t):
    return t.t().contiguous()


# one split and several, row counts that end inside a tile of 256 and inside a block of 32, three matrices
@pytest.mark.gpu
@pytest.mark.parametrize("n,ms,k", [(64, (4100,), 512), (128, (5120, 1024, 1024), 5120), (192, (2048, 256, 256), 2048),
                                    (128, (1200,), 13824), (64, (6000, 36, 300), 1280)])
@pytest.mark.parametrize("bias", [False, True])
def test_products_repeat_the_windows(n, ms, k, bias):
    mats = [matrix(m, k, i) for i, m in enumerate(ms)]
    x = rand(n, k, seed=5).to(BF16)
    b = rand(sum(ms), seed=6).to(BF16) if bias else None
    assert nf4.dv2_prompt_serves(mats, k, 0)

    def window(at):
        if len(mats) == 3:
            return nf4.dv2_gemm_qkv(*mats, cols(x[at]), bias=b)
        return nf4.nf4_gemm(*mats[0][:2], cols(x[at]), ms[0], k, k, 64, bias=b)

    assert torch.equal(nf4.dv2_prompt_gemm(mats, x, k, bias=b), windows(window, n))


@pytest.mark.gpu
@pytest.mark.parametrize("n,m,k", [(128, 13824, 5120), (64, 4000, 6144), (64, 1100, 1024), (64, 16384, 6144)])
def test_swiglu_repeats_the_windows(n, m, k):
    gate, up = matrix(m, k, 1), matrix(m, k, 2)
    x = rand(n, k, seed=3).to(BF16)
    assert nf4.dv2_prompt_serves([gate, up], k, 1)
    assert torch.equal(nf4.dv2_prompt_gemm([gate, up], x, k, swiglu=True),
                       windows(lambda at: nf4.dv2_gemm_swiglu(gate, up, cols(x[at])), n))


@pytest.mark.gpu
@pytest.mark.parametrize("n,m,k", [(128, 5120, 5120), (64, 2048, 2048), (128, 1040, 13824), (64, 6144, 16384)])
@pytest.mark.parametrize("bias", [False, True])
def test_residual_and_norm_repeat_the_windows(n, m, k, bias):
    packed, scale, _ = matrix(m, k, 1)
    x, res, g = rand(n, k, seed=2).to(BF16), rand(n, m, seed=3).to(BF16), rand(m, seed=4).to(BF16)
    b = rand(m, seed=5).to(BF16) if bias else None
    assert nf4.dv2_prompt_serves([(packed, scale, m)], k, 2)
    assert torch.equal(nf4.dv2_prompt_rms(res, g, 1e-6), windows(lambda at: nf4.dv2_rms_cols(cols(res[at]), g, 1e-6), n))
    sums, norms = [], []
    for lo in range(0, n, 64):
        sq = torch.zeros(nf4.dv2_sq_blocks(m, 64) * 64, device="cuda")
        y, written = nf4.nf4_gemm(packed, scale, cols(x[lo:lo + 64]), m, k, k, 64, bias=b, residual=cols(res[lo:lo + 64]),
                                  colsq=sq)
        assert written
        sums.append(y.t())
        norms.append(nf4.dv2_rms_cols(y, g, 1e-6, colsq=sq).t())
    plain = res.clone()
    assert nf4.dv2_prompt_add_rms(packed, scale, x, m, k, plain, bias=b) is None
    h = nf4.dv2_prompt_add_rms(packed, scale, x, m, k, res, bias=b, norm_w=g, eps=1e-6)
    assert torch.equal(res, torch.cat(sums)) and torch.equal(plain, res) and torch.equal(h, torch.cat(norms))


@pytest.mark.gpu
@pytest.mark.parametrize("n,n_q,n_kv,hd,start", [(1, 2, 1, 8, 0), (65, 6, 2, 128, 7), (70, 4, 4, 6, 3)])
def test_rope_rows_store_what_the_columns_store(n, n_q, n_kv, hd, start):
    room = start + n + 2
    cos, sin = rand(room, hd, seed=1).to(BF16), rand(room, hd, seed=2).to(BF16)
    qkv = rand(n, (n_q + 2 * n_kv) * hd, seed=3).to(BF16)
    q, k, v = (t.contiguous() for t in torch.split(qkv, [n_q * hd, n_kv * hd, n_kv * hd], dim=1))
    caches = [torch.zeros(room, n_kv, hd, dtype=BF16, device="cuda") for _ in range(4)]
    want = torch.empty_like(q)
    for lo in range(0, n, 64):
        q_out = torch.empty_like(q[lo:lo + 64])
        nf4.dv2_rope_kv_cols(*(cols(t[lo:lo + 64]) for t in (q, k, v)), q_out, caches[0], caches[1], cos, sin,
                             torch.tensor(start + lo, device="cuda"))
        want[lo:lo + 64] = q_out
    assert torch.equal(nf4.dv2_rope_kv_rows(qkv, n_q, caches[2], caches[3], cos, sin, start), want)
    assert torch.equal(caches[0], caches[2]) and torch.equal(caches[1], caches[3])


#: two layers of the decoders: gate and up window by window, plain, with fused wqkv and a split SwiGLU, long K
SPECS = [(dv2.QWEN25_3B, 192, 5), (dv2.QWEN25_14B, 200, 0), (dv2.INTERNLM25_20B, 130, 9), (dv2.QWEN25_32B, 128, 70)]


@pytest.mark.gpu
@pytest.mark.parametrize("spec,n,start", SPECS, ids=[s[0].name for s in SPECS])
def test_a_prompt_repeats_its_windows(spec, n, start):
    spec = dataclasses.replace(spec, n_layers=2, vocab=512, max_seq=288, eos_id=2)
    weights = dv2.DeviceWeights.random(spec, seed=3)
    ids = [int(t) for t in np.random.default_rng(1).integers(0, spec.vocab, size=start + n)]
    states = [dv2.DecodeState.allocate(spec, device="cuda") for _ in range(2)]
    for state, together in zip(states, (True, False)):
        pre = dv2.ChunkPrefill(state, weights)
        assert pre.whole_windows(127) == 0 and pre.whole_windows(200) == 192
        assert dv2.ChunkPrefill(state, weights, width=32).whole_windows(200) == 0
        if not together:
            pre.whole_windows = lambda n: 0
        if start:
            dv2.consume_prompt(state, weights, ids[:start], prefill=pre)
        dv2.consume_prompt(state, weights, ids[start:], start=start, prefill=pre)
        with pytest.raises(ValueError):
            pre.run_windows(torch.zeros(100, dtype=torch.long), 0)
    a, b = states
    assert int(a.position.item()) == int(b.position.item()) == start + n
    assert torch.equal(a.kv.k, b.kv.k) and torch.equal(a.kv.v, b.kv.v)
    assert torch.equal(a.arena.logits, b.arena.logits) and int(a.next_token.item()) == int(b.next_token.item())


@pytest.mark.gpu
def test_a_prompt_of_several_passes(monkeypatch):
    """More tokens than one pass takes: two whole passes, one of a single window, and a remainder."""
    spec = dataclasses.replace(dv2.QWEN25_14B, n_layers=2, vocab=512, max_seq=384, eos_id=2)
    weights = dv2.DeviceWeights.random(spec, seed=3)
    ids = [int(t) for t in np.random.default_rng(2).integers(0, spec.vocab, size=347)]
    states = []
    for per_pass in (128, 2048):
        monkeypatch.setattr(dv2.ChunkPrefill, "PASS_MAX", per_pass)
        state = dv2.DecodeState.allocate(spec, device="cuda")
        pre = dv2.ChunkPrefill(state, weights)
        assert pre.whole_windows(340) == 320
        dv2.consume_prompt(state, weights, ids[:7], prefill=pre)
        dv2.consume_prompt(state, weights, ids[7:], start=7, prefill=pre)
        states.append(state)
    a, b = states
    assert int(a.position.item()) == int(b.position.item()) == 347
    assert torch.equal(a.kv.k, b.kv.k) and torch.equal(a.kv.v, b.kv.v) and torch.equal(a.arena.logits, b.arena.logits)


# the sizes of a long prompt: 28 token tiles, splits and none, three matrices
@pytest.mark.gpu
@pytest.mark.parametrize("ms,k,kind", [((5120, 1024, 1024), 5120, 0), ((5120,), 5120, 2), ((2048,), 11008, 2), ((13824, 13824), 5120, 1)])
def test_products_of_a_long_prompt(ms, k, kind):
    n = 1792
    mats = [matrix(m, k, i) for i, m in enumerate(ms)]
    x = rand(n, k, seed=5).to(BF16)
    assert nf4.dv2_prompt_serves(mats, k, kind)
    if kind == 0:
        assert torch.equal(nf4.dv2_prompt_gemm(mats, x, k), windows(lambda at: nf4.dv2_gemm_qkv(*mats, cols(x[at])), n))
    elif kind == 1:
        assert torch.equal(nf4.dv2_prompt_gemm(mats, x, k, swiglu=True),
                           windows(lambda at: nf4.dv2_gemm_swiglu(*mats, cols(x[at])), n))
    else:
        m = ms[0]
        res, g = rand(n, m, seed=3).to(BF16), rand(m, seed=4).to(BF16)
        sums, norms = [], []
        for lo in range(0, n, 64):
            sq = torch.zeros(nf4.dv2_sq_blocks(m, 64) * 64, device="cuda")
            y, written = nf4.nf4_gemm(*mats[0][:2], cols(x[lo:lo + 64]), m, k, k, 64, residual=cols(res[lo:lo + 64]), colsq=sq)
            assert written
            sums.append(y.t())
            norms.append(nf4.dv2_rms_cols(y, g, 1e-6, colsq=sq).t())
        h = nf4.dv2_prompt_add_rms(*mats[0][:2], x, m, k, res, norm_w=g)
        assert torch.equal(res, torch.cat(sums)) and torch.equal(h, torch.cat(norms))


# rows 2 i and 2 i + 1 of a tile in two matrices, workgroups of a single chunk of K and of two
@pytest.mark.gpu
@pytest.mark.parametrize("n,ms,k", [(64, (5120, 1021, 1027), 5120), (128, (4100,), 256), (64, (2048,), 1024),
                                    (64, (4100,), 1280)])
def test_products_at_the_ends_of_the_pipeline(n, ms, k):
    mats = [matrix(m, k, i) for i, m in enumerate(ms)]
    x = rand(n, k, seed=5).to(BF16)
    assert nf4.dv2_prompt_serves(mats, k, 0)
    if len(ms) == 3:
        want = windows(lambda at: nf4.dv2_gemm_qkv(*mats, cols(x[at])), n)
    else:
        want = windows(lambda at: nf4.nf4_gemm(*mats[0][:2], cols(x[at]), ms[0], k, k, 64), n)
    assert torch.equal(nf4.dv2_prompt_gemm(mats, x, k), want)
