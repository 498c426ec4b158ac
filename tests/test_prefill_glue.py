"""GPU parity of the feature-major prefill glue (RMSNorm, RoPE + cache write, chunk
attention, SwiGLU, bias/residual) and of the chunked prefill built from it."""

from __future__ import annotations

import numpy as np
import pytest
import torch
import torch.nn.functional as F

from deepfold_amd import decodev2 as dv2
from deepfold_amd import nf4
from deepfold_amd.decodev2.synth import build
from oracle import nf4_oracle as oc
from oracle import step_oracle as so

from helpers import DEV, bf16_bits, bf16_tensor, to_f32, up, up_scale
from test_nf4_kernels import attn_ref, rope_tables, rot_half

pytestmark = pytest.mark.gpu


def say(*a):
    print(*a, flush=True)


def rnd(shape, seed, scale=1.0):
    rng = np.random.default_rng(seed)
    return oc.bf16_round((rng.standard_normal(shape) * scale).astype(np.float32))


# (13824, 64): more rows per workgroup than one pass of its threads writes out
@pytest.mark.parametrize("rows,n", [(64, 1), (256, 7), (5120, 32), (1000, 16), (2050, 31), (5120, 64), (300, 40),
                                    (13824, 64)])
def test_rms_cols(rows, n):
    say("rms_cols", rows, n)
    x = rnd((rows, n), rows + n, 1.5)
    w = rnd((rows,), 3, 1.0)
    eps = 1e-6
    got = to_f32(nf4.dv2_rms_cols(bf16_tensor(x), bf16_tensor(w), eps))
    x64 = x.astype(np.float64)
    ref = x64 * w.astype(np.float64)[:, None] / np.sqrt((x64 ** 2).mean(axis=0, keepdims=True) + eps)
    assert np.abs(got - ref).max() <= 2 ** -7 * max(1.0, np.abs(ref).max())
    # the N=1 kernel of the decode step is the same arithmetic, column by column
    for c in (0, n - 1):
        y = torch.empty(rows, dtype=torch.bfloat16, device=DEV)
        nf4.nf4_rms(bf16_tensor(np.ascontiguousarray(x[:, c])), bf16_tensor(w), y, eps)
        assert np.abs(to_f32(y) - got[:, c]).max() <= 2 ** -7 * max(1.0, np.abs(ref).max())
    # library cross-check
    t = F.rms_norm(bf16_tensor(np.ascontiguousarray(x.T)).float(), (rows,), bf16_tensor(w).float(), eps)
    assert np.abs(got - t.cpu().numpy().T).max() <= 2 ** -7 * max(1.0, np.abs(ref).max())


# 32 and 16 chains a column, rows that end inside a step and inside a batch of 32, above and below the lines from which
# the library takes two launches (1536 rows up to 31 columns, 1024 from 33 on) and the wrapper asks for them
@pytest.mark.parametrize("rows,n", [(5120, 17), (1024, 31), (1025, 24), (1536, 31), (1569, 24), (5120, 63), (1039, 33),
                                    (4099, 50), (1023, 40)])
def test_rms_cols_in_two_launches(rows, n):
    say("rms_cols two launches", rows, n)
    x, w = bf16_tensor(rnd((rows, n), rows + n, 1.5)), bf16_tensor(rnd((rows,), 3, 1.0))
    one = torch.empty_like(x)
    lib = nf4._load_ext()
    assert lib.chr_dv2_rms_cols(x.data_ptr(), w.data_ptr(), one.data_ptr(), rows, n, 1e-6, nf4._stream()) == 0
    assert torch.equal(nf4.dv2_rms_cols(x, w, 1e-6), one)
    two, ws = torch.zeros_like(x), torch.full((lib.chr_dv2_rms_cols_ws_floats(),), float("nan"), device=DEV)
    assert lib.chr_dv2_rms_cols_ws(x.data_ptr(), w.data_ptr(), two.data_ptr(), rows, n, 1e-6, ws.data_ptr(), nf4._stream()) == 0
    assert torch.equal(two, one)
    assert torch.isnan(ws).all().item() == (lib.chr_dv2_rms_cols_ws_for(rows, n, 1) == 0)
    assert lib.chr_dv2_rms_cols_ws(x.data_ptr(), w.data_ptr(), one.data_ptr(), rows, n, 1e-6, None, None) == -1


def test_rms_cols_rejects_wide_chunks():
    x = torch.zeros((64, 65), dtype=torch.bfloat16, device=DEV)
    with pytest.raises(RuntimeError):
        nf4.dv2_rms_cols(x, torch.ones(64, dtype=torch.bfloat16, device=DEV), 1e-6)


@pytest.mark.parametrize("n_q,n_kv,hd,n,start", [(4, 2, 16, 5, 0), (16, 2, 128, 32, 40),
                                                 (6, 3, 256, 3, 61), (8, 8, 64, 32, 0), (8, 2, 64, 64, 17)])
def test_rope_kv_cols(n_q, n_kv, hd, n, start):
    say("rope_kv_cols", n_q, n_kv, hd, n, start)
    max_seq = 96
    cos, sin = rope_tables(max_seq, hd)
    q = rnd((n_q * hd, n), 1)
    k = rnd((n_kv * hd, n), 2)
    v = rnd((n_kv * hd, n), 3)
    kc = torch.zeros((max_seq, n_kv, hd), dtype=torch.bfloat16, device=DEV)
    vc = torch.zeros_like(kc)
    q_rows = torch.zeros((n, n_q * hd), dtype=torch.bfloat16, device=DEV)
    dcos, dsin = bf16_tensor(cos), bf16_tensor(sin)
    nf4.dv2_rope_kv_cols(bf16_tensor(q), bf16_tensor(k), bf16_tensor(v), q_rows, kc, vc, dcos, dsin,
                         torch.tensor(start, dtype=torch.int64, device=DEV))
    for t in range(n):
        c, s = cos[start + t], sin[start + t]
        qr = rot_half(q[:, t].reshape(n_q, hd).astype(np.float64), c, s)
        kr = rot_half(k[:, t].reshape(n_kv, hd).astype(np.float64), c, s)
        assert np.abs(to_f32(q_rows[t]).reshape(n_q, hd) - qr).max() <= 2 ** -6
        assert np.abs(to_f32(kc[start + t]) - kr).max() <= 2 ** -6
        assert (to_f32(vc[start + t]) == v[:, t].reshape(n_kv, hd)).all()
        # bit for bit the decode step's one-token kernel
        dq = bf16_tensor(np.ascontiguousarray(q[:, t]).reshape(n_q, hd))
        dk = bf16_tensor(np.ascontiguousarray(k[:, t]).reshape(n_kv, hd))
        dv = bf16_tensor(np.ascontiguousarray(v[:, t]).reshape(n_kv, hd))
        kc1 = torch.zeros_like(kc)
        vc1 = torch.zeros_like(kc)
        nf4.nf4_rope_kv(dq, dk, dv, kc1, vc1, dcos, dsin,
                        torch.tensor(start + t, dtype=torch.int64, device=DEV))
        assert (bf16_bits(dq).reshape(-1) == bf16_bits(q_rows[t]).reshape(-1)).all()
        assert (bf16_bits(kc1[start + t]) == bf16_bits(kc[start + t])).all()
    assert (to_f32(kc[:start]) == 0).all() and (to_f32(kc[start + n:]) == 0).all()
    assert (to_f32(vc[:start]) == 0).all() and (to_f32(vc[start + n:]) == 0).all()


def test_rope_kv_cols_skips_rows_past_the_cache():
    n_q, n_kv, hd, n, max_seq = 2, 1, 16, 4, 8
    cos, sin = rope_tables(max_seq, hd)
    kc = torch.zeros((max_seq, n_kv, hd), dtype=torch.bfloat16, device=DEV)
    vc = torch.zeros_like(kc)
    q_rows = torch.zeros((n, n_q * hd), dtype=torch.bfloat16, device=DEV)
    nf4.dv2_rope_kv_cols(bf16_tensor(rnd((n_q * hd, n), 1)), bf16_tensor(rnd((n_kv * hd, n), 2)),
                         bf16_tensor(rnd((n_kv * hd, n), 3)), q_rows, kc, vc, bf16_tensor(cos),
                         bf16_tensor(sin), torch.tensor(6, dtype=torch.int64, device=DEV))
    torch.cuda.synchronize()
    assert (to_f32(kc[:6]) == 0).all() and (to_f32(kc[6:]) != 0).any()
    assert (to_f32(q_rows[2:]) == 0).all()


@pytest.mark.parametrize("n_q,n_kv,hd,max_seq,first,n,waves", [
    (4, 2, 16, 64, 1, 8, 16), (16, 2, 128, 256, 100, 32, 16), (40, 8, 128, 600, 481, 32, 16),
    (6, 3, 256, 80, 40, 5, 4), (4, 2, 48, 64, 1, 32, 1), (8, 8, 64, 40, 9, 32, 16),
    # grouped-query models with at most 8 wavefronts: cache rows shared by the heads of a KV head
    (40, 8, 128, 600, 481, 32, 4), (16, 2, 128, 256, 100, 64, 8), (4, 2, 64, 96, 30, 17, 4),
    (12, 2, 64, 128, 1, 64, 2), (8, 2, 128, 200, 130, 9, 1), (10, 2, 128, 64, 3, 5, 3)])
def test_attn_chunk(n_q, n_kv, hd, max_seq, first, n, waves):
    say("attn_chunk", n_q, n_kv, hd, max_seq, first, n, waves)
    q = rnd((n, n_q * hd), 11)
    kc = rnd((max_seq, n_kv, hd), 12)
    vc = rnd((max_seq, n_kv, hd), 13)
    last = first + n - 1
    kc[last:] = 1e4  # rows no token of the chunk may see
    vc[last:] = -1e4
    scale = hd ** -0.5
    dq, dk, dv = bf16_tensor(q), bf16_tensor(kc), bf16_tensor(vc)
    fl = torch.tensor(first, dtype=torch.int32, device=DEV)
    out_f = torch.zeros((n_q * hd, n), dtype=torch.bfloat16, device=DEV)
    out_t = torch.zeros((n, n_q * hd), dtype=torch.bfloat16, device=DEV)
    nf4.dv2_attn_chunk(dq, dk, dv, out_f, fl, scale, n_waves=waves)
    nf4.dv2_attn_chunk(dq, dk, dv, out_t, fl, scale, n_waves=waves, feature_major=False)
    assert (bf16_bits(out_f.t().contiguous()) == bf16_bits(out_t)).all()
    got = to_f32(out_t)
    one = torch.zeros(n_q * hd, dtype=torch.bfloat16, device=DEV)
    for t in range(n):
        ref = attn_ref(q[t].reshape(n_q, hd).astype(np.float64), kc.astype(np.float64),
                       vc.astype(np.float64), first + t, scale, n_q // n_kv)
        assert np.abs(got[t].reshape(n_q, hd) - ref).max() <= 0.02, t
        # bit for bit the decode step's attention at the same prefix length
        nf4.dv2_attn(dq[t].view(n_q, hd), dk, dv, one, torch.tensor(first + t, dtype=torch.int32, device=DEV), scale,
                     n_waves=waves)
        assert (bf16_bits(one) == bf16_bits(out_t[t])).all(), t


@pytest.mark.parametrize("n_q,n_kv,max_seq,first,n,odd", [
    (8, 8, 96, 40, 33, False),    # one query head a KV head: 16 tokens a tile, two tiles and one query
    (6, 2, 130, 1, 64, False),    # three: a tile begins inside a token; rows end on and around whole tiles of 64
    (40, 8, 200, 0, 2, False),    # the first token sees nothing
    (40, 8, 200, 14, 4, False), (16, 2, 200, 46, 3, False),  # the last tile ends around a step of 16 rows
    (40, 8, 200, 63, 5, False), (16, 2, 200, 126, 4, False), (34, 2, 80, 30, 9, False), (4, 4, 64, 60, 9, False),
    (40, 8, 320, 250, 70, True), (6, 2, 150, 20, 40, True), (1, 1, 70, 30, 17, True)])
def test_attn_chunk_on_the_matrix_cores(n_q, n_kv, max_seq, first, n, odd):
    """Four wavefronts, 128 dims: every token has the bits of the decode step's kernel, also where rows behind a
    token's own (``odd``: and rows it sees) hold infinities and NaN.  Which of the forms a chunk of this kind takes
    hangs on its heads and tokens; test_attn_chunk_form.py runs this test where each is sure to be taken."""
    say("attn_chunk, 128 dims", n_q, n_kv, max_seq, first, n, odd)
    q, kc, vc = rnd((n, n_q * 128), 31, 2.0), rnd((max_seq, n_kv, 128), 32), rnd((max_seq, n_kv, 128), 33)
    last = min(first + n - 1, max_seq)
    kc[last:], vc[last:] = np.nan, np.inf
    if odd:
        vc[first + n // 2, :, 5], vc[first + n // 2 + 1, 0, 7], vc[first - 3, 0, 100:103] = np.nan, np.inf, -np.inf
        kc[last - 2] = np.nan
    dq, dk, dv = bf16_tensor(q), bf16_tensor(kc), bf16_tensor(vc)
    out = torch.zeros((n, n_q * 128), dtype=torch.bfloat16, device=DEV)
    nf4.dv2_attn_chunk(dq, dk, dv, out, torch.tensor(first, dtype=torch.int32, device=DEV), 128 ** -0.5, n_waves=4,
                       feature_major=False)
    one = torch.zeros(n_q * 128, dtype=torch.bfloat16, device=DEV)
    for t in range(n):
        nf4.dv2_attn(dq[t].view(n_q, 128), dk, dv, one, torch.tensor(first + t, dtype=torch.int32, device=DEV),
                     128 ** -0.5, n_waves=4)
        nan = torch.isnan(one)
        assert odd or not nan.any(), t
        assert torch.equal(nan, torch.isnan(out[t])), t
        assert (bf16_bits(one.masked_fill(nan, 0)) == bf16_bits(out[t].masked_fill(nan, 0))).all(), t


def test_attn_chunk_clamps_to_the_cache():
    n_q, n_kv, hd, max_seq, n = 2, 1, 16, 8, 4
    q, kc, vc = rnd((n, n_q * hd), 1), rnd((max_seq, n_kv, hd), 2), rnd((max_seq, n_kv, hd), 3)
    out = torch.zeros((n, n_q * hd), dtype=torch.bfloat16, device=DEV)
    nf4.dv2_attn_chunk(bf16_tensor(q), bf16_tensor(kc), bf16_tensor(vc), out,
                       torch.tensor(7, dtype=torch.int32, device=DEV), hd ** -0.5, feature_major=False)
    ref = attn_ref(q[3].reshape(n_q, hd).astype(np.float64), kc.astype(np.float64),
                   vc.astype(np.float64), max_seq, hd ** -0.5, 2)
    assert np.abs(to_f32(out[3]).reshape(n_q, hd) - ref).max() <= 0.02


@pytest.mark.parametrize("shape", [(13824, 32), (100, 3), (1, 1)])
def test_swiglu_elems(shape):
    g, u = rnd(shape, 5, 2.0), rnd(shape, 6, 1.0)
    got = nf4.dv2_swiglu_elems(bf16_tensor(g), bf16_tensor(u))
    want = F.silu(bf16_tensor(g)) * bf16_tensor(u)
    d = np.abs(to_f32(got) - to_f32(want))
    # expf against torch's exponential: at most one bf16 step of the result
    assert (d <= 2 ** -7 * np.maximum(np.abs(to_f32(want)), 2 ** -20)).all()
    g64 = g.astype(np.float64)
    ref = g64 / (1 + np.exp(-g64)) * u
    assert np.abs(to_f32(got) - ref).max() <= 2 ** -6 * max(1.0, np.abs(ref).max())


def test_add_cols():
    rows, n = 300, 17
    y, a, b = rnd((rows, n), 1), rnd((rows, n), 2), rnd((rows,), 3)
    dy, da, db = bf16_tensor(y), bf16_tensor(a), bf16_tensor(b)
    want = dy + (da + db[:, None])
    nf4.dv2_add_cols(dy, da, db)
    assert (bf16_bits(dy) == bf16_bits(want)).all()
    dy = bf16_tensor(y)
    nf4.dv2_add_cols(dy, da)
    assert (bf16_bits(dy) == bf16_bits(bf16_tensor(y) + da)).all()
    dy = bf16_tensor(y)
    nf4.dv2_add_cols(dy, bias=db)
    assert (bf16_bits(dy) == bf16_bits(bf16_tensor(y) + db[:, None])).all()
    with pytest.raises(RuntimeError):
        nf4.dv2_add_cols(dy)


@pytest.mark.parametrize("m,k,n", [(256, 512, 8), (130, 1088, 5), (5120, 5120, 32), (384, 256, 2)])
def test_gemm_with_bias_and_residual_in_its_reduction(m, k, n):
    say("gemm_add", m, k, n)
    rng = np.random.default_rng(m + n)
    p, s_ = oc.c_encode((rng.standard_normal((m, k)) * 0.05).astype(np.float32))
    dp, ds = up(p), up_scale(s_)
    kp = p.shape[1] * 2
    x = bf16_tensor(rnd((k, n), 1))
    bias = bf16_tensor(rnd((m,), 2))
    res = rnd((m, n), 3)
    plain = nf4.nf4_gemm(dp, ds, x, m, k, kp)
    for use_bias, use_res in ((True, False), (False, True), (True, True)):
        want = plain
        if use_bias:
            want = want + bias[:, None]
        r = bf16_tensor(res)
        if use_res:
            want = r + want
        got = nf4.nf4_gemm(dp, ds, x, m, k, kp, bias=bias if use_bias else None,
                           residual=r if use_res else None)
        assert (bf16_bits(got) == bf16_bits(want)).all(), (use_bias, use_res)
        if use_res:
            assert got.data_ptr() == r.data_ptr()  # added in place
    with pytest.raises(RuntimeError):
        nf4.nf4_gemm(dp, ds, x[:, :1].contiguous(), m, k, kp, bias=bias)


# (13824, 1088, 64): 54 blocks of column sums per thread of the norm, more than one batch of loads
@pytest.mark.parametrize("m,k,n", [(5120, 5120, 64), (5120, 13824, 32), (2050, 1088, 16), (130, 5120, 8),
                                   (5120, 5120, 40), (256, 128, 64), (13824, 1088, 64),
                                   # the tile that finishes its rows itself leaves the sums too:
                                   # unsplit, with ragged row blocks, and at 16 columns (where it does not)
                                   (7168, 5120, 32), (5000, 5120, 64), (4999, 5120, 32), (13824, 5120, 64),
                                   (7168, 5120, 16)])
def test_gemm_leaves_column_sums_for_the_norm(m, k, n):
    """The split-K reduce that stores y also leaves y's column sums of squares per block of
    rows, and so does the tile that finishes its rows itself at 32 and 64 columns; the RMSNorm
    that takes them gives what the one that reads the tile gives."""
    say("gemm_add_sq", m, k, n)
    rng = np.random.default_rng(m + k + n)
    p, s_ = oc.c_encode((rng.standard_normal((m, k)) * 0.05).astype(np.float32))
    dp, ds = up(p), up_scale(s_)
    kp = p.shape[1] * 2
    x = bf16_tensor(rnd((k, n), 1))
    res = rnd((m, n), 3, 2.0)
    blocks = nf4.dv2_sq_blocks(m, n)
    per = 1024 // n if 1024 % n == 0 else 0
    colsq = torch.full((max(1, blocks) * n,), float("nan"), dtype=torch.float32, device=DEV)
    r0 = bf16_tensor(res)
    want = nf4.nf4_gemm(dp, ds, x, m, k, kp, 64, residual=r0)
    r1 = bf16_tensor(res)
    got, written = nf4.nf4_gemm(dp, ds, x, m, k, kp, 64, residual=r1, colsq=colsq)
    assert (bf16_bits(got) == bf16_bits(want)).all()  # same product, same roundings
    plan = nf4.nf4_plan(m, k, n)
    split = plan["grid_y"]
    in_tile = plan["block"] == 1024 and plan["bm"] in (32, 64) and n in (32, 64)
    assert written == (256 % n == 0 and (split > 1 or in_tile)), (written, plan)
    if not written:
        return
    y = to_f32(got).astype(np.float64)
    sq = colsq[: blocks * n].view(blocks, n).double().cpu().numpy()
    for b in (0, blocks // 2, blocks - 1):
        ref = (y[per * b: per * b + per] ** 2).sum(axis=0)
        assert np.abs(sq[b] - ref).max() <= 1e-5 * max(1.0, ref.max()), b
    w = bf16_tensor(rnd((m,), 4))
    a = nf4.dv2_rms_cols(got, w, 1e-6)
    b_ = nf4.dv2_rms_cols(got, w, 1e-6, colsq=colsq)
    # the two sums differ in order only: at most one bf16 step where a value sits on a tie
    da = np.abs(to_f32(a) - to_f32(b_))
    assert (da <= 2 ** -7 * np.maximum(np.abs(to_f32(a)), 2.0 ** -20)).all()
    assert (da > 0).mean() < 0.01


@pytest.mark.parametrize("m,k,n", [(256, 512, 64), (130, 1088, 33), (5120, 5120, 64), (384, 256, 40),
                                   (13824, 5120, 48)])
def test_wide_chunk_equals_two_narrow_ones(m, k, n):
    """33..64 columns in one pass over the weights: every column must come out as it does
    from the 32-column tile (same K order, same split)."""
    say("gemm wide", m, k, n)
    rng = np.random.default_rng(m + n)
    p, s_ = oc.c_encode((rng.standard_normal((m, k)) * 0.05).astype(np.float32))
    dp, ds = up(p), up_scale(s_)
    kp = p.shape[1] * 2
    x = bf16_tensor(rnd((k, n), 1))
    wide = nf4.nf4_gemm(dp, ds, x, m, k, kp, max_n=64)
    lo = nf4.nf4_gemm(dp, ds, x[:, :32].contiguous(), m, k, kp)
    first = min(32, n - 2)  # at least two columns: one alone would go to the GEMV
    hi = nf4.nf4_gemm(dp, ds, x[:, first:].contiguous(), m, k, kp)
    assert tuple(wide.shape) == (m, n)
    # the same split by the same kernel (block size, rows per block and LDS bytes tell the
    # tiles and their forms apart)
    plans = [nf4.nf4_plan(m, k, c) for c in (n, 32, n - first)]
    same_split = len({(q["grid_y"], q["block"], q["bm"], q["smem_bytes"]) for q in plans}) == 1
    for got, want_ in ((wide[:, :32].contiguous(), lo), (wide[:, first:].contiguous(), hi.view(m, n - first))):
        if same_split:  # same K order, same partial sums: the same bits
            assert (bf16_bits(got) == bf16_bits(want_)).all()
        else:           # wider chunks split K less: equal up to the fp32 summation order
            d = (got.float() - want_.float()).abs().max().item()
            assert d <= 2 ** -7 * max(1.0, want_.float().abs().max().item())
    bias, res = bf16_tensor(rnd((m,), 2)), bf16_tensor(rnd((m, n), 3))
    want = res + (wide + bias[:, None])
    got = nf4.nf4_gemm(dp, ds, x, m, k, kp, max_n=64, bias=bias, residual=res)
    assert (bf16_bits(got) == bf16_bits(want)).all()
    with pytest.raises(RuntimeError):
        nf4.nf4_gemm(dp, ds, x, m, k, kp)  # the reference's ceiling without max_n


@pytest.fixture
def stream_wherever_it_fits():
    """The planner leaves launches of few weights to the split tiles; these cases want the
    tile whose workgroups finish their rows themselves on small stacks too."""
    nf4.nf4_gemm_stream_policy(1)
    yield
    nf4.nf4_gemm_stream_policy(0)


@pytest.mark.parametrize("mq,mk,k,n,bias", [(256, 64, 512, 8, True), (5120, 1024, 5120, 64, True),
                                            (130, 70, 1088, 5, False), (2048, 256, 2048, 32, False),
                                            (130, 70, 1024, 16, True),   # ragged 32-row blocks
                                            (6000, 1500, 512, 16, True),  # ragged 64-row blocks
                                            (600, 200, 4096, 32, False)])  # K over several workgroups
def test_stacked_qkv_equals_three_gemms(mq, mk, k, n, bias, stream_wherever_it_fits):
    say("gemm_qkv", mq, mk, k, n, bias)
    rng = np.random.default_rng(mq + n)
    mats = []
    for m in (mq, mk, mk):
        p, s_ = oc.c_encode((rng.standard_normal((m, k)) * 0.05).astype(np.float32))
        mats.append((up(p), up_scale(s_), m))
    kp = mats[0][0].shape[1] * 2
    x = bf16_tensor(rnd((k, n), 1))
    b = bf16_tensor(rnd((mq + 2 * mk,), 2)) if bias else None
    got = nf4.dv2_gemm_qkv(*mats, x, bias=b)
    assert tuple(got.shape) == (mq + 2 * mk, n)
    row = 0
    for packed, scale, m in mats:
        want = nf4.nf4_gemm(packed, scale, x, m, k, kp, max_n=64)
        if bias:
            want = want + b[row:row + m, None]
        # the stack has its own split-K (more row blocks, fewer splits): equal up to the
        # fp32 summation order
        d = (got[row:row + m].float() - want.float()).abs().max().item()
        assert d <= 2 ** -7 * max(1.0, want.float().abs().max().item()), (row, d)
        row += m
    with pytest.raises(RuntimeError):
        nf4.dv2_gemm_qkv(mats[0], mats[1], (mats[2][0], mats[2][1], mk + 1), x)


@pytest.mark.parametrize("m,k,n", [(256, 512, 8), (13824, 5120, 64), (130, 1088, 5), (384, 256, 2),
                                   (130, 1024, 24), (2048, 2048, 32),
                                   (4500, 512, 8), (13824, 5120, 32),  # 64-row blocks
                                   (512, 6144, 16)])                   # K over several workgroups
def test_stacked_gate_up_with_swiglu_in_the_reduce(m, k, n, stream_wherever_it_fits):
    say("gemm_swiglu", m, k, n)
    rng = np.random.default_rng(m + n)
    mats = []
    for _ in range(2):
        p, s_ = oc.c_encode((rng.standard_normal((m, k)) * 0.05).astype(np.float32))
        mats.append((up(p), up_scale(s_), m))
    kp = mats[0][0].shape[1] * 2
    x = bf16_tensor(rnd((k, n), 1))
    got = nf4.dv2_gemm_swiglu(mats[0], mats[1], x)
    g = nf4.nf4_gemm(mats[0][0], mats[0][1], x, m, k, kp, max_n=64)
    u = nf4.nf4_gemm(mats[1][0], mats[1][1], x, m, k, kp, max_n=64)
    want = F.silu(g) * u
    # the stack has its own split-K, so gate and up may each differ from the single GEMMs in
    # the last bf16 digit before the activation: 2^-7 (gate through silu) + 2^-8 (up) + two
    # roundings of 2^-9 is just over 2^-6 of the product
    d = (got.float() - want.float()).abs()
    tol = 2 ** -5 * torch.maximum(want.float().abs(), torch.full_like(d, 2 ** -10))
    assert tuple(got.shape) == (m, n) and bool((d <= tol).all())
    with pytest.raises(RuntimeError):
        nf4.dv2_gemm_swiglu(mats[0], (mats[1][0], mats[1][1], m - 1), x)


# ---- the chunked prefill built from them ------------------------------------------------

LONG = [4, 5, 6, 7, 1, 2, 3, 4]


def session(spec, seed, packed_embed=False):
    model = build(spec, seed, packed_embed=packed_embed)
    weights = dv2.DeviceWeights.from_synth(model, "cuda")
    state = dv2.DecodeState.allocate(spec, device="cuda")
    return model, state, weights


@pytest.mark.parametrize("spec,seed", [(dv2.TINY_LLAMA, 0), (dv2.TINY_INTERNLM, 1), (dv2.MEDIUM_LLAMA, 0)])
@pytest.mark.parametrize("use_graph", [False, True])
def test_feature_major_prefill_gives_the_oracle_ids(spec, seed, use_graph):
    say("chunk prefill", spec.name, use_graph)
    model, state, weights = session(spec, seed)
    want = so.greedy_ids(model, LONG, 6)
    pre = dv2.ChunkPrefill(state, weights, use_graph=use_graph)
    for chunk in (2, 3, 8, None):
        for _ in range(2):  # the second pass replays the graphs the first one captured
            state.reset()
            got = dv2.generate(state, weights, LONG, 6, chunk=chunk, prefill=pre)
            assert got == want, chunk
            assert int(state.valid_len.item()) == len(LONG) + len(got) - 1


def test_feature_major_prefill_tracks_the_torch_glue():
    spec = dv2.MEDIUM_LLAMA
    rng = np.random.default_rng(0)
    prompt = [int(t) for t in rng.integers(0, spec.vocab, size=min(70, spec.max_seq - 8))]
    _, a, w = session(spec, 2, packed_embed=True)
    b = dv2.DecodeState.allocate(spec, device="cuda")
    dv2.consume_prompt(a, w, prompt)
    pre = dv2.ChunkPrefill(b, w)
    dv2.consume_prompt(b, w, prompt, prefill=pre)
    n = len(prompt)
    assert int(a.valid_len.item()) == int(b.valid_len.item()) == n
    ka, kb = a.kv.k[:, :n].float(), b.kv.k[:, :n].float()
    va, vb = a.kv.v[:, :n].float(), b.kv.v[:, :n].float()
    assert (ka - kb).abs().max().item() <= 0.03 * max(1.0, ka.abs().max().item())
    assert (va - vb).abs().max().item() <= 0.03 * max(1.0, va.abs().max().item())
    la, lb = a.arena.logits.float().view(-1), b.arena.logits.float().view(-1)
    assert (la - lb).abs().max().item() <= 0.03 * max(1.0, la.abs().max().item())
    # a replay of the captured graphs on a fresh request gives the same bits as its first run
    first = b.kv.k[:, :n].clone(), b.arena.logits.clone()
    b.reset()
    dv2.consume_prompt(b, w, prompt, prefill=pre)
    assert torch.equal(first[0], b.kv.k[:, :n]) and torch.equal(first[1], b.arena.logits)


def test_sixty_four_token_chunks():
    spec = dv2.with_max_seq(dv2.MEDIUM_LLAMA, 256)
    rng = np.random.default_rng(1)
    prompt = [int(t) for t in rng.integers(0, spec.vocab, size=150)]
    model, a, w = session(spec, 4, packed_embed=True)
    b = dv2.DecodeState.allocate(spec, device="cuda")
    pre32 = dv2.ChunkPrefill(a, w, width=32)
    pre64 = dv2.ChunkPrefill(b, w)
    assert (pre32.width, pre64.width) == (32, 64)
    dv2.consume_prompt(a, w, prompt, prefill=pre32)   # 32+32+32+32+22
    dv2.consume_prompt(b, w, prompt, prefill=pre64)   # 64+64+22
    n = len(prompt)
    assert int(a.valid_len.item()) == int(b.valid_len.item()) == n
    # per column the wide GEMM tile computes what the narrow one does, but the RMSNorm sums
    # its squares in an order that depends on the chunk width: equal up to bf16 rounding
    for ta, tb in ((a.kv.k[:, :n], b.kv.k[:, :n]), (a.kv.v[:, :n], b.kv.v[:, :n]),
                   (a.arena.logits, b.arena.logits)):
        ta, tb = ta.float(), tb.float()
        assert (ta - tb).abs().max().item() <= 0.03 * max(1.0, ta.abs().max().item())
    # greedy ids follow the oracle until a pick whose top-two logits are nearly tied
    want, margins = so.greedy_ids(model, prompt[:70], 5, return_margins=True)
    thin = next((i for i, m in enumerate(margins) if m < 0.02), len(want))
    got = dv2.generate(b, w, prompt[:70], 5, prefill=pre64)
    assert thin >= 3 and got[:thin] == want[:thin]


def test_chunk_prefill_errors():
    spec = dv2.TINY_LLAMA
    _, state, w = session(spec, 0)
    pre = dv2.ChunkPrefill(state, w, use_graph=False)
    with pytest.raises(ValueError):
        pre.run(torch.zeros(0, dtype=torch.long), 0)
    with pytest.raises(ValueError):
        pre.run(torch.zeros(65, dtype=torch.long), 0)
    with pytest.raises(ValueError):
        pre.run(torch.zeros(4, dtype=torch.long), spec.max_seq - 2)
