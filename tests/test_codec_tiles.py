"""The codec kernels at the edges of their tiles, bit for bit against the CPU codec: rows that are no
whole 16-byte pieces, unaligned buffers, the last workgroup, and the quantiser at every value where
the nearest level changes."""

from __future__ import annotations

import ctypes

import numpy as np
import pytest
import torch

from deepfold_amd import nf4
from oracle import nf4_oracle as oc

pytestmark = pytest.mark.gpu


def weights(m, k, seed):
    return (np.random.default_rng(seed).standard_normal((m, k)) * 0.03).astype(np.float32)


# 16 groups (quantiser) and 1024 weights (decoder) x 4 a workgroup: one, one more, one less
@pytest.mark.parametrize("m,k", [(1, 1), (1, 63), (3, 66), (64, 64), (65, 64), (7, 1111), (4, 1028), (33, 1020), (129, 2047)])
@pytest.mark.parametrize("shift", [0, 1])
def test_both_ways_bit_exact(m, k, shift):
    w = weights(m, k, seed=m + k)
    p, s = oc.c_encode(w)
    kp = oc.k_pad(k)
    src = torch.zeros(m * k + shift, device="cuda")[shift:]          # shift: off the 16-byte grid
    src.copy_(torch.from_numpy(w).reshape(-1))
    packed = torch.zeros(m * kp // 2 + shift, dtype=torch.uint8, device="cuda")[shift:]   # and at an odd byte
    scale = torch.zeros(m * kp // 64, dtype=torch.float16, device="cuda")
    status = torch.zeros(1, dtype=torch.int32, device="cuda")
    d = nf4._Dev(m, k, kp, packed.data_ptr(), scale.data_ptr())
    lib, stream = nf4._load_ext(), torch.cuda.current_stream().cuda_stream
    assert lib.chr_nf4_quantize(src.data_ptr(), ctypes.byref(d), status.data_ptr(), stream) == 0
    assert int(status.item()) == 0
    assert np.array_equal(packed.cpu().numpy(), np.asarray(p).reshape(-1))
    assert np.array_equal(scale.cpu().numpy().view(np.uint16), np.asarray(s).view(np.uint16).reshape(-1))
    out = torch.full((m * k + shift,), float("nan"), device="cuda")[shift:]
    got = nf4.nf4_dequant(packed.clone(), scale, m, k, kp, out=out)
    assert np.array_equal(got.cpu().numpy().view(np.uint32), oc.c_decode(p, s, m, k).reshape(-1).view(np.uint32))


def test_every_change_of_level():
    levels = np.array([bits for bits in (
        0xBF800000, 0xBF3239B1, 0xBF066B30, 0xBECA32A0, 0xBE91A24D, 0xBE3D353F, 0xBDBA7871, 0x00000000, 0x3DA2FAFF,
        0x3E24CAE3, 0x3E7C04DD, 0x3EAD033A, 0x3EE1A4B8, 0x3F1007AB, 0x3F3913B3, 0x3F800000)], np.uint32).view(np.float32)
    mids = ((levels[1:].astype(np.float64) + levels[:-1]) / 2).astype(np.float32)
    borders = (np.arange(33) / 16 - 1).astype(np.float32)
    near = []
    for v in np.concatenate([levels, mids, borders]):
        up = down = np.float32(v)
        near.append(up)
        for _ in range(8):
            up, down = np.nextafter(up, np.float32(4)), np.nextafter(down, np.float32(-4))
            near += [up, down]
    near = np.clip(np.array(near, np.float32), -1, 1)
    near = np.concatenate([near, [0.0, -0.0, 1e-40, -1e-40, 1e-20]]).astype(np.float32)
    pad = -len(near) % 63
    body = np.concatenate([near, np.zeros(pad, np.float32)]).reshape(-1, 63)
    w = np.concatenate([np.ones((body.shape[0], 1), np.float32), body], axis=1)   # a scale of one: u is the weight
    for f in (1.0, 2.0 ** -20, 3.0, 65504.0, 1e6, 2.0 ** -24, 1e-9, 5e-8):
        x = (w * np.float32(f)).astype(np.float32)
        p, s = oc.c_encode(x)
        gp, gs = nf4.nf4_quantize(torch.from_numpy(x).cuda())
        assert np.array_equal(gp.cpu().numpy(), np.asarray(p)), f
        assert np.array_equal(gs.cpu().numpy().view(np.uint16), np.asarray(s).view(np.uint16)), f


# the quantiser divides only where the reciprocal's product lies within 2^-21 of a change of level: weights on both
# sides of that band, and within it, at scales whose reciprocal is rounded, at subnormal and at the largest ones
@pytest.mark.parametrize("lo,hi", [(1, 1024), (1024, 0x3C00), (0x3C00, 0x7C00)])
def test_the_reciprocal_and_the_division_choose_one_code(lo, hi):
    levels = oc.LUT.astype(np.float64)
    mids = (levels[1:] + levels[:-1]) / 2
    steps = np.array([0, 1, 2, 3, 7, 15, 29, 31, 32, 33, 35, 63]) * 2.0 ** -26
    u = (mids[:, None] + np.concatenate([steps, -steps])[None, :]).reshape(-1)
    u = np.concatenate([u, np.zeros(-len(u) % 63)]).reshape(-1, 63)
    rng = np.random.default_rng(lo)
    scales = np.concatenate([[lo, hi - 1], rng.integers(lo, hi, 62)]).astype(np.uint16).view(np.float16).astype(np.float64)
    w = np.concatenate([np.ones((len(u), 1)), u], axis=1)[None] * scales[:, None, None]
    w = w.reshape(-1, 64).astype(np.float32)
    p, s = oc.c_encode(w)
    gp, gs = nf4.nf4_quantize(torch.from_numpy(w).cuda())
    assert np.array_equal(gs.cpu().numpy().view(np.uint16), np.asarray(s).view(np.uint16).reshape(gs.shape))
    assert np.array_equal(gp.cpu().numpy(), np.asarray(p).reshape(gp.shape))


@pytest.mark.parametrize("bad", [float("nan"), float("inf"), float("-inf")])
def test_a_group_that_is_not_finite_is_left_alone(bad):
    w = weights(5, 130, seed=1)
    w[3, 70] = bad
    packed = torch.full((5, 96), 0xEE, dtype=torch.uint8, device="cuda")
    scale = torch.full((5, 3), 7.0, dtype=torch.float16, device="cuda")
    status = torch.zeros(1, dtype=torch.int32, device="cuda")
    src = torch.from_numpy(w).cuda()
    d = nf4._Dev(5, 130, 192, packed.data_ptr(), scale.data_ptr())
    assert nf4._load_ext().chr_nf4_quantize(src.data_ptr(), ctypes.byref(d), status.data_ptr(),
                                            torch.cuda.current_stream().cuda_stream) == 0
    assert int(status.item()) == 1
    w[3, 70] = 0.0
    p, s = (np.asarray(t).copy() for t in oc.c_encode(w))
    p.reshape(5, 3, 32)[3, 1] = 0xEE
    s.reshape(5, 3)[3, 1] = np.float16(7.0)
    assert np.array_equal(packed.cpu().numpy(), p.reshape(5, 96))
    assert np.array_equal(scale.cpu().numpy().view(np.uint16), s.view(np.uint16).reshape(5, 3))


# from 2^23 weights on the ragged decoder takes eight a thread, 2048 a workgroup: none of these counts is a multiple,
# one is a single weight above the line
@pytest.mark.parametrize("m,k,shift", [(1, (1 << 23) + 1, 0), (2100, 4003, 0), (2100, 4003, 1), (2050, 4096, 1)])
def test_ragged_decoder_of_many_weights(m, k, shift):
    kp = oc.k_pad(k)
    rng = np.random.default_rng(m)
    p = rng.integers(0, 256, size=(m, kp // 2), dtype=np.uint8)
    s = (rng.random((m, kp // 64)).astype(np.float16) * np.float16(0.1)).view(np.uint16)
    assert m * k >= 1 << 23 and (k % 4 != 0 or shift) and (m * k % 2048 != 0 or shift)
    room = torch.full((m * k + shift + 1,), float("nan"), device="cuda")
    out = room[shift:shift + m * k]
    got = nf4.nf4_dequant(torch.from_numpy(p).cuda(), torch.from_numpy(s.view(np.float16)).cuda(), m, k, kp, out=out)
    assert np.array_equal(got.cpu().numpy().view(np.uint32), oc.c_decode(p, s, m, k).reshape(-1).view(np.uint32))
    assert bool(torch.isnan(room[shift + m * k:]).all()) and bool(torch.isnan(room[:shift]).all())
