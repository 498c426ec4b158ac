"""One library call a layer of the decode step: the bits of the five calls it stands for."""

from __future__ import annotations

import ctypes
import dataclasses

import pytest
import torch

from deepfold_amd import decodev2 as dv2
from deepfold_amd import nf4
from deepfold_amd.decodev2 import step as step_mod


def test_null_and_bad_layers_are_refused():
    lib = nf4._load_ext()
    layer, step = nf4._Layer(), nf4._Step()
    assert lib.chr_dv2_step_layer(None, ctypes.byref(step), None) == -1
    assert lib.chr_dv2_step_layer(ctypes.byref(layer), None, None) == -1
    layer.qkv_rows = 2
    assert lib.chr_dv2_step_layer(ctypes.byref(layer), ctypes.byref(step), None) == -3
    layer.qkv_rows = 1
    assert lib.chr_dv2_step_layer(ctypes.byref(layer), ctypes.byref(step), None) == -1  # the first launch's code


def five_calls(state, weights, sq):
    ar, eps = state.arena, state.spec.rms_eps
    for li, ly in enumerate(weights.layers):
        q, k, v = step_mod._qkv(state, ly, ar.x, ly.norm1, sq)
        step_mod._attend_into_o(state, li, ly, q, k, v, sq)
        nf4.nf4_swiglu(ly.gate.packed, ly.gate.scale, ly.up.packed, ly.up.scale, ar.x.view(-1), ly.gate.M, ly.gate.K,
                       ly.gate.K_pad, ar.down_in.view(-1), ly.norm2, eps, sumsq_in=sq)
        step_mod._gemv_accum(ly.down, ar.down_in, ar.x, sq)


@pytest.mark.gpu
@pytest.mark.parametrize("spec", [dv2.QWEN25_3B, dv2.INTERNLM25_20B], ids=lambda s: s.name)
def test_layer_call_repeats_the_separate_calls(spec, monkeypatch):
    spec = dataclasses.replace(spec, n_layers=3, vocab=640, max_seq=64, eos_id=2)
    weights = dv2.DeviceWeights.random(spec, seed=5)
    answers = []
    for native in (True, False):
        calls = []
        real = step_mod._layers_native if native else five_calls
        monkeypatch.setattr(step_mod, "_layers_native", lambda *a: (calls.append(1), real(*a)))
        state = dv2.DecodeState.allocate(spec, device="cuda")
        logits = []
        for token in (3, 77, 600, 9):
            dv2.teacher_force_token(state, weights, token)
            logits.append(state.arena.logits.clone())
        assert len(calls) == 4                       # this model's step hands its sums over
        answers.append((torch.cat(logits), state.kv.k.clone(), state.kv.v.clone()))
        monkeypatch.undo()
    for a, b in zip(*answers):
        assert torch.equal(a, b)
    # what the separate calls refuse stays refused
    state = dv2.DecodeState.allocate(spec, device="cuda")
    good = weights.layers[1].gate
    for bad in (dataclasses.replace(good, packed=good.packed.to(torch.int16)),
                dataclasses.replace(good, packed=good.packed.reshape(-1)[:-64]),
                dataclasses.replace(good, scale=good.scale.cpu())):
        weights.layers[1].gate = bad
        with pytest.raises(RuntimeError):
            dv2.teacher_force_token(state, weights, 3)
    weights.layers[1].gate = good
