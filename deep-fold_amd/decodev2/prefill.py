"""Chunked prompt prefill (``gpu/decodev2/prefill.py:26-141``): at most 32 prompt
positions per pass, linears on the MFMA GEMM.

Two forms.  ``forward_prefill`` is the reference's sequence: token-major torch glue
around the GEMMs, never captured.  ``ChunkPrefill`` keeps every activation in the
GEMM's own feature-major ``[features, N]`` layout, runs the glue (RMSNorm, RoPE + cache
write, causal attention, SwiGLU, bias/residual) as library launches, and replays each
chunk width as a captured graph, so a layer costs its kernels and not the host's
dispatch."""

from __future__ import annotations

import torch

from ..nf4 import (LIVE_MAX_N, PLAN_MAX_N, dv2_add_cols, dv2_attn_chunk, dv2_gemm_qkv, dv2_gemm_swiglu,
                   dv2_prompt_add_rms, dv2_prompt_gemm, dv2_prompt_rms, dv2_prompt_serves, dv2_rms_cols,
                   dv2_rope_kv_cols, dv2_rope_kv_rows, dv2_sq_blocks, dv2_swiglu_elems, nf4_gemm)
from .embed import gather_embed
from .linear import DeviceLinear, DeviceWeights, nf4_linear
from .ops import causal_attend, rms, split_qkv, swiglu
from .rope import apply_rope_torch
from .state import DecodeState

__all__ = ["forward_prefill", "prefill_chunk_width", "ChunkPrefill"]


def prefill_chunk_width(state: DecodeState, chunk: int | None = None) -> int:
    cap = min(int(LIVE_MAX_N), int(state.spec.max_seq))
    return cap if chunk is None else max(1, min(int(chunk), cap))


def forward_prefill(state: DecodeState, weights: DeviceWeights, token_ids: torch.Tensor, start: int,
                    *, logits: bool = True) -> None:
    """Teacher-force ``token_ids`` into KV slots ``start..start+n-1``.  ``lm_head``
    runs only when ``logits`` (the last chunk), on the last row."""
    ids = token_ids.reshape(-1).to(device=state.device, dtype=torch.long)
    n = int(ids.numel())
    if n < 1:
        raise ValueError("prefill chunk must be non-empty")
    start = int(start)
    seq = start + n
    spec = state.spec
    if seq > spec.max_seq:
        raise ValueError(f"prefill {start}..{seq} exceeds max_seq={spec.max_seq}")
    x = gather_embed(weights.embed, ids)
    cos, sin = state.cos[start:seq], state.sin[start:seq]
    for li, layer in enumerate(weights.layers):
        h = rms(x, layer.norm1, spec.rms_eps)
        q, k, v = split_qkv(layer, h, spec)
        q = apply_rope_torch(q, cos, sin)
        k = apply_rope_torch(k, cos, sin)
        state.kv.write_range(li, start, k, v)
        k_all, v_all = state.kv.view(li, seq)
        attn = causal_attend(q, k_all, v_all, spec, start)
        x = x + nf4_linear(layer.o, attn)
        h = rms(x, layer.norm2, spec.rms_eps)
        x = x + nf4_linear(layer.down, swiglu(nf4_linear(layer.gate, h), nf4_linear(layer.up, h)))
    state.position.fill_(seq)
    state.valid_len.fill_(seq)
    if not logits:
        return
    hidden = rms(x[-1:], weights.final_norm, spec.rms_eps)
    state.arena.logits.copy_(nf4_linear(weights.lm_head, hidden).reshape(1, -1))
    state.pick_next(commit=False)


def _gemm_cols(mat: DeviceLinear, x: torch.Tensor, residual: torch.Tensor | None = None,
               colsq: torch.Tensor | None = None):
    """``[K, N] -> [M, N]`` with the bias, if any, added per row; with ``residual`` the
    result is added to it in place.  One column (a one-token chunk) goes to the GEMV and
    takes its bias and residual from separate launches.  With ``colsq`` the return value is
    whether the launch left the result's column sums of squares there."""
    if x.size(1) >= 2:
        if colsq is not None:
            return nf4_gemm(mat.packed, mat.scale, x, mat.M, mat.K, mat.K_pad, int(PLAN_MAX_N),
                            bias=mat.bias, residual=residual, colsq=colsq)[1]
        return nf4_gemm(mat.packed, mat.scale, x, mat.M, mat.K, mat.K_pad, int(PLAN_MAX_N),
                        bias=mat.bias, residual=residual)
    y = nf4_gemm(mat.packed, mat.scale, x, mat.M, mat.K, mat.K_pad)
    if mat.bias is not None:
        dv2_add_cols(y, bias=mat.bias)
    if residual is not None:
        dv2_add_cols(residual, y)
        return False if colsq is not None else residual
    return False if colsq is not None else y


def _plain(mats) -> bool:
    """Blobs laid out and aligned as the several-window products read them."""
    for m in mats:
        packed, scale = m.packed, m.scale
        if packed.data_ptr() & 15 or scale.data_ptr() & 7 or not (packed.is_contiguous() and scale.is_contiguous()):
            return False
    return True


class ChunkPrefill:
    """Feature-major prefill of one request's prompt chunks.

    ``run(ids, start, logits)`` has ``forward_prefill``'s contract.  All launches of a
    chunk read the chunk's ids, its first cache slot and the prefix length of its first
    token from fixed device buffers, so one captured graph per chunk width serves every
    position (``use_graph``); without graphs the same launches are issued eagerly.

    ``width`` is the chunk ``consume_prompt`` cuts prompts into: up to 64 tokens, twice the
    reference's 32, so the weights are streamed half as often (the 33..64-column GEMM tile
    dequantises each weight once for both 32-column blocks).

    ``run_windows`` takes several whole windows in one token-major pass, layer by layer, with
    the bits ``run`` leaves on one after the other; ``whole_windows(n)`` says how many of ``n``
    tokens ``consume_prompt`` sends there.  Such a pass is launched eagerly (``use_graph`` or not)
    and holds the activations of all its tokens."""

    MAX_WIDTH = int(PLAN_MAX_N)
    #: tokens of one pass over several windows: bounds its activations and partials
    PASS_MAX = 2048

    def __init__(self, state: DecodeState, weights: DeviceWeights, *, use_graph: bool = True,
                 width: int | None = None) -> None:
        self.state = state
        self.weights = weights
        self.use_graph = bool(use_graph)
        dev = state.device
        spec = state.spec
        cap = min(self.MAX_WIDTH, int(spec.max_seq))
        self.width = cap if width is None else max(1, min(int(width), cap))
        self.ids = torch.zeros(self.MAX_WIDTH, dtype=torch.long, device=dev)
        self.start = torch.zeros((), dtype=torch.int64, device=dev)
        self.first_len = torch.zeros((), dtype=torch.int32, device=dev)
        self.last_hidden = torch.zeros(spec.hidden, dtype=torch.bfloat16, device=dev)
        # column sums of squares of the residual stream, left by the launch that last wrote it
        self._colsq = torch.zeros(dv2_sq_blocks(spec.hidden, self.MAX_WIDTH) * self.MAX_WIDTH,
                                  dtype=torch.float32, device=dev)
        self._graphs: dict[int, torch.cuda.CUDAGraph] = {}
        # stacked q/k/v biases for the one-launch q/k/v GEMM (zeros where a matrix has none)
        self._qkv_bias: list[torch.Tensor | None] = []
        for layer in weights.layers:
            mats = (layer.q, layer.k, layer.v)
            if layer.wqkv is not None or all(m.bias is None for m in mats):
                self._qkv_bias.append(None)
            else:
                self._qkv_bias.append(torch.cat([
                    m.bias if m.bias is not None else torch.zeros(m.M, dtype=torch.bfloat16, device=dev)
                    for m in mats]).contiguous())

    def _serves_windows(self) -> bool:
        """Whether the products of the model are ones the pass over several windows repeats; gate and
        up may also go through it window by window.  The library is asked once per distinct shape, every
        layer's blobs are looked at (weights may be exchanged between prompts)."""
        spec = self.state.spec
        if spec.hidden % 16 != 0 or spec.hidden > 16384:
            return False
        seen = set()
        for ly in self.weights.layers:
            qkv = (ly.q, ly.k, ly.v) if ly.wqkv is None else (ly.wqkv,)
            if ly.gate.bias is not None or ly.up.bias is not None or (ly.wqkv is not None and ly.wqkv.bias is not None):
                return False
            mats = (*qkv, ly.o, ly.down)
            if not _plain(mats):
                return False
            shape = tuple([(m.M, m.K) for m in mats])
            if shape not in seen:
                seen.add(shape)
                if not all(dv2_prompt_serves([(m.packed, m.scale, m.M) for m in of], of[0].K, kind)
                           for kind, of in ((2, (ly.o,)), (0, qkv), (2, (ly.down,)))):
                    return False
        return True

    def whole_windows(self, n: int) -> int:
        """Tokens in front of an ``n``-token prompt that go through together: its whole windows,
        where there are two or more of the default width.  Two, as two graph replays and as one pass
        (ms): 3B 8.35 / 6.42, 14B 12.75 / 8.66, 32B 24.7 / 15.0, two layers of the 3B 0.66 / 0.58."""
        whole = int(n) - int(n) % self.MAX_WIDTH
        if self.width != self.MAX_WIDTH or whole < 2 * self.MAX_WIDTH or not self._serves_windows():
            return 0
        return whole

    def _windows_pass(self, ids: torch.Tensor, start: int) -> None:
        state, weights, spec = self.state, self.weights, self.state.spec
        n = int(ids.numel())
        x = gather_embed(weights.embed, ids)                                        # [n, hidden]
        attn = torch.empty((n, spec.q_dim), dtype=torch.bfloat16, device=x.device)
        h = dv2_prompt_rms(x, weights.layers[0].norm1, spec.rms_eps)
        together: dict = {}  # gate and up by shape: whether a launch takes all windows of them
        for li, layer in enumerate(weights.layers):
            qkv = (layer.wqkv,) if layer.wqkv is not None else (layer.q, layer.k, layer.v)
            y = dv2_prompt_gemm([(m.packed, m.scale, m.M) for m in qkv], h, spec.hidden, bias=self._qkv_bias[li])
            k_cache, v_cache = state.kv.layer(li)
            q = dv2_rope_kv_rows(y, spec.n_q, k_cache, v_cache, state.cos, state.sin, start)
            dv2_attn_chunk(q, k_cache, v_cache, attn, self.first_len, spec.attn_scale, feature_major=False)
            h = dv2_prompt_add_rms(layer.o.packed, layer.o.scale, attn, layer.o.M, layer.o.K, x, bias=layer.o.bias,
                                   norm_w=layer.norm2, eps=spec.rms_eps)
            gate, up = ((m.packed, m.scale, m.M) for m in (layer.gate, layer.up))
            shape = (layer.gate.M, layer.up.M, _plain((layer.gate, layer.up)))
            if shape not in together:
                together[shape] = shape[-1] and dv2_prompt_serves([gate, up], spec.hidden, 1)
            if together[shape]:
                act = dv2_prompt_gemm([gate, up], h, spec.hidden, swiglu=True)
            else:
                act = torch.empty((n, layer.gate.M), dtype=torch.bfloat16, device=x.device)
                for lo in range(0, n, self.MAX_WIDTH):
                    at = slice(lo, lo + self.MAX_WIDTH)
                    act[at] = dv2_gemm_swiglu(gate, up, h[at].t().contiguous()).t()
            last = li + 1 == len(weights.layers)
            h = dv2_prompt_add_rms(layer.down.packed, layer.down.scale, act, layer.down.M, layer.down.K, x,
                                   bias=layer.down.bias, norm_w=None if last else weights.layers[li + 1].norm1,
                                   eps=spec.rms_eps)
        self.last_hidden.copy_(x[n - 1])

    def _chunk(self, n: int) -> None:
        state, weights, spec = self.state, self.weights, self.state.spec
        x = gather_embed(weights.embed, self.ids[:n]).t().contiguous()  # [hidden, n]
        q_rows = torch.empty((n, spec.q_dim), dtype=torch.bfloat16, device=x.device)
        attn = torch.empty((spec.q_dim, n), dtype=torch.bfloat16, device=x.device)
        sq = None  # self._colsq while it holds x's sums (the embedding gather leaves none)
        for li, layer in enumerate(weights.layers):
            h = dv2_rms_cols(x, layer.norm1, spec.rms_eps, colsq=sq)
            if layer.wqkv is not None:
                y = _gemm_cols(layer.wqkv, h)  # rows are [Q | K | V]
                q, k, v = y[:spec.q_dim], y[spec.q_dim:spec.q_dim + spec.kv_dim], y[spec.q_dim + spec.kv_dim:]
            elif n >= 2:
                y = dv2_gemm_qkv(*((m.packed, m.scale, m.M) for m in (layer.q, layer.k, layer.v)), h,
                                 bias=self._qkv_bias[li])
                q, k, v = y[:spec.q_dim], y[spec.q_dim:spec.q_dim + spec.kv_dim], y[spec.q_dim + spec.kv_dim:]
            else:
                q, k, v = _gemm_cols(layer.q, h), _gemm_cols(layer.k, h), _gemm_cols(layer.v, h)
            k_cache, v_cache = state.kv.layer(li)
            dv2_rope_kv_cols(q, k, v, q_rows, k_cache, v_cache, state.cos, state.sin, self.start)
            dv2_attn_chunk(q_rows, k_cache, v_cache, attn, self.first_len, spec.attn_scale)
            sq = self._colsq if _gemm_cols(layer.o, attn, residual=x, colsq=self._colsq) else None
            h = dv2_rms_cols(x, layer.norm2, spec.rms_eps, colsq=sq)
            if n >= 2 and layer.gate.bias is None and layer.up.bias is None:
                act = dv2_gemm_swiglu((layer.gate.packed, layer.gate.scale, layer.gate.M),
                                      (layer.up.packed, layer.up.scale, layer.up.M), h)
            else:
                act = dv2_swiglu_elems(_gemm_cols(layer.gate, h), _gemm_cols(layer.up, h))
            sq = self._colsq if _gemm_cols(layer.down, act, residual=x, colsq=self._colsq) else None
        self.last_hidden.copy_(x[:, n - 1])

    def _replay(self, n: int) -> None:
        if not self.use_graph:
            self._chunk(n)
            return
        g = self._graphs.get(n)
        if g is None:
            # one eager pass first: it sizes the GEMM's dynamic LDS and warms the allocator
            self._chunk(n)
            g = torch.cuda.CUDAGraph()
            with torch.cuda.graph(g):
                self._chunk(n)
            self._graphs[n] = g
            return  # the capture pass does not run; the eager pass above already did the work
        g.replay()

    def run(self, token_ids: torch.Tensor, start: int, *, logits: bool = True) -> None:
        ids, start = self._checked(token_ids, start)
        n = int(ids.numel())
        if n > self.MAX_WIDTH:
            raise ValueError(f"prefill chunk of {n} tokens exceeds {self.MAX_WIDTH}")
        self.ids[:n].copy_(ids)
        self.start.fill_(start)
        self.first_len.fill_(start + 1)
        self._replay(n)
        self._finish(start + n, logits)

    def run_windows(self, token_ids: torch.Tensor, start: int, *, logits: bool = True) -> None:
        n = int(token_ids.numel())
        if self.whole_windows(n) != n:
            raise ValueError(f"{n} tokens are not two or more whole windows this model takes together")
        self._run_windows(token_ids, start, logits=logits)

    def _run_windows(self, token_ids: torch.Tensor, start: int, *, logits: bool) -> None:
        """``run_windows`` of as many tokens as ``whole_windows`` has just named."""
        ids, start = self._checked(token_ids, start)
        n = int(ids.numel())
        for first in range(0, n, self.PASS_MAX):
            part = ids[first:first + self.PASS_MAX]
            self.first_len.fill_(start + first + 1)
            self._windows_pass(part, start + first)
        self._finish(start + n, logits)

    def _checked(self, token_ids: torch.Tensor, start: int) -> tuple[torch.Tensor, int]:
        state, spec = self.state, self.state.spec
        ids = token_ids.reshape(-1).to(device=state.device, dtype=torch.long)
        n = int(ids.numel())
        if n < 1:
            raise ValueError("prefill chunk must be non-empty")
        start = int(start)
        if start < 0 or start + n > spec.max_seq:
            raise ValueError(f"prefill {start}..{start + n} exceeds max_seq={spec.max_seq}")
        return ids, start

    def _finish(self, seq: int, logits: bool) -> None:
        state, spec = self.state, self.state.spec
        state.position.fill_(seq)
        state.valid_len.fill_(seq)
        if not logits:
            return
        hidden = rms(self.last_hidden.view(1, -1), self.weights.final_norm, spec.rms_eps)
        state.arena.logits.copy_(nf4_linear(self.weights.lm_head, hidden).reshape(1, -1))
        state.pick_next(commit=False)
