"""Host mirror of ``qwen_asr::kernels`` over device memory.

Every function keeps the reference's name, argument order and meaning
(crates/qwen-asr/src/kernels/mod.rs and decoder.rs), with Rust slices replaced
by device-resident ``torch`` tensors (torch supplies device memory and the
current HIP stream; all arithmetic runs in the gfx950 kernels of
``libqasr_hip.so`` through the C-ABI of include/qasr.h).

Error behaviour mirrors the reference: where the Rust code would panic on a
slice that is too short, these raise ``IndexError`` before anything is
launched; a wrong dtype/device raises ``TypeError``; a status returned by the
C-ABI raises ``QasrError``.

Calls only enqueue work on the current stream; nothing here synchronises.
"""
from __future__ import annotations

import ctypes
from dataclasses import dataclass

import torch

from . import _lib
from ._lib import QasrError  # noqa: F401  (re-export)

__all__ = [
    "add_inplace", "rms_norm", "add_rms_norm", "add_rms_norm_quant", "rms_norm_per_head", "apply_rope_neox",
    "head_rms_norm_rope", "swiglu_multiply", "swiglu_multiply_inplace", "swiglu_split", "silu",
    "gelu", "gelu_erf", "layer_norm", "sinusoidal_pe", "pe_add", "tok_embed_f32_to_f32",
    "tok_embed_bf16_to_f32", "tok_embed_int8_to_f32", "embed_gather_f32", "embed_gather_bf16",
    "embed_gather_i8", "quantize_f32_to_int8", "quantize_rows_i8", "linear_nobias_int8",
    "linear_int8", "interleave_gate_up", "gate_up_swiglu_w8a8", "gate_up_swiglu_w8a8_f32in",
    "pack_w8a8_tiles", "gate_up_swiglu_w8a8_packed", "RopeCache", "QuantWeight",
]


def _ptr(t: torch.Tensor | None) -> ctypes.c_void_p:
    return ctypes.c_void_p(0 if t is None else t.data_ptr())


def _stream() -> ctypes.c_void_p:
    return ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)


def _need(t: torch.Tensor, dtype: torch.dtype, n: int, name: str) -> None:
    if not isinstance(t, torch.Tensor):
        raise TypeError(f"{name}: expected a torch tensor, got {type(t).__name__}")
    if t.device.type != "cuda":
        raise TypeError(f"{name}: must be a device tensor (got {t.device})")
    if t.dtype != dtype:
        raise TypeError(f"{name}: expected {dtype}, got {t.dtype}")
    if not t.is_contiguous():
        raise ValueError(f"{name}: must be contiguous")
    if t.numel() < n:
        raise IndexError(f"{name}: range end index {n} out of range for slice of length {t.numel()}")


F32, I8, I32, U16 = torch.float32, torch.int8, torch.int32, torch.int16


class _Calls:
    """The entry points as functions of the binding extension: a tensor argument
    is followed by the element count it must hold (checked as ``_need`` does),
    and the stream is the current one. Bound on first use, all at once."""

    def __getattr__(self, name: str):
        if name.startswith("__"):
            raise AttributeError(name)
        self.__dict__.update(_lib.bind(_need, (F32, I8, I32, U16)))
        if name not in self.__dict__:
            raise AttributeError(name)
        return self.__dict__[name]


_call = _Calls()


# ---------------------------------------------------------------------------
# Basic / normalisation (kernels/mod.rs)
# ---------------------------------------------------------------------------
def add_inplace(a: torch.Tensor, b: torch.Tensor, n: int) -> None:
    """``a[i] += b[i]`` for i < n (kernels/mod.rs:486-488)."""
    _call.qasr_add_inplace_f32(a, n, b, n, n)


def rms_norm(out, x, weight, seq_len: int, hidden: int, eps: float) -> None:
    """Row RMSNorm (kernels/mod.rs:897-918)."""
    _call.qasr_rms_norm_f32(out, seq_len * hidden, x, seq_len * hidden, weight, hidden, seq_len, hidden, eps)


def add_rms_norm(x, delta, weight, out, seq_len: int, hidden: int, eps: float) -> None:
    """Fused ``add_inplace(x, delta)`` + ``rms_norm(out, x)`` (decoder.rs:908+910)."""
    n = seq_len * hidden
    _call.qasr_add_rms_norm_f32(x, n, delta, n, weight, hidden, out, n, seq_len, hidden, eps)


def add_rms_norm_quant(x, delta, weight, out, q, q_scales, seq_len: int, hidden: int,
                       eps: float) -> None:
    """Fused ``x += delta`` (skipped if delta is None), ``y = rms_norm(x)`` and
    per-row int8 quantization of y into ``q``/``q_scales``; ``out`` (may be None)
    receives y."""
    n = seq_len * hidden
    _call.qasr_add_rms_norm_quant_f32(x, n, delta, n, weight, hidden, out, n, q, n, q_scales, seq_len, seq_len, hidden,
                                      eps)


def layer_norm(out, x, weight, bias, seq_len: int, hidden: int, eps: float) -> None:
    """Row LayerNorm (kernels/mod.rs:866-895)."""
    _call.qasr_layer_norm_f32(out, seq_len * hidden, x, seq_len * hidden, weight, hidden, bias, hidden, seq_len, hidden,
                              eps)



def add_layer_norm(x, delta, weight, bias, out, seq_len: int, hidden: int, eps: float) -> None:
    """``x += delta`` then ``out = layer_norm(x)`` in one pass: an encoder
    residual add (encoder.rs:386, 397) and the LayerNorm that reads its rows
    next (encoder.rs:389-390, 370-371, 401-402); equal to ``add_inplace`` +
    ``layer_norm`` bit for bit."""
    n = seq_len * hidden
    _call.qasr_add_layer_norm_f32(x, n, delta, n, weight, hidden, bias, hidden, out, n, seq_len, hidden, eps)


def rms_norm_per_head(x, weight, seq_len: int, n_heads: int, head_dim: int, eps: float) -> None:
    """In-place per-head RMSNorm (kernels/mod.rs:920-935)."""
    _call.qasr_rms_norm_per_head_f32(x, seq_len * n_heads * head_dim, weight, head_dim, seq_len, n_heads, head_dim, eps)


def apply_rope_neox(x, cos_vals, sin_vals, seq: int, n_heads: int, head_dim: int) -> None:
    """In-place NeoX RoPE, row s uses cos/sin row s (kernels/mod.rs:1247-1267)."""
    _call.qasr_apply_rope_neox_f32(x, seq * n_heads * head_dim, cos_vals, seq * head_dim, sin_vals, seq * head_dim, seq,
                                   n_heads, head_dim)


def head_rms_norm_rope(q, k, q_norm_w, k_norm_w, cos_tab, sin_tab, positions, seq: int,
                       n_heads: int, n_kv_heads: int, head_dim: int, eps: float) -> None:
    """Fused q/k head RMSNorm + RoPE at per-row positions (decoder.rs:888-892).

    ``positions`` is an int32 device tensor of ``seq`` entries or None (row s at
    position s). ``cos_tab``/``sin_tab`` are RopeCache tables; a position outside
    the table poisons that row with NaN.
    """
    rows = cos_tab.numel() // head_dim
    _call.qasr_head_rms_norm_rope_f32(q if n_heads else None, seq * n_heads * head_dim,
                                      k if n_kv_heads else None, seq * n_kv_heads * head_dim,
                                      q_norm_w if n_heads else None, head_dim,
                                      k_norm_w if n_kv_heads else None, head_dim, cos_tab, head_dim,
                                      sin_tab, cos_tab.numel(), positions, seq, seq, n_heads, n_kv_heads, head_dim,
                                      rows, eps)


def head_rms_norm_rope_kv(q, k, v, q_norm_w, k_norm_w, rope: "RopeCache", positions, start_pos: int,
                          seq: int, n_heads: int, n_kv_heads: int, head_dim: int, eps: float,
                          k_cache, v_cache, cache_rows: int) -> None:
    """q/k head RMSNorm + RoPE with the KV-cache store fused in
    (decoder.rs:888-895: norm, rope, then ``k_at``/``v_at`` copies).

    Without ``positions`` row s is position ``start_pos + s`` of one sequence
    and ``k_cache``/``v_cache`` are that layer's ``[cache_rows, kv_dim]`` block
    (``KvCache.k_layer_block``). With ``positions`` (int32, ``seq`` entries) row s
    is its own decode stream and the caches are ``[seq, cache_rows, kv_dim]``.
    k and v are read only; q is rotated in place.
    """
    kv_dim = n_kv_heads * head_dim
    if rope.head_dim != head_dim:
        raise ValueError("RopeCache head_dim does not match")
    heads, kv = n_heads != 0, n_kv_heads != 0
    cache = (seq if positions is not None else 1) * cache_rows * kv_dim
    _call.qasr_head_rms_norm_rope_kv_f32(q if heads else None, seq * n_heads * head_dim, k if kv else None,
                                         seq * kv_dim, v if kv else None, seq * kv_dim, q_norm_w if heads else None,
                                         head_dim, k_norm_w if kv else None, head_dim, rope.cos, 0, rope.sin, 0,
                                         positions, seq, start_pos, seq, n_heads, n_kv_heads, head_dim, rope.cap,
                                         eps, k_cache if kv else None, cache, v_cache if kv else None, cache,
                                         cache_rows)


def causal_attention(out, q, k, v, seq_q: int, seq_k: int, n_heads: int, n_kv_heads: int,
                     head_dim: int, scale: float, q_offset: int) -> None:
    """Causal GQA attention over a KV block (kernels/mod.rs:1124-1207)."""
    _call.qasr_causal_attention_f32(out, seq_q * n_heads * head_dim, q, seq_q * n_heads * head_dim,
                                    k if seq_k else None, seq_k * n_kv_heads * head_dim,
                                    v if seq_k else None, seq_k * n_kv_heads * head_dim, seq_q, seq_k, n_heads,
                                    n_kv_heads, head_dim, scale, q_offset)


def batched_decode_workspace(batch: int, n_heads: int, head_dim: int, cache_rows: int,
                             device="cuda") -> torch.Tensor | None:
    """Workspace for batched_decode_attention's chunked form (None if the cache
    is a single chunk): allocate once, reuse per call on one stream."""
    n = _lib.lib().qasr_batched_decode_attention_workspace_floats(batch, n_heads, head_dim, cache_rows)
    return torch.empty(n, dtype=F32, device=device) if n else None


def batched_decode_split_workspace(batch: int, n_heads: int, head_dim: int, cache_rows: int,
                                   device="cuda") -> torch.Tensor | None:
    """As batched_decode_workspace, large enough for a small batch's shorter
    chunks (None if the cache is one chunk all the same)."""
    n = _lib.lib().qasr_batched_decode_attention_split_workspace_floats(batch, n_heads, head_dim, cache_rows)
    return torch.empty(n, dtype=F32, device=device) if n else None


def batched_decode_order(order, positions, batch: int, cache_rows: int) -> None:
    """order (int32 [2 * batch]) = (stream, position) pairs, the streams with the
    most keys first, for batched_decode_attention's ``order``."""
    _call.qasr_batched_decode_order_i32(order, 2 * batch, positions, batch, batch, cache_rows)


def batched_decode_attention(out, q, k_cache, v_cache, cache_rows: int, positions, batch: int, n_heads: int,
                             n_kv_heads: int, head_dim: int, scale: float, workspace=None, out_q=None,
                             out_scales=None, order=None) -> None:
    """Decode attention of ``batch`` streams, each over rows 0..positions[m] of its
    own cache block ``[batch, cache_rows, n_kv_heads * head_dim]`` (decoder.rs:900-903
    per stream). With ``workspace`` (batched_decode_workspace) every stream's
    keys are cut into chunks of 512 (shorter ones for a few streams, with
    batched_decode_split_workspace) and the chunk partials merged; without it
    one workgroup per (stream, kv head) walks all of its keys. ``out_q`` /
    ``out_scales`` (int8 [batch * n_heads * head_dim], f32 [batch]) also get each
    stream's row quantized per row, as quantize_rows_i8 would on ``out``."""
    if (out_q is None) != (out_scales is None):
        raise ValueError("out_q and out_scales go together")
    kv = n_kv_heads * head_dim
    _call.qasr_batched_decode_attention_f32(out, batch * n_heads * head_dim, q, batch * n_heads * head_dim,
                                            k_cache, batch * cache_rows * kv, v_cache, batch * cache_rows * kv,
                                            cache_rows, positions, batch, batch, n_heads, n_kv_heads, head_dim, scale,
                                            workspace, 1, 0 if workspace is None else workspace.numel(),
                                            out_q, batch * n_heads * head_dim, out_scales, batch, order, 2 * batch)


def attention_workspace(seq_q: int, n_heads: int, head_dim: int, device="cuda") -> torch.Tensor:
    """Workspace for causal_attention_split: allocate once, reuse per call on
    one stream."""
    n = _lib.lib().qasr_causal_attention_workspace_floats(seq_q, n_heads, head_dim)
    return torch.empty(n, dtype=F32, device=device)


def causal_attention_split(out, q, k, v, seq_q: int, seq_k: int, n_heads: int, n_kv_heads: int,
                           head_dim: int, scale: float, q_offset: int, workspace) -> None:
    """causal_attention with the keys split over workgroups (decode shape);
    partials go to ``workspace`` (see attention_workspace)."""
    _call.qasr_causal_attention_split_f32(out, seq_q * n_heads * head_dim, q, seq_q * n_heads * head_dim,
                                          k if seq_k else None, seq_k * n_kv_heads * head_dim,
                                          v if seq_k else None, seq_k * n_kv_heads * head_dim, seq_q, seq_k, n_heads,
                                          n_kv_heads, head_dim, scale, q_offset, workspace, 0, workspace.numel())


def decode_attention(out, q, k, v, q_norm_w, k_norm_w, rope: "RopeCache", pos: int, n_heads: int,
                     n_kv_heads: int, head_dim: int, eps: float, scale: float, k_cache, v_cache,
                     cache_rows: int, workspace) -> None:
    """One decode token: q/k head RMSNorm + RoPE at ``pos``, the K/V rows into the
    layer's cache block and causal attention over rows 0..pos, equal bit for bit
    to head_rms_norm_rope_kv + causal_attention_split (decoder.rs:888-903). With
    the keys split over workgroups it is one attention launch; ``q`` is scratch
    (it may come back normalised and rotated)."""
    kv_dim = n_kv_heads * head_dim
    if rope.head_dim != head_dim:
        raise ValueError("RopeCache head_dim does not match")
    _call.qasr_decode_attention_f32(out, n_heads * head_dim, q, n_heads * head_dim, k, kv_dim, v, kv_dim,
                                    q_norm_w, head_dim, k_norm_w, head_dim, rope.cos, 0, rope.sin, 0, rope.cap, pos,
                                    n_heads, n_kv_heads, head_dim, eps, scale, k_cache, cache_rows * kv_dim,
                                    v_cache, cache_rows * kv_dim, cache_rows, workspace, 0, workspace.numel())


def decode_attention_linear_int8(y, out, q, k, v, q_norm_w, k_norm_w, rope: "RopeCache", pos: int, n_heads: int,
                                 n_kv_heads: int, head_dim: int, eps: float, scale: float, k_cache, v_cache,
                                 cache_rows: int, workspace, w: QuantWeight, out_dim: int) -> None:
    """``decode_attention`` and the o projection of its row into ``y``, bit for bit; ``out``
    and ``q`` are scratch."""
    kv_dim, q_dim = n_kv_heads * head_dim, n_heads * head_dim
    if rope.head_dim != head_dim:
        raise ValueError("RopeCache head_dim does not match")
    _call.qasr_decode_attention_linear_int8_f32(y, out_dim, out, q_dim, q, q_dim, k, kv_dim, v, kv_dim, q_norm_w,
                                                head_dim, k_norm_w, head_dim, rope.cos, 0, rope.sin, 0, rope.cap, pos,
                                                n_heads, n_kv_heads, head_dim, eps, scale, k_cache,
                                                cache_rows * kv_dim, v_cache, cache_rows * kv_dim, cache_rows,
                                                workspace, 0, workspace.numel(), w.data, out_dim * q_dim, w.scales,
                                                out_dim, out_dim)


def argmax_rows(idx, x, rows: int, cols: int) -> None:
    """Per-row argmax with the lm_head loop's semantics (decoder.rs:941-949)."""
    _call.qasr_argmax_rows_f32(idx, rows, x, rows * cols, rows, cols)


def lm_head_workspace(vocab: int, device="cuda", rows: int = 1, in_dim: int = 0) -> torch.Tensor:
    """Workspace for the lm_head argmax of up to ``rows`` rows of ``in_dim`` (bytes as a uint8
    tensor). One made for fewer rows is taken too; rows that do not fit it then run on the
    general projection."""
    n = _lib.lib().qasr_lm_head_argmax_rows_workspace_bytes(vocab, rows, in_dim)
    return torch.empty(max(n, 8), dtype=torch.uint8, device=device)


def lm_head_int8_argmax(idx, logits, x, w: QuantWeight, rows: int, in_dim: int, vocab: int,
                        workspace: torch.Tensor | None = None) -> None:
    """INT8 lm_head logits + greedy argmax (decoder.rs:935-963). With a
    ``lm_head_workspace`` and one row the argmax is reduced inside the matvec; several
    rows that fit it as digit rows run on the int8 matrix cores."""
    ws_bytes = 0 if workspace is None else workspace.numel() * workspace.element_size()
    _call.qasr_lm_head_int8_argmax_f32(idx, rows, logits, rows * vocab, x, rows * in_dim, w.data, vocab * in_dim,
                                       w.scales, vocab, rows, in_dim, vocab, workspace, ws_bytes)


class KvCache:
    """Device KV cache with the reference's layout and growth rule
    (decoder.rs:129-228): ``k``/``v`` are ``[n_layers, max_seq, kv_dim]`` fp32,
    ``grow`` doubles ``max_seq`` until it covers the request and copies the first
    ``len`` rows of every layer."""

    def __init__(self, n_layers: int, max_seq: int, kv_dim: int, device="cuda"):
        self.n_layers, self.max_seq, self.kv_dim, self.len = n_layers, max_seq, kv_dim, 0
        self.k = torch.zeros(n_layers * max_seq * kv_dim, dtype=F32, device=device)
        self.v = torch.zeros_like(self.k)

    def grow(self, required: int) -> None:
        if required <= self.max_seq:
            return
        new_max = self.max_seq
        while new_max < required:
            new_max *= 2
        k = torch.zeros(self.n_layers * new_max * self.kv_dim, dtype=F32, device=self.k.device)
        v = torch.zeros_like(k)
        n = self.len * self.kv_dim
        for layer in range(self.n_layers):
            src, dst = layer * self.max_seq * self.kv_dim, layer * new_max * self.kv_dim
            k[dst:dst + n].copy_(self.k[src:src + n])
            v[dst:dst + n].copy_(self.v[src:src + n])
        self.k, self.v, self.max_seq = k, v, new_max

    def k_layer_block(self, layer: int) -> torch.Tensor:
        off = layer * self.max_seq * self.kv_dim
        return self.k[off:off + self.max_seq * self.kv_dim]

    def v_layer_block(self, layer: int) -> torch.Tensor:
        off = layer * self.max_seq * self.kv_dim
        return self.v[off:off + self.max_seq * self.kv_dim]

    def layer_blocks(self) -> tuple:
        """Every layer's k block and v block: one torch call for all layers."""
        n = max(self.max_seq * self.kv_dim, 1)
        return self.k.split(n), self.v.split(n)

    def k_layer(self, layer: int) -> torch.Tensor:
        return self.k_layer_block(layer)[: self.len * self.kv_dim]

    def v_layer(self, layer: int) -> torch.Tensor:
        return self.v_layer_block(layer)[: self.len * self.kv_dim]


class RopeCache:
    """Device RoPE table with the reference's growth rule (decoder.rs:234-306).

    ``ensure(required_pos, head_dim, theta)`` grows capacity by doubling from
    1024; new rows are filled on the GPU from the f32 inverse frequencies
    ``1/theta^(2d/head_dim)`` (computed on the host by the library, as the
    reference does). A change of head_dim rebuilds the table from row 0.
    """

    def __init__(self, device: str | torch.device = "cuda"):
        self.device = torch.device(device)
        self.cos = torch.empty(0, dtype=F32, device=self.device)
        self.sin = torch.empty(0, dtype=F32, device=self.device)
        self.cap = 0
        self.head_dim = 0
        self.theta = None

    def ensure(self, required_pos: int, head_dim: int, theta: float) -> None:
        if self.head_dim != head_dim or self.theta != theta:
            self.cap = 0
            self.head_dim = head_dim
            self.theta = theta
            self.cos = torch.empty(0, dtype=F32, device=self.device)
            self.sin = torch.empty(0, dtype=F32, device=self.device)
        if required_pos <= self.cap:
            return
        new_cap = self.cap if self.cap > 0 else 1024
        while new_cap < required_pos:
            new_cap *= 2
        cos = torch.empty(new_cap * head_dim, dtype=F32, device=self.device)
        sin = torch.empty(new_cap * head_dim, dtype=F32, device=self.device)
        if self.cap:
            cos[: self.cap * head_dim].copy_(self.cos)
            sin[: self.cap * head_dim].copy_(self.sin)
        _lib.call("qasr_rope_table_fill_f32", _ptr(cos), _ptr(sin), self.cap, new_cap, head_dim,
                  theta, _stream())
        self.cos, self.sin, self.cap = cos, sin, new_cap

    def cos_at(self, pos: int) -> torch.Tensor:
        return self.cos[pos * self.head_dim:(pos + 1) * self.head_dim]

    def sin_at(self, pos: int) -> torch.Tensor:
        return self.sin[pos * self.head_dim:(pos + 1) * self.head_dim]

    def cos_range(self, start: int, length: int) -> torch.Tensor:
        return self.cos[start * self.head_dim:(start + length) * self.head_dim]

    def sin_range(self, start: int, length: int) -> torch.Tensor:
        return self.sin[start * self.head_dim:(start + length) * self.head_dim]


# ---------------------------------------------------------------------------
# Activations
# ---------------------------------------------------------------------------
def swiglu_multiply(out, gate_up, seq_len: int, intermediate: int) -> None:
    """SwiGLU on the row-interleaved gate/up buffer (kernels/mod.rs:965-985)."""
    _call.qasr_swiglu_multiply_f32(out, seq_len * intermediate, gate_up, seq_len * 2 * intermediate, seq_len,
                                   intermediate)


def swiglu_multiply_inplace(gate, up) -> None:
    """``gate = silu(gate) * up`` (kernels/mod.rs:988-994)."""
    n = gate.numel()
    _call.qasr_swiglu_split_f32(gate, n, gate, n, up, n, n)


def swiglu_split(out, gate, up, n: int) -> None:
    """``out = silu(gate) * up`` on split buffers (decode SwiGLU, decoder.rs:916-921)."""
    _call.qasr_swiglu_split_f32(out, n, gate, n, up, n, n)


def silu(x, n: int) -> None:
    """In-place SiLU (kernels/mod.rs:941-946)."""
    _call.qasr_silu_f32(x, n, n)


def gelu(x, n: int) -> None:
    """In-place tanh-approximation GELU, reference arithmetic (kernels/mod.rs:948-963)."""
    _call.qasr_gelu_tanh_f32(x, n, n)


def gelu_erf(x, n: int) -> None:
    """In-place exact GELU 0.5*x*(1+erf(x/sqrt(2)))."""
    _call.qasr_gelu_erf_f32(x, n, n)


# ---------------------------------------------------------------------------
# Position embeddings (encoder)
# ---------------------------------------------------------------------------
def sinusoidal_pe(pe, n_pos: int, d_model: int) -> None:
    """Sinusoidal PE table [n_pos, d_model] (kernels/mod.rs:1213-1226)."""
    _need(pe, F32, n_pos * d_model, "pe")
    _lib.call("qasr_sinusoidal_pe_f32", _ptr(pe), n_pos, d_model, _stream())


def pe_add(x, pe, rows: int, d_model: int, n_pos: int) -> None:
    """``x[r] += pe[r % n_pos]`` (encoder.rs:340-343 with the table reused)."""
    _call.qasr_pe_add_f32(x, rows * d_model, pe, n_pos * d_model, rows, d_model, n_pos)


def pe_add_layer_norm(x, pe, out, weight, bias, rows: int, d_model: int, n_pos: int,
                      eps: float) -> None:
    """``x[r] += pe[r % n_pos]`` then ``out = layer_norm(x)`` in one pass: the
    encoder's PE add (encoder.rs:341-343) and layer 0's LayerNorm of the same
    rows (encoder.rs:370-371); equal to ``pe_add`` + ``layer_norm`` bit for bit."""
    _call.qasr_pe_add_layer_norm_f32(x, rows * d_model, pe, n_pos * d_model, out, rows * d_model, weight, d_model,
                                     bias, d_model, rows, d_model, n_pos, eps)


# ---------------------------------------------------------------------------
# Token embeddings (decoder.rs:631-646)
# ---------------------------------------------------------------------------
@dataclass
class QuantWeight:
    """Device view of a .qint8 weight (quantize.rs:77-84): int8 [out_dim, in_dim] + f32 scales."""

    data: torch.Tensor
    scales: torch.Tensor
    out_dim: int
    in_dim: int


def embed_gather_f32(out, table, ids, n: int, dim: int) -> None:
    _call.qasr_embed_gather_f32(out, n * dim, table, dim, ids, n, n, dim, table.numel() // dim)


def embed_gather_bf16(out, table, ids, n: int, dim: int) -> None:
    """Batched tok_embed_bf16_to_f32; ``table`` holds bf16 bits as int16 or bfloat16."""
    if table.dtype == torch.bfloat16:
        table = table.view(U16)
    _call.qasr_embed_gather_bf16(out, n * dim, table, dim, ids, n, n, dim, table.numel() // dim)


def embed_gather_i8(out, w: QuantWeight, ids, n: int, dim: int) -> None:
    """Batched tok_embed_int8_to_f32."""
    _call.qasr_embed_gather_i8(out, n * dim, w.data, w.out_dim * dim, w.scales, w.out_dim, ids, n, n, dim, w.out_dim)


def _one_id(token_id: int, device) -> torch.Tensor:
    return torch.tensor([token_id], dtype=I32, device=device)


def tok_embed_f32_to_f32(dst, table, token_id: int, dim: int) -> None:
    embed_gather_f32(dst, table, _one_id(token_id, dst.device), 1, dim)


def tok_embed_bf16_to_f32(dst, tok_emb_bf16, token_id: int, dim: int) -> None:
    """One token (decoder.rs:631-636)."""
    embed_gather_bf16(dst, tok_emb_bf16, _one_id(token_id, dst.device), 1, dim)


def tok_embed_int8_to_f32(dst, w: QuantWeight, token_id: int, dim: int) -> None:
    """One token (decoder.rs:639-646)."""
    embed_gather_i8(dst, w, _one_id(token_id, dst.device), 1, dim)


# ---------------------------------------------------------------------------
# INT8
# ---------------------------------------------------------------------------
def quantize_rows_i8(q, scales, x, rows: int, cols: int) -> None:
    """Per-row int8 quantization into caller buffers (quantize.rs:633-662)."""
    _call.qasr_quantize_rows_i8(q, rows * cols, scales, rows, x, rows * cols, rows, cols)


def quantize_f32_to_int8(f32_data, out_dim: int, in_dim: int):
    """Returns ``(int8 data, f32 scales)`` like quantize.rs:633-662 (device tensors)."""
    q = torch.empty(out_dim * in_dim, dtype=I8, device=f32_data.device)
    s = torch.empty(out_dim, dtype=F32, device=f32_data.device)
    quantize_rows_i8(q, s, f32_data, out_dim, in_dim)
    return q, s


def linear_nobias_int8(y, x, w_int8, scales, seq_len: int, in_dim: int, out_dim: int) -> None:
    """W8A32 ``y = scale * (W_int8 @ x)`` (kernels/mod.rs:650-661)."""
    _call.qasr_linear_nobias_int8_f32(y, seq_len * out_dim, x, seq_len * in_dim, w_int8, out_dim * in_dim,
                                      scales, out_dim, seq_len, in_dim, out_dim)


def linear_nobias_int8_multi(ys, ws: list, x, seq_len: int, in_dim: int) -> None:
    """Several W8A32 projections of the same x in one launch (q/k/v, decoder.rs:881-886);
    ``ws`` are QuantWeights, ``ys[m]`` gets ``seq_len * ws[m].out_dim`` floats."""
    _call.qasr_linear_nobias_int8_multi_f32(ys, ws, x, seq_len * in_dim, seq_len, in_dim)


def digit_rows(digits, exps, x, rows: int, cols: int, wide: bool = False) -> None:
    """Rows of x as four int8 digit planes (``digits`` [4 * rows * cols]) and a power of
    two per row (``exps``, int32), for the ``*_digits`` projections. The digits hold x to
    2^-30 of the row's largest element; with ``wide`` a row whose elements range too far
    for that is marked, and a projection given ``x`` multiplies it in fp32 instead."""
    fn = _call.qasr_digit_rows_wide_f32 if wide else _call.qasr_digit_rows_f32
    fn(digits, 4 * rows * cols, exps, rows, x, rows * cols, rows, cols)


def add_rms_norm_digits(x, delta, weight, x_norm, digits, exps, rows: int, cols: int, eps: float,
                        delta_parts: int = 1, wide: bool = False, all_rows: bool = True) -> None:
    """x += delta (None: not; ``delta_parts`` slices to be added), then the digit rows of
    its RMSNorm; ``x_norm`` (or None) receives the normalised rows too. ``wide`` as in
    ``digit_rows``; then ``x_norm`` is needed, and without ``all_rows`` receives the marked
    rows only."""
    n = rows * cols
    if wide:
        _call.qasr_add_rms_norm_digits_wide_f32(x, n, delta, delta_parts * n, delta_parts, weight, cols, x_norm, n,
                                                int(all_rows), digits, 4 * n, exps, rows, rows, cols, eps)
    else:
        _call.qasr_add_rms_norm_digits_f32(x, n, delta, delta_parts * n, delta_parts, weight, cols, x_norm, n, digits,
                                           4 * n, exps, rows, rows, cols, eps)


def linear_digits_parts(seq_len: int, in_dim: int, out_dim: int) -> int:
    """The ``parts`` worth taking for a projection of this size."""
    return _lib.lib().qasr_linear_digits_parts(seq_len, in_dim, out_dim)


def linear_digits_int8(ys, ws: list, digits, exps, seq_len: int, in_dim: int, residual: bool = False,
                       parts: int = 1, x=None) -> None:
    """W8A32 projections of the same digit rows in one launch (up to 3 QuantWeights);
    with ``residual`` each is added to its y. ``parts`` > 1 cuts in_dim: each y holds that
    many slices ``[parts, seq_len, out_dim]`` to be added (``add_rms_norm_digits``). ``x``:
    the rows' floats, for those marked wide (without it they give NaN)."""
    _call.qasr_linear_digits_wide_int8_f32(ys, ws, digits, 4 * seq_len * in_dim, exps, seq_len, x, seq_len * in_dim,
                                           seq_len, in_dim, int(residual), parts, parts * seq_len)


def gate_up_swiglu_digits_int8(out, w: QuantWeight, digits, exps, seq_len: int, in_dim: int, intermediate: int,
                               prefill: bool = False, x=None) -> None:
    """The interleaved gate/up projection of digit rows with the decode loop's SwiGLU, or
    swiglu_multiply's (``prefill``); ``x`` as in ``linear_digits_int8``."""
    _call.qasr_gate_up_swiglu_digits_wide_int8_f32(out, seq_len * intermediate, w.data, 2 * intermediate * in_dim,
                                                   w.scales, 2 * intermediate, digits, 4 * seq_len * in_dim, exps,
                                                   seq_len, x, seq_len * in_dim, seq_len, in_dim, intermediate,
                                                   int(prefill))


def qkv_heads_digits_int8(q, k_cache, v_cache, cache_rows: int, wq: QuantWeight, wk: QuantWeight, wv: QuantWeight,
                          digits, exps, seq_len: int, in_dim: int, n_heads: int, n_kv_heads: int, head_dim: int,
                          q_norm_w, k_norm_w, rope: "RopeCache", start_pos: int, eps: float, x=None) -> None:
    """``qkv_heads_int8`` from digit rows; ``x`` as in ``linear_digits_int8``."""
    qd, kv = n_heads * head_dim, n_kv_heads * head_dim
    if rope.head_dim != head_dim:
        raise ValueError("RopeCache head_dim does not match")
    _call.qasr_qkv_heads_digits_wide_int8_f32(q, seq_len * qd, k_cache, cache_rows * kv, v_cache, cache_rows * kv,
                                              cache_rows, wq.data, qd * in_dim, wq.scales, qd, wk.data, kv * in_dim,
                                              wk.scales, kv, wv.data, kv * in_dim, wv.scales, kv, digits,
                                              4 * seq_len * in_dim, exps, seq_len, x, seq_len * in_dim, seq_len,
                                              in_dim, n_heads, n_kv_heads, head_dim, q_norm_w, head_dim, k_norm_w,
                                              head_dim, rope.cos, 0, rope.sin, 0, rope.cap, start_pos, eps)


def qkv_heads_int8(q, k_cache, v_cache, cache_rows: int, wq: QuantWeight, wk: QuantWeight, wv: QuantWeight,
                   x, seq_len: int, in_dim: int, n_heads: int, n_kv_heads: int, head_dim: int, q_norm_w,
                   k_norm_w, rope: "RopeCache", start_pos: int, eps: float) -> None:
    """A prefill chunk's q/k/v projections + q/k head norms + RoPE + the K/V
    cache rows in one launch (decoder.rs:795-810). Same results, bit for bit, as
    ``linear_nobias_int8_multi`` followed by ``head_rms_norm_rope_kv`` (positions
    None); ``k_cache``/``v_cache`` are the layer's ``[cache_rows, kv_dim]`` blocks.
    head_dim 128, seq_len >= 8 and in_dim % 64 == 0 (else the library raises)."""
    qd, kv = n_heads * head_dim, n_kv_heads * head_dim
    if rope.head_dim != head_dim:
        raise ValueError("RopeCache head_dim does not match")
    _call.qasr_qkv_heads_int8_f32(q, seq_len * qd, k_cache, cache_rows * kv, v_cache, cache_rows * kv, cache_rows,
                                  wq.data, qd * in_dim, wq.scales, qd, wk.data, kv * in_dim, wk.scales, kv,
                                  wv.data, kv * in_dim, wv.scales, kv, x, seq_len * in_dim, seq_len, in_dim, n_heads,
                                  n_kv_heads, head_dim, q_norm_w, head_dim, k_norm_w, head_dim, rope.cos, 0,
                                  rope.sin, 0, rope.cap, start_pos, eps)


def norm_slices(hidden: int) -> int:
    """Partial sums of squares per token that ``linear_int8_residual`` writes
    (one per 64 columns of the residual stream)."""
    return (hidden + 63) // 64


def linear_int8_residual(h, ss, x, w: QuantWeight, seq_len: int, in_dim: int, out_dim: int, hg=None,
                         gain=None) -> None:
    """The prefill residual add folded into the o / down projection
    (decoder.rs:821-822, 837-838): ``h += linear_nobias_int8(x, w)`` bit for bit;
    ``ss[t, s]`` = the sum of squares of the updated ``h[t, 64s:64s+64]``, and
    with ``hg``/``gain`` also ``hg = h * gain`` -- what the next folded RMSNorm
    reads. seq_len >= 8 and in_dim % 64 == 0 (else the library raises)."""
    if (hg is None) != (gain is None):
        raise ValueError("linear_int8_residual: hg and gain go together")
    _call.qasr_linear_int8_residual_f32(h, seq_len * out_dim, ss, seq_len * norm_slices(out_dim), hg, seq_len * out_dim,
                                        gain, out_dim, x, seq_len * in_dim, w.data, out_dim * in_dim, w.scales, out_dim,
                                        seq_len, in_dim, out_dim)


def rms_norm_gate_up_swiglu_multiply_int8(out, hg, ss, eps: float, x_norm, w: QuantWeight, seq_len: int,
                                          in_dim: int, intermediate: int) -> None:
    """The prefill post-attention RMSNorm folded into the gate/up GEMM + SwiGLU
    (decoder.rs:826-833): ``hg`` = h * norm gain and ``ss`` from
    ``linear_int8_residual``; each token's outputs are multiplied by its 1 / rms.
    ``x_norm`` ([seq_len, in_dim], may be ``hg``) receives the normalised rows
    only on shapes the folded kernel does not take."""
    _call.qasr_rms_norm_gate_up_swiglu_multiply_int8_f32(out, seq_len * intermediate, hg, seq_len * in_dim,
                                                         ss, seq_len * norm_slices(in_dim), norm_slices(in_dim), eps,
                                                         x_norm, seq_len * in_dim, w.data, 2 * intermediate * in_dim,
                                                         w.scales, 2 * intermediate, seq_len, in_dim, intermediate)


def rms_norm_qkv_heads_int8(q, k_cache, v_cache, cache_rows: int, wq: QuantWeight, wk: QuantWeight,
                            wv: QuantWeight, hg, ss, norm_eps: float, x_norm, seq_len: int, in_dim: int,
                            n_heads: int, n_kv_heads: int, head_dim: int, q_norm_w, k_norm_w, rope: "RopeCache",
                            start_pos: int, eps: float) -> None:
    """``qkv_heads_int8`` on the layer-input RMSNorm folded in: ``hg`` = h *
    input_norm and ``ss`` from ``linear_int8_residual`` (decoder.rs:789-810);
    ``x_norm`` as in ``rms_norm_gate_up_swiglu_multiply_int8``."""
    qd, kv = n_heads * head_dim, n_kv_heads * head_dim
    if rope.head_dim != head_dim:
        raise ValueError("RopeCache head_dim does not match")
    _call.qasr_rms_norm_qkv_heads_int8_f32(q, seq_len * qd, k_cache, cache_rows * kv, v_cache, cache_rows * kv,
                                           cache_rows, wq.data, qd * in_dim, wq.scales, qd, wk.data, kv * in_dim,
                                           wk.scales, kv, wv.data, kv * in_dim, wv.scales, kv, hg, seq_len * in_dim,
                                           ss, seq_len * norm_slices(in_dim), norm_slices(in_dim), norm_eps,
                                           x_norm, seq_len * in_dim, seq_len, in_dim, n_heads, n_kv_heads, head_dim,
                                           q_norm_w, head_dim, k_norm_w, head_dim, rope.cos, 0, rope.sin, 0, rope.cap,
                                           start_pos, eps)


def gate_up_swiglu_int8(out, x, w: QuantWeight, seq_len: int, in_dim: int, intermediate: int) -> None:
    """W8A32 gate/up projection on the interleaved weight + the decode loop's
    SwiGLU (decoder.rs:912-921), one launch; gate/up values are not stored."""
    _call.qasr_gate_up_swiglu_int8_f32(out, seq_len * intermediate, x, seq_len * in_dim,
                                       w.data, 2 * intermediate * in_dim, w.scales, 2 * intermediate, seq_len, in_dim,
                                       intermediate)


def add_rms_norm_linear_nobias_int8_multi(ys, ws: list, h_out, x, delta, norm_w, in_dim: int,
                                          eps: float) -> None:
    """One decode token: h = x + delta (``delta`` None: h = x), the RMSNorm of h,
    and the projections of the normalised row in one launch (decoder.rs:924->878
    then 881-886). ``h_out`` (None: not written) gets h and must be a different
    buffer from x and delta; ``ys[m]`` equals add_rms_norm + linear_nobias_int8_multi
    bit for bit."""
    _call.qasr_add_rms_norm_linear_nobias_int8_multi_f32(ys, ws, h_out, in_dim, x, in_dim, delta, in_dim, norm_w,
                                                         in_dim, in_dim, eps)


def add_rms_norm_gate_up_swiglu_int8(out, h_out, x, delta, norm_w, w: QuantWeight, in_dim: int,
                                     intermediate: int, eps: float) -> None:
    """One decode token: the post-attention add + RMSNorm, the gate/up projection
    and the decode SwiGLU in one launch (decoder.rs:908-921); equals add_rms_norm
    followed by gate_up_swiglu_int8 bit for bit."""
    _call.qasr_add_rms_norm_gate_up_swiglu_int8_f32(out, intermediate, h_out, in_dim, x, in_dim, delta, in_dim,
                                                    norm_w, in_dim, w.data, 2 * intermediate * in_dim,
                                                    w.scales, 2 * intermediate, in_dim, intermediate, eps)


def gate_up_swiglu_multiply_int8(out, x, w: QuantWeight, seq_len: int, in_dim: int, intermediate: int) -> None:
    """The prefill's W8A32 gate/up projection on the interleaved weight + swiglu_multiply
    (decoder.rs:831-834; the fast_exp SwiGLU), one launch; gate/up values are not stored."""
    _call.qasr_gate_up_swiglu_multiply_int8_f32(out, seq_len * intermediate, x, seq_len * in_dim,
                                                w.data, 2 * intermediate * in_dim, w.scales, 2 * intermediate, seq_len,
                                                in_dim, intermediate)


def linear_int8(y, x, w_int8, scales, bias, seq_len: int, in_dim: int, out_dim: int) -> None:
    """W8A32 linear with optional bias (kernels/mod.rs:664-673)."""
    _call.qasr_linear_int8_f32(y, seq_len * out_dim, x, seq_len * in_dim, w_int8, out_dim * in_dim, scales, out_dim,
                               bias, out_dim, seq_len, in_dim, out_dim)


def interleave_gate_up(gate: QuantWeight, up: QuantWeight) -> QuantWeight:
    """Fused row-interleaved gate/up weight (decoder.rs:701-719), built on the device."""
    inter, hidden = gate.out_dim, gate.in_dim
    if (up.out_dim, up.in_dim) != (inter, hidden):
        raise ValueError("gate and up must have the same shape")
    _need(gate.data, I8, inter * hidden, "gate.data")
    _need(up.data, I8, inter * hidden, "up.data")
    _need(gate.scales, F32, inter, "gate.scales")
    _need(up.scales, F32, inter, "up.scales")
    data = torch.empty(2 * inter * hidden, dtype=I8, device=gate.data.device)
    scales = torch.empty(2 * inter, dtype=F32, device=gate.data.device)
    _lib.call("qasr_interleave_gate_up_i8", _ptr(data), _ptr(scales), _ptr(gate.data),
              _ptr(gate.scales), _ptr(up.data), _ptr(up.scales), inter, hidden, _stream())
    return QuantWeight(data, scales, 2 * inter, hidden)


def gate_up_swiglu_w8a8(out, w: QuantWeight, xq, x_scales, batch: int, in_dim: int,
                        intermediate: int) -> None:
    """W8A8 gate/up projection + SwiGLU on the interleaved weight (int32-exact dots)."""
    _call.qasr_gate_up_swiglu_w8a8(out, batch * intermediate, w.data, 2 * intermediate * in_dim,
                                   w.scales, 2 * intermediate, xq, batch * in_dim, x_scales, batch, batch, in_dim,
                                   intermediate)


def gate_up_swiglu_w8a8_f32in(out, w: QuantWeight, x, in_dim: int, intermediate: int) -> None:
    """Batch-1 W8A8 gate/up + SwiGLU quantizing the fp32 input vector in-kernel."""
    _call.qasr_gate_up_swiglu_w8a8_f32in(out, intermediate, w.data, 2 * intermediate * in_dim,
                                         w.scales, 2 * intermediate, x, in_dim, in_dim, intermediate)


def pack_w8a8_tiles(w: QuantWeight) -> QuantWeight:
    """MFMA tile layout of an int8 weight (see include/qasr.h); scales are shared."""
    _need(w.data, I8, w.out_dim * w.in_dim, "w.data")
    packed = torch.empty(w.out_dim * w.in_dim, dtype=I8, device=w.data.device)
    _lib.call("qasr_pack_w8a8_tiles", _ptr(packed), _ptr(w.data), w.out_dim, w.in_dim, _stream())
    return QuantWeight(packed, w.scales, w.out_dim, w.in_dim)


def linear_w8a8_packed(y, w_packed: QuantWeight, xq, x_scales, batch: int, in_dim: int, out_dim: int) -> None:
    """Batched W8A8 projection: y[m, n] = ((f32)dot * x_scales[m]) * scales[n]."""
    _call.qasr_linear_w8a8_packed(y, batch * out_dim, w_packed.data, out_dim * in_dim, w_packed.scales, out_dim,
                                  xq, batch * in_dim, x_scales, batch, batch, in_dim, out_dim)


def qkv_heads_w8a8_packed(q_out, k_cache, v_cache, cache_rows: int, w_packed: QuantWeight, xq, x_scales,
                          q_norm_w, k_norm_w, rope: "RopeCache", positions, batch: int, in_dim: int,
                          n_heads: int, n_kv_heads: int, head_dim: int, eps: float) -> None:
    """q/k/v projections of ``batch`` streams + q/k head norms + RoPE at each
    stream's position + the K/V cache rows, one launch (decoder.rs:881-895 per
    stream). ``k_cache``/``v_cache``: [batch, cache_rows, n_kv_heads * head_dim]."""
    n = (n_heads + 2 * n_kv_heads) * head_dim
    kv = n_kv_heads * head_dim
    _call.qasr_qkv_heads_w8a8_packed(q_out, batch * n_heads * head_dim, k_cache, batch * cache_rows * kv,
                                     v_cache, batch * cache_rows * kv, cache_rows, w_packed.data, n * in_dim,
                                     w_packed.scales, n, xq, batch * in_dim, x_scales, batch, q_norm_w, head_dim,
                                     k_norm_w, head_dim, rope.cos, 0, rope.sin, 0, rope.cap, positions, batch, batch,
                                     in_dim, n_heads, n_kv_heads, head_dim, eps)


def gate_up_swiglu_w8a8_packed(out, w_packed: QuantWeight, xq, x_scales, batch: int, in_dim: int,
                               intermediate: int) -> None:
    """gate_up_swiglu_w8a8 on a pack_w8a8_tiles weight (same results)."""
    _call.qasr_gate_up_swiglu_w8a8_packed(out, batch * intermediate, w_packed.data, 2 * intermediate * in_dim,
                                          w_packed.scales, 2 * intermediate, xq, batch * in_dim, x_scales, batch, batch,
                                          in_dim, intermediate)
