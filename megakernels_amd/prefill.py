"""The prompt forward on the GPU: the dense forward of ``llama.py`` over whole prompts with one HIP kernel between two
matrix products (``csrc/mk_prefill.hip``) in place of a chain of small PyTorch operations.

PyTorch owns the memory and the stream and computes the plain matrix products; everything else - embedding, RMS norm,
residual adds, rotary embedding, cache append, causal attention, SiLU, argmax - is this library's.  There is no
fallback for a missing library: a GPU forward that it covers raises ``RuntimeError``.
"""

from __future__ import annotations

import ctypes
from pathlib import Path

import torch
import torch.nn.functional as F
from torch import Tensor

LIBRARY = Path(__file__).resolve().parent / "csrc" / "libmk_prefill.so"

_I, _P = ctypes.c_int32, ctypes.c_void_p


class Shape(ctypes.Structure):
    """``mk_prefill_shape`` of ``include/mk_prefill.h``."""

    _fields_ = [(n, _I) for n in (
        "batch", "seq", "num_attention_heads", "num_kv_heads", "head_dim", "hidden_size", "intermediate_size", "vocab_size",
        "kv_max_len", "rope_positions", "interleaved")] + [("rms_norm_eps", ctypes.c_float)]


_POINTERS = {"embed": 6, "add_norm": 4, "rope": 9, "attention": 4, "silu_mul": 3, "argmax": 2}
_lib = None


def load_library():
    global _lib
    if _lib is None:
        if not LIBRARY.exists():
            raise RuntimeError(f"{LIBRARY} is missing: build it with `python {LIBRARY.with_name('build.py')}` (needs hipcc)")
        lib = ctypes.CDLL(str(LIBRARY))
        for name, count in _POINTERS.items():
            function = getattr(lib, f"mk_prefill_{name}")
            function.argtypes = [ctypes.POINTER(Shape)] + [_P] * (count + 1)  # ... and the stream
            function.restype = ctypes.c_int
        lib.mk_prefill_last_error.restype = ctypes.c_char_p
        _lib = lib
    return _lib


def covers(model, ids: Tensor) -> bool:
    """Whether the HIP forward takes this call: more than one position per sequence, bf16 weights on the GPU, and an
    architecture its kernels are built for (head_dim 64 or 128, four query heads per KV head, widths in 16-byte pieces).
    Everything else runs through the plain PyTorch forward."""
    c = model.config
    return (ids.is_cuda and ids.shape[-1] > 1 and ids.device == model.device and model.dtype == torch.bfloat16
            and c.head_dim in (64, 128) and c.num_attention_heads == 4 * c.num_key_value_heads
            and c.hidden_size % 8 == 0 and c.hidden_size <= 8192 and c.intermediate_size % 8 == 0 and c.vocab_size % 8 == 0
            and model.model.rope_cos.dtype == torch.float32)


def forward(model, ids: Tensor, positions: Tensor) -> tuple[Tensor, Tensor]:
    """``(hidden states [B, S, hidden], greedy ids [B, S])`` of the prompt ``ids [B, S]`` at ``positions [S]``; the keys
    and values go to the model's cache."""
    lib = load_library()
    c, p = model.config, model.stacked_params
    B, S = ids.shape
    H, KVH, D = c.num_attention_heads, c.num_key_value_heads, c.head_dim
    device = ids.device
    k_cache, v_cache = model.stacked_kv_cache
    if B > k_cache.shape[1] or positions.shape != (S,):
        raise RuntimeError(f"{B} sequences of {S} tokens at positions {tuple(positions.shape)} do not fit the cache {tuple(k_cache.shape)}")
    ids = ids.to(torch.int64).contiguous()
    positions = positions.to(device=device, dtype=torch.int64).contiguous()
    shape = Shape(B, S, H, KVH, D, c.hidden_size, c.intermediate_size, c.vocab_size, k_cache.shape[2],
                  model.model.rope_cos.shape[0], int(bool(model.extra_config.interleave_rope)), c.rms_norm_eps)
    padded = lib.mk_prefill_padded_seq(S)

    def rows(width):
        return torch.empty(B, S, width, dtype=torch.bfloat16, device=device)

    h, x, q, attn, prod = rows(c.hidden_size), rows(c.hidden_size), rows(H * D), rows(H * D), rows(c.intermediate_size)
    keys = torch.empty(2, B * KVH * D * padded, dtype=torch.bfloat16, device=device)
    out_ids = torch.empty(B, S, dtype=torch.int64, device=device)

    with torch.cuda.device(device):
        stream = torch.cuda.current_stream(device).cuda_stream

        def call(name, *tensors):
            if getattr(lib, f"mk_prefill_{name}")(ctypes.byref(shape), *[t.data_ptr() for t in tensors], stream) != 0:
                raise RuntimeError(f"mk_prefill_{name}: {lib.mk_prefill_last_error().decode()}")

        call("embed", ids, positions, model.model.embed_tokens.weight, p.attn_ln_weight, h, x)
        for layer in range(c.num_hidden_layers):
            qkv = F.linear(x, p.qkv_proj[layer])
            call("rope", qkv, positions, model.model.rope_cos, model.model.rope_sin, k_cache[layer], v_cache[layer], q, keys[0], keys[1])
            call("attention", q, keys[0], keys[1], attn)
            call("add_norm", F.linear(attn, p.o_proj[layer]), p.mlp_ln_weight[layer], h, x)
            call("silu_mul", F.linear(x, p.gate_proj[layer]), F.linear(x, p.up_proj[layer]), prod)
            last = layer + 1 == c.num_hidden_layers
            norm = model.lm_head.input_norm.weight if last else p.attn_ln_weight[layer + 1]
            call("add_norm", F.linear(prod, p.down_proj[layer]), norm, h, x)
        call("argmax", F.linear(x, model.lm_head.lm_head.weight), out_ids)
    return h, out_ids
