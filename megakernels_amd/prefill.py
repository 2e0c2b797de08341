"""The prompt forward on the GPU: the dense forward of ``llama.py`` over whole prompts (``csrc/mk_prefill.hip``).

PyTorch owns the memory and the stream.  A prompt of up to some thousand positions (of a model wider than 2048: of some
hundred to one or two thousand) runs as one call, its matrix products included.  For the others PyTorch computes the plain products,
and everything between them - embedding, RMS norm, residual adds, rotary embedding, cache append, causal attention, SiLU,
argmax - is this library's.  There is no fallback for a missing library: a GPU forward that it covers raises ``RuntimeError``.
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


class Model(ctypes.Structure):
    """``mk_prefill_model`` of ``include/mk_prefill.h``."""

    _fields_ = [(n, _P) for n in (
        "embed", "attn_norm", "qkv", "o", "mlp_norm", "gate", "up", "down", "final_norm", "head", "rope_cos", "rope_sin",
        "k_cache", "v_cache")] + [("num_layers", _I), ("cache_batch", _I)]


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
        for kind, plan in (("", "tile"), ("wide_", "wide")):
            workspace_bytes, forward, tiling = (getattr(lib, f"mk_prefill_{n}") for n in (f"{kind}workspace_bytes", f"{kind}forward", f"{plan}_plan"))
            workspace_bytes.argtypes, workspace_bytes.restype = [ctypes.POINTER(Shape)], ctypes.c_int64
            forward.argtypes, forward.restype = [ctypes.POINTER(Shape), ctypes.POINTER(Model)] + [_P] * 6, ctypes.c_int
            tiling.argtypes, tiling.restype = [ctypes.POINTER(Shape), ctypes.c_int, ctypes.POINTER(_I)], ctypes.c_int
        lib.mk_prefill_last_error.restype = ctypes.c_char_p
        _lib = lib
    return _lib


def _tensors(model) -> list[Tensor]:
    """The model's bf16 tensors in the order of ``Model``, the rope tables left out."""
    p = model.stacked_params
    return [model.model.embed_tokens.weight, p.attn_ln_weight, p.qkv_proj, p.o_proj, p.mlp_ln_weight, p.gate_proj, p.up_proj,
            p.down_proj, model.lm_head.input_norm.weight, model.lm_head.lm_head.weight, *model.stacked_kv_cache]


def _fits(model, device: int) -> bool:
    """Whether every tensor is what the kernels take it for: bf16 (the rotary tables fp32) on that device, contiguous, in
    16-byte pieces, and of the shape that the configuration says.  The kernels take sizes from the configuration and addresses
    from the tensors, which are public attributes: a shorter one would be read, or the cache written, past its end.  More
    layers than the configuration counts are only more memory."""
    c = model.config
    L, hid, inter, vocab, D = c.num_hidden_layers, c.hidden_size, c.intermediate_size, c.vocab_size, c.head_dim
    q_rows, kv_rows = c.num_attention_heads * D, c.num_key_value_heads * D
    tensors = _tensors(model)
    embed, attn_norm, qkv, o, mlp_norm, gate, up, down, final_norm, head, k_cache, v_cache = [t.shape for t in tensors]
    for shape, expected in ((attn_norm, (L, hid)), (qkv, (L, q_rows + 2 * kv_rows, hid)), (o, (L, hid, q_rows)), (mlp_norm, (L, hid)),
                            (gate, (L, inter, hid)), (up, (L, inter, hid)), (down, (L, hid, inter))):
        if shape != expected and (shape[1:] != expected[1:] or shape[0] < L):
            return False
    rope = (model.model.rope_cos, model.model.rope_sin)
    cos, sin = [t.shape for t in rope]
    if (L < 1 or embed != (vocab, hid) or head != embed or final_norm != (hid,)
            or k_cache != v_cache or len(k_cache) != 5 or k_cache[0] < L or k_cache[3] != c.num_key_value_heads or k_cache[4] != D
            or cos != sin or len(cos) != 2 or cos[1] != D):
        return False
    for dtype, group in ((torch.bfloat16, tensors), (torch.float32, rope)):
        for t in group:
            if t.dtype is not dtype or t.get_device() != device or not t.is_contiguous() or t.data_ptr() % 16:
                return False
    return True


def _recorded() -> bool:
    """Whether someone writes down the operations that this call runs (``torch.compile``, ``torch.jit.trace``, a dispatch
    mode such as ``make_fx``'s or a flop counter).  A launch through ctypes is none that they see: the record would hold
    empty outputs."""
    return torch.compiler.is_compiling() or torch.jit.is_tracing() or torch._C._len_torch_dispatch_stack() > 0


def covers(model, ids: Tensor, positions: Tensor) -> bool:
    """Whether the HIP forward takes this call: more than one position per sequence, bf16 weights on the GPU in the layout
    that the model's constructors make and of the shapes that its configuration says, and an architecture its kernels are
    built for (head_dim 64 or 128, four query heads per KV head, widths in 16-byte pieces).  Everything else runs through the
    plain PyTorch forward, which also says what is wrong with indices or weights of another type or shape, and so does every
    call whose operations are being recorded."""
    if _recorded():
        return False
    c = model.config
    index = (torch.int64, torch.int32)
    return (ids.is_cuda and ids.shape[-1] > 1 and ids.device == model.device and ids.dtype in index and positions.dtype in index
            and positions.shape == ids.shape[1:] and 0 < ids.shape[0] <= model.stacked_kv_cache[0].shape[1]
            and ids.shape[0] <= 65535 and ids.numel() <= 1 << 22
            and c.head_dim in (64, 128) and c.num_attention_heads == 4 * c.num_key_value_heads
            and c.hidden_size % 8 == 0 and c.hidden_size <= 8192 and c.intermediate_size % 8 == 0 and c.vocab_size % 8 == 0
            and _fits(model, ids.get_device()))


def forward(model, ids: Tensor, positions: Tensor) -> tuple[Tensor, Tensor]:
    """``(hidden states [B, S, hidden], greedy ids [B, S])`` of the prompt ``ids [B, S]`` at ``positions [S]``; the keys
    and values go to the model's cache."""
    lib = load_library()
    c, p = model.config, model.stacked_params
    B, S = ids.shape
    H, KVH, D = c.num_attention_heads, c.num_key_value_heads, c.head_dim
    device = ids.device
    k_cache, v_cache = model.stacked_kv_cache
    ids = ids.to(torch.int64).contiguous()
    positions = positions.to(device=device, dtype=torch.int64).contiguous()
    shape = Shape(B, S, H, KVH, D, c.hidden_size, c.intermediate_size, c.vocab_size, k_cache.shape[2],
                  model.model.rope_cos.shape[0], int(bool(model.extra_config.interleave_rope)), c.rms_norm_eps)
    workspace_bytes = lib.mk_prefill_workspace_bytes(ctypes.byref(shape))
    if workspace_bytes < 0:
        raise RuntimeError(f"mk_prefill_workspace_bytes: {lib.mk_prefill_last_error().decode()}")
    if workspace_bytes:
        return _forward_whole(lib, model, shape, workspace_bytes, ids, positions)
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


def _forward_whole(lib, model, shape, workspace_bytes: int, ids: Tensor, positions: Tensor) -> tuple[Tensor, Tensor]:
    """A prompt that is not too long: one call launches the whole forward, matrix products included.  Issued one by one from
    Python, the launches of a short prompt took longer than the GPU needs for them."""
    c, device = model.config, ids.device
    *weights, k_cache, v_cache = (t.data_ptr() for t in _tensors(model))
    pointers = Model(*weights, model.model.rope_cos.data_ptr(), model.model.rope_sin.data_ptr(), k_cache, v_cache,
                     c.num_hidden_layers, model.stacked_kv_cache[0].shape[1])
    h = torch.empty(*ids.shape, c.hidden_size, dtype=torch.bfloat16, device=device)
    workspace = torch.empty(workspace_bytes, dtype=torch.uint8, device=device)
    out_ids = torch.empty(ids.shape, dtype=torch.int64, device=device)
    with torch.cuda.device(device):
        stream = torch.cuda.current_stream(device).cuda_stream
        if lib.mk_prefill_forward(ctypes.byref(shape), ctypes.byref(pointers), ids.data_ptr(), positions.data_ptr(), h.data_ptr(),
                                  workspace.data_ptr(), out_ids.data_ptr(), stream) != 0:
            raise RuntimeError(f"mk_prefill_forward: {lib.mk_prefill_last_error().decode()}")
    return h, out_ids
