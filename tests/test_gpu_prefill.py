"""The prompt forward's HIP kernels against the plain PyTorch forward on the CPU: hidden states, cache rows and greedy
ids, at the sizes where tiles, waves and position groups begin and end."""

import math

import pytest
import torch

from helpers import config_1b_slice, config_8b_slice, config_tiny
from megakernels_amd import prefill
from megakernels_amd.llama import LlamaForCausalLM, rms_norm
from megakernels_amd.model_types import BatchState, ExtraModelConfig

pytestmark = pytest.mark.gpu


def config_heads_of_128():
    """As wide as the 1B layers, with heads of 128."""
    cfg = config_1b_slice(layers=1, vocab=1024)
    cfg.num_attention_heads, cfg.num_key_value_heads, cfg.head_dim, cfg.intermediate_size = 16, 4, 128, 4096
    return cfg


def _model(cfg, max_len, batch=1, interleave=True, seed=3):
    model = LlamaForCausalLM.from_random(
        cfg, ExtraModelConfig(interleave_rope=interleave, max_len_override=max_len, max_batch_size=batch), seed=seed)
    model.model.embed_tokens.weight.mul_(50)   # unit embedding rows: attention over unlike positions
    return model


def _in_64_bits(model):
    """The model's twin whose plain forward rounds nowhere to bf16."""
    twin = model.to("cpu")
    twin.stacked_params = type(twin.stacked_params)(**{k: v.double() for k, v in vars(twin.stacked_params).items()})
    twin.stacked_kv_cache = tuple(c.double() for c in twin.stacked_kv_cache)
    for holder in (twin.model.embed_tokens, twin.lm_head.input_norm, twin.lm_head.lm_head):
        holder.weight = holder.weight.double()
    return twin


def _compare(cfg, seq, batch=1, interleave=True, positions=None, max_len=None):
    print(f"prefill hidden={cfg.hidden_size} D={cfg.head_dim} seq={seq} batch={batch} interleave={interleave}", flush=True)
    model = _model(cfg, max_len or seq + 3, batch, interleave)
    model_gpu = model.to("cuda:0")
    ids = torch.randint(0, cfg.vocab_size, (batch, seq), generator=torch.Generator().manual_seed(seq))
    positions = torch.arange(seq) if positions is None else positions
    assert prefill.covers(model_gpu, ids.to("cuda:0"), positions)
    ref = model(BatchState(input_ids=ids, position_ids=positions))
    out = model_gpu(BatchState(input_ids=ids.to("cuda:0"), position_ids=positions.to("cuda:0")))
    # Both forwards round to bf16 at the same points and sum in fp32 in different orders, so any of the dozen roundings
    # of a layer may fall the other way: 2^-9 of a value each, independent of each other.
    bound = math.sqrt(12 * cfg.num_hidden_layers) * 2.0**-9
    # Few rows: the norm's two roundings are one, at another point, so the two forwards share fewer of them.  What holds
    # there is that the GPU's rounds no more often: it is as close to the forward without roundings as the plain one is,
    # up to the scatter of two such distances (a quarter, at the smallest size of a thousand values).
    exact = None
    if batch * seq <= 64:
        twin = _in_64_bits(model)
        exact = twin(BatchState(input_ids=ids, position_ids=positions)).hidden_states, *twin.stacked_kv_cache
    for i, (name, a, b) in enumerate((("hidden", out.hidden_states, ref.hidden_states),
                                      ("k", model_gpu.stacked_kv_cache[0], model.stacked_kv_cache[0]),
                                      ("v", model_gpu.stacked_kv_cache[1], model.stacked_kv_cache[1]))):
        a, b = a.cpu().double(), b.double()
        if exact:
            assert a.shape == b.shape and float((a - exact[i]).norm()) <= 1.25 * float((b - exact[i]).norm()), name
            continue
        assert a.shape == b.shape and float((a - b).norm() / b.norm()) <= bound, name
    # greedy ids: the chosen token's logit is the largest one up to what the hidden states differ by
    x = rms_norm(ref.hidden_states, model.lm_head.input_norm.weight, cfg.rms_norm_eps).float()
    logits = x @ model.lm_head.lm_head.weight.float().T
    chosen = logits.gather(-1, out.output_ids.cpu()[..., None])[..., 0]
    slack = 6 * bound * logits.std(dim=-1) + 2.0**-7 * logits.amax(-1).abs()
    assert bool((chosen >= logits.amax(-1) - slack).all())
    assert out.output_ids.shape == (batch, seq) and out.output_ids.dtype == torch.int64


@pytest.mark.parametrize("seq", [2, 15, 31, 32, 33, 63, 64, 65, 127, 130, 257])
def test_prefill_tiny(seq):
    _compare(config_tiny(), seq)


@pytest.mark.parametrize("seq", [5, 64, 193, 777])   # 777: the largest tiles, and a K of four parts
def test_prefill_1b_layers(seq):
    _compare(config_1b_slice(), seq)


@pytest.mark.parametrize("seq", [33, 192, 320])
def test_prefill_8b_layer(seq):
    _compare(config_8b_slice(), seq)


@pytest.mark.parametrize("interleave", [True, False])
def test_prefill_batch_and_both_rotary_layouts(interleave):
    _compare(config_tiny(), 70, batch=3, interleave=interleave)
    _compare(config_8b_slice(), 40, batch=2, interleave=interleave)
    _compare(config_heads_of_128(), 50, batch=3, interleave=interleave)
    _compare(config_heads_of_128(), 500, batch=2, interleave=interleave)   # the largest tiles


@pytest.mark.parametrize("interleave", [True, False])
@pytest.mark.parametrize("batch,seq", [(2, 8), (3, 16), (2, 17), (9, 7), (32, 2)])
def test_prefill_of_few_rows_in_several_sequences(batch, seq, interleave):
    _compare(config_tiny(), seq, batch=batch, interleave=interleave)
    _compare(config_heads_of_128(), seq, batch=batch, interleave=interleave)


def test_prefill_of_few_rows_at_positions_out_of_order():
    order = torch.randperm(90, generator=torch.Generator().manual_seed(1))[:37]
    _compare(config_tiny(), 37, positions=order, max_len=90)


def test_prefill_of_few_rows_takes_the_first_of_equal_logits():
    cfg = config_tiny()
    cfg.vocab_size = 1048   # a last block of 24 columns
    cfg.tie_word_embeddings = False
    model = _model(cfg, 40)
    model.lm_head.lm_head.weight.zero_()
    for first in (0, 17, 1047):
        model.lm_head.lm_head.weight[first:] = model.model.embed_tokens.weight[5]   # equal logits from `first` on
        model_gpu = model.to("cuda:0")
        ids = torch.randint(0, cfg.vocab_size, (1, 33), generator=torch.Generator().manual_seed(0))
        out = model_gpu(BatchState(input_ids=ids.to("cuda:0"), position_ids=torch.arange(33, device="cuda:0"))).output_ids.cpu()
        logit = rms_norm(model(BatchState(input_ids=ids, position_ids=torch.arange(33))).hidden_states,
                         model.lm_head.input_norm.weight, cfg.rms_norm_eps).float() @ model.model.embed_tokens.weight[5].float()
        # a logit's sign is sure beyond six of its rounding errors, the dozen roundings of each of two layers
        sure = logit.abs() > 6 * math.sqrt(24) * 2.0**-9 * logit.std()
        assert bool(sure.sum() > 20) and bool((out == torch.where(logit > 0, first, 0))[sure].all())
        model.lm_head.lm_head.weight.zero_()


def test_prefill_at_positions_out_of_order_and_from_the_end():
    seq = 66
    order = torch.randperm(100, generator=torch.Generator().manual_seed(1))[:seq]
    _compare(config_tiny(), seq, positions=order, max_len=100)
    # negative positions count from the end of the cache and of the rotary table
    _compare(config_tiny(), seq, positions=torch.arange(seq) - seq, max_len=1024)


def test_prefill_long_enough_for_blocks_of_eight_waves():
    # 2 sequences x 2 KV heads x 128 tiles of 64 positions
    cfg = config_tiny(layers=1)
    cfg.max_position_embeddings = 8192
    _compare(cfg, 64 * 127 + 5, batch=2)


def test_index_tensors_of_other_kinds():
    cfg, seq = config_tiny(), 40
    model = _model(cfg, seq).to("cuda:0")
    ids = torch.randint(0, cfg.vocab_size, (1, seq), device="cuda:0")
    positions = torch.arange(seq, device="cuda:0")
    expected = model(BatchState(input_ids=ids, position_ids=positions))
    strided = torch.stack((ids, ids + 1), dim=-1)[..., 0]
    for other_ids, other_positions in ((ids.int(), positions.int()), (strided, positions.cpu()), (ids[0], positions[None])):
        out = model(BatchState(input_ids=other_ids, position_ids=other_positions))
        assert torch.equal(out.hidden_states, expected.hidden_states) and torch.equal(out.output_ids, expected.output_ids)
    assert not prefill.covers(model, ids.double(), positions) and not prefill.covers(model, ids, positions[:1])
    with pytest.raises(RuntimeError):
        model(BatchState(input_ids=ids.double(), position_ids=positions))
    model.stacked_params.gate_proj = model.stacked_params.gate_proj.transpose(1, 2).contiguous().transpose(1, 2)
    assert not prefill.covers(model, ids, positions)   # another layout: the plain forward


@pytest.mark.parametrize("seq", [40, 90])
def test_whole_forward_in_a_captured_graph(seq):
    cfg = config_tiny()
    model = _model(cfg, seq).to("cuda:0")
    batch = BatchState(input_ids=torch.randint(0, cfg.vocab_size, (1, seq), device="cuda:0"), position_ids=torch.arange(seq, device="cuda:0"))
    expected = model(batch).hidden_states.clone()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = model(batch)
    for _ in range(3):
        model.stacked_kv_cache[0].zero_()
        with torch.inference_mode():
            out.hidden_states.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out.hidden_states, expected) and bool(model.stacked_kv_cache[0].any())


def test_argmax_takes_the_first_maximum_and_nan_above_all():
    lib = prefill.load_library()
    import ctypes

    vocab = 1024
    logits = torch.randn(5, vocab).to(torch.bfloat16)
    logits[0] = -3.0
    logits[1, [700, 9, 300]] = 50.0
    logits[2, [40, 600]] = float("nan")
    logits[3] = -float("inf")
    logits[4] = -0.0
    logits[4, 17] = 0.0
    on_gpu = logits.to("cuda:0")
    ids = torch.full((5,), -1, dtype=torch.int64, device="cuda:0")
    shape = prefill.Shape(1, 5, 8, 2, 64, 512, 1024, vocab, 8, 8, 1, 1e-5)
    assert lib.mk_prefill_argmax(ctypes.byref(shape), on_gpu.data_ptr(), ids.data_ptr(), torch.cuda.current_stream().cuda_stream) == 0
    assert ids.cpu().tolist() == [0, 9, 40, 0, 0] == logits.argmax(-1).tolist()


def test_shapes_outside_the_kernels_are_refused():
    import ctypes

    lib = prefill.load_library()
    for field, value in (("head_dim", 96), ("num_attention_heads", 16), ("hidden_size", 516), ("seq", 0), ("vocab_size", 1001)):
        shape = prefill.Shape(1, 5, 8, 2, 64, 512, 1024, 1024, 8, 8, 1, 1e-5)
        setattr(shape, field, value)
        assert lib.mk_prefill_argmax(ctypes.byref(shape), None, None, None) < 0
        assert lib.mk_prefill_last_error()
