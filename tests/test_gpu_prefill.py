"""The prompt forward's HIP kernels against the plain PyTorch forward on the CPU: hidden states, cache rows and greedy
ids, at the sizes where tiles, waves and position groups begin and end."""

import ctypes
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


def config_heads_wider_than_the_stream(hidden=2048):
    """6144 columns of queries, keys and values from a narrower hidden state."""
    cfg = config_1b_slice(layers=1, vocab=1024)
    cfg.hidden_size, cfg.head_dim, cfg.intermediate_size = hidden, 128, 1024
    return cfg


# Sizes above 64 rows at which the forward uses, between them, every tiling that it has for the 1B layers (test_prefill_dispatch.py
# holds these lists, with those below, against the library's own plans), and every kernel instance.
TILED_1B = [70, 150, 200, 253, 300, 540, 777, 1020]
TILED_HEAD = [(128256, 70), (128256, 200), (128200, 777)]                 # vocabulary, rows; 128200: a last tile of 200 columns
TILED_WIDE_HEADS = [(2048, 700), (512, 1400)]                             # hidden size, rows
TILED_NARROW = [(192, 700), (192, 2100)]                                  # hidden sizes that wide tiles do not take
TILED_ARGMAX = [(1048, 90), (10008, 300), (40008, 100), (40008, 200)]     # vocabulary, rows, of the tiny configuration
# The same where wide tiles are among the shapes: layers of the 1B and of the 8B architecture, vocabularies for its last product, and
# heads of 128 from a narrower hidden state.
WIDE_1B = [257, 300, 400, 600, 1100, 1300, 1500, 2300, 2700, 4096]   # 600, 1300, 4096: halves of 256 x 256 tiles
WIDE_8B = [513, 705, 1100, 1300, 1700]
WIDE_HEAD = [(8200, 300), (8200, 700), (24584, 700)]                      # vocabulary, rows; last tiles of 8 columns, halves


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


def _compare(cfg, seq, batch=1, interleave=True, positions=None, max_len=None, norms=False, measured=False):
    print(f"prefill hidden={cfg.hidden_size} D={cfg.head_dim} seq={seq} batch={batch} interleave={interleave} norms={norms}", flush=True)
    model = _model(cfg, max_len or seq + 3, batch, interleave)
    if norms:   # weights from a third to three, as trained ones are
        gen = torch.Generator().manual_seed(9)
        for weight in (model.stacked_params.attn_ln_weight, model.stacked_params.mlp_ln_weight, model.lm_head.input_norm.weight):
            weight.copy_(torch.empty(weight.shape).uniform_(-1.1, 1.1, generator=gen).exp())
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
    if batch * seq <= 64 or measured:
        twin = _in_64_bits(model)
        exact = twin(BatchState(input_ids=ids, position_ids=positions)).hidden_states, *twin.stacked_kv_cache
    if measured:
        # Where a layer adds more than the stream held, its roundings add up to more than their number says.  How much more, the
        # plain forward's own distance says: its deviation, and a quarter as above, take the place of 2^-9 / sqrt(3) a rounding.
        own = float((ref.hidden_states.double() - exact[0]).norm() / exact[0].norm())
        print(f"  the plain forward is {own / bound:.2f} bounds off by itself", flush=True)
        bound = max(bound, 1.25 * math.sqrt(3) * own)
    for i, (name, a, b) in enumerate((("hidden", out.hidden_states, ref.hidden_states),
                                      ("k", model_gpu.stacked_kv_cache[0], model.stacked_kv_cache[0]),
                                      ("v", model_gpu.stacked_kv_cache[1], model.stacked_kv_cache[1]))):
        a, b = a.cpu().double(), b.double()
        # every single value, too: a dozen independent roundings a layer, each with a deviation of 2^-9 / sqrt(3), add up to
        # something like a normal distribution, whose eighth deviation is not met among some millions of values (2.2 bounds
        # at most, of 4.6, in these tests); a value's last rounding is relative to itself
        near = exact[i] if exact else b
        off = (a - near).abs() / torch.maximum(near.pow(2).mean(-1, keepdim=True).sqrt(), near.abs()).clamp_min(1e-30)
        print(f"  {name}: largest difference {float(off.max()) / bound:.2f} of the norm's bound", flush=True)
        assert float(off.max()) <= 8 / math.sqrt(3) * bound, name
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


@pytest.mark.parametrize("seq", [5, 64, 193, 777])   # 777: wide tiles, and a K of four parts
def test_prefill_1b_layers(seq):
    _compare(config_1b_slice(), seq)


@pytest.mark.parametrize("seq", TILED_1B)
def test_every_tiling_of_the_1b_layers(seq):
    _compare(config_1b_slice(), seq)


@pytest.mark.parametrize("vocab,seq", TILED_HEAD)
def test_head_of_the_full_vocabulary(vocab, seq):
    _compare(config_1b_slice(layers=1, vocab=vocab), seq)


@pytest.mark.parametrize("seq", [7, 20, 50, 130, 1100])   # few rows in 16, 32, 64; tiles, narrow and wide
def test_norm_weights_of_every_size(seq):
    _compare(config_1b_slice(vocab=1024), seq, norms=True)


@pytest.mark.parametrize("seq", [40, 320])
def test_norm_weights_between_the_librarys_products(seq):
    cfg = config_8b_slice(layers=2)
    shape = prefill.Shape(1, seq, cfg.num_attention_heads, cfg.num_key_value_heads, cfg.head_dim, cfg.hidden_size, cfg.intermediate_size,
                          cfg.vocab_size, seq, seq, 1, cfg.rms_norm_eps)
    assert prefill.load_library().mk_prefill_workspace_bytes(ctypes.byref(shape)) == 0
    _compare(cfg, seq, norms=True, measured=True)   # (a norm weight of another layer or kind: a distance of 100 % and more)


@pytest.mark.parametrize("seq", [7, 20, 50])   # the other tests' models of few rows fit the last-level cache
def test_prefill_of_few_rows_with_weights_past_the_caches(seq):
    cfg = config_1b_slice(vocab=65536)
    assert 2 * cfg.hidden_size * cfg.vocab_size + 2 * 3 * cfg.num_hidden_layers * cfg.hidden_size * cfg.intermediate_size > 300 << 20
    _compare(cfg, seq)


@pytest.mark.parametrize("seq", [7, 20, 50])
def test_prefill_of_few_rows_with_heads_wider_than_the_stream(seq):
    _compare(config_heads_wider_than_the_stream(), seq)
    _compare(config_heads_wider_than_the_stream(), seq, interleave=False)


@pytest.mark.parametrize("seq", [33, 192, 320])
def test_prefill_8b_layer(seq):
    _compare(config_8b_slice(), seq)


@pytest.mark.parametrize("interleave", [True, False])
def test_prefill_batch_and_both_rotary_layouts(interleave):
    _compare(config_tiny(), 70, batch=3, interleave=interleave)
    _compare(config_8b_slice(), 40, batch=2, interleave=interleave)
    _compare(config_heads_of_128(), 50, batch=3, interleave=interleave)
    _compare(config_heads_of_128(), 500, batch=2, interleave=interleave)
    for hidden, rows in TILED_WIDE_HEADS:
        _compare(config_heads_wider_than_the_stream(hidden), rows, interleave=interleave)   # qkv in the larger tiles


@pytest.mark.parametrize("interleave", [True, False])
@pytest.mark.parametrize("batch,seq", [(2, 8), (3, 16), (2, 17), (9, 7), (32, 2)])
def test_prefill_of_few_rows_in_several_sequences(batch, seq, interleave):
    _compare(config_tiny(), seq, batch=batch, interleave=interleave)
    _compare(config_heads_of_128(), seq, batch=batch, interleave=interleave)


def test_prefill_of_few_rows_at_positions_out_of_order():
    order = torch.randperm(90, generator=torch.Generator().manual_seed(1))[:37]
    _compare(config_tiny(), 37, positions=order, max_len=90)


def _first_of_equal_logits(vocab, seq):
    print(f"equal logits: vocabulary {vocab} seq {seq}", flush=True)
    cfg = config_tiny()
    cfg.vocab_size = vocab
    cfg.tie_word_embeddings = False
    model = _model(cfg, seq + 7)
    head = model.lm_head.lm_head.weight
    favoured = model.model.embed_tokens.weight[5]
    ids = torch.randint(0, cfg.vocab_size, (1, seq), generator=torch.Generator().manual_seed(0))
    hidden = model(BatchState(input_ids=ids, position_ids=torch.arange(seq))).hidden_states
    logit = rms_norm(hidden, model.lm_head.input_norm.weight, cfg.rms_norm_eps).float() @ favoured.float()
    # a logit's sign is sure beyond six of its rounding errors, the dozen roundings of each of two layers
    sure = logit.abs() > 6 * math.sqrt(24) * 2.0**-9 * logit.std()
    assert bool(sure.sum() > 20)
    for first in (0, 17, vocab - 1):
        head.zero_()
        head[first:] = favoured   # equal logits from `first` on
        model_gpu = model.to("cuda:0")
        out = model_gpu(BatchState(input_ids=ids.to("cuda:0"), position_ids=torch.arange(seq, device="cuda:0"))).output_ids.cpu()
        assert bool((out == torch.where(logit > 0, first, 0))[sure].all())


@pytest.mark.parametrize("seq", WIDE_1B)
def test_every_wide_tiling_of_the_1b_layers(seq):
    _compare(config_1b_slice(layers=1, vocab=1024), seq)


@pytest.mark.parametrize("seq", WIDE_8B)
def test_every_wide_tiling_of_the_8b_layers(seq):
    _compare(config_8b_slice(inter=14336), seq, interleave=seq % 200 != 100)


@pytest.mark.parametrize("interleave", [True, False])
def test_wide_tiles_of_several_sequences_and_wide_heads(interleave):
    _compare(config_1b_slice(layers=1, vocab=1024), 531, batch=3, interleave=interleave)
    _compare(config_heads_wider_than_the_stream(1024), 1500, interleave=interleave)
    _compare(config_heads_wider_than_the_stream(), 1900, interleave=interleave)
    order = torch.randperm(900, generator=torch.Generator().manual_seed(1))[:777]
    _compare(config_1b_slice(layers=1, vocab=1024), 777, positions=order, max_len=900, interleave=interleave)


@pytest.mark.parametrize("vocab,seq", WIDE_HEAD)
def test_wide_tiles_take_the_first_of_equal_logits(vocab, seq):
    _first_of_equal_logits(vocab, seq)


@pytest.mark.parametrize("vocab,seq", WIDE_HEAD)
def test_argmax_of_wide_tiles_with_no_positive_logit_and_with_nan(vocab, seq):
    cfg = config_tiny()
    cfg.vocab_size, cfg.tie_word_embeddings = vocab, False
    model = _model(cfg, seq)
    head = model.lm_head.lm_head.weight
    norm = model.lm_head.input_norm.weight
    ids = torch.randint(0, cfg.vocab_size, (1, seq), generator=torch.Generator().manual_seed(0))
    batch = BatchState(input_ids=ids.to("cuda:0"), position_ids=torch.arange(seq, device="cuda:0"))
    norm.zero_()   # logits are zeros of both signs
    assert bool((model.to("cuda:0")(batch).output_ids == 0).all())
    norm.fill_(1.0)
    head[4100], head[vocab - 1] = float("nan"), float("nan")   # above everything, the first of them
    assert bool((model.to("cuda:0")(batch).output_ids == 4100).all())


@pytest.mark.parametrize("vocab,seq", WIDE_HEAD + TILED_ARGMAX)
def test_argmax_of_tiles_where_every_logit_is_negative(vocab, seq):
    """Logits of -1 and -2 times what every row holds in column 0, the larger ones several times over."""
    cfg = config_tiny()
    cfg.vocab_size, cfg.tie_word_embeddings = vocab, False
    model = _model(cfg, seq)
    model.model.embed_tokens.weight[:, 0] = 500.0
    head = model.lm_head.lm_head.weight
    ids = torch.randint(0, cfg.vocab_size, (1, seq), generator=torch.Generator().manual_seed(0))
    batch = BatchState(input_ids=ids.to("cuda:0"), position_ids=torch.arange(seq, device="cuda:0"))
    for equal in ((700, 701, 1000, vocab - 1), (vocab - 3, vocab - 1), (vocab - 1,), (0, 64)):
        head.zero_()
        head[:, 0] = -2.0
        head[list(equal), 0] = -1.0
        out = model.to("cuda:0")(batch)
        assert float(out.hidden_states[..., 0].min()) > 0
        assert bool((out.output_ids == equal[0]).all()), equal


@pytest.mark.parametrize("seq,tiles", [(300, 4), (700, 3)])
def test_silu_of_every_gate_in_wide_tiles(seq, tiles):
    """Every bf16 gate through the two kernels' own exponential and division, against the kernel that has the library's: gate
    `n` is weight `n` of the gate projection times one, up is one, and the down projection leaves it in column `n`."""
    lib = prefill.load_library()
    cfg = config_1b_slice(layers=1, vocab=1024)
    hid, inter = cfg.hidden_size, cfg.intermediate_size
    model = _model(cfg, seq).to("cuda:0")
    p, embed = model.stacked_params, model.model.embed_tokens.weight
    shape = prefill.Shape(1, seq, cfg.num_attention_heads, cfg.num_key_value_heads, cfg.head_dim, hid, inter, cfg.vocab_size, seq,
                          model.model.rope_cos.shape[0], 1, cfg.rms_norm_eps)
    plan = (ctypes.c_int32 * 4)()
    assert lib.mk_prefill_wide_plan(ctypes.byref(shape), 2, plan) == 0 and plan[0] == tiles
    for t in (p.qkv_proj, p.o_proj, p.gate_proj, p.up_proj, p.down_proj, embed):
        t.zero_()
    embed[:, 0] = 64.0
    p.mlp_ln_weight[0, 0] = 1 / hid**0.5   # normed, column 0 is one
    p.up_proj[0, :hid, 0] = 1.0
    p.down_proj[0, :, :hid] = torch.eye(hid)
    batch = BatchState(input_ids=torch.zeros(1, seq, dtype=torch.int64, device="cuda:0"), position_ids=torch.arange(seq, device="cuda:0"))

    def through(gates):   # of columns 1 and up
        p.gate_proj[0, 1:hid, 0] = gates
        return model(batch).hidden_states[0, :, 1:]

    every = torch.arange(65536, dtype=torch.int32).to(torch.int16).view(torch.bfloat16).cuda()
    least = 2.0**-126   # smaller ones the matrix cores may flush, on the way in or out
    gates = every[every.isfinite() & (every.abs() >= least)]
    gates = torch.nn.functional.pad(gates, (0, -len(gates) % 8))
    ones, expected = torch.ones_like(gates), torch.empty_like(gates)
    one_row = prefill.Shape(1, 1, 4, 1, 64, 64, len(gates), 8, 1, 1, 1, 1e-5)
    assert lib.mk_prefill_silu_mul(ctypes.byref(one_row), gates.data_ptr(), ones.data_ptr(), expected.data_ptr(), None) == 0
    torch.cuda.synchronize()
    for first in range(0, len(gates), hid - 1):
        part, want = gates[first:first + hid - 1], expected[first:first + hid - 1]
        got = through(torch.nn.functional.pad(part, (0, hid - 1 - len(part))))[:, :len(part)]
        want = want.expand_as(got)
        sure = want.abs() >= least
        assert torch.equal(got[sure], want[sure]) and bool((got[~sure].abs() <= least).all()), first
    for special, want in ((math.inf, math.inf), (-math.inf, math.nan), (math.nan, math.nan)):
        gate = torch.zeros(hid - 1)
        gate[9] = special
        assert torch.allclose(through(gate)[:, 9].float(), torch.tensor(want, device="cuda:0"), equal_nan=True)


@pytest.mark.parametrize("hidden,seq", TILED_NARROW)
def test_narrow_tiles_of_long_prompts_of_narrow_models(hidden, seq):
    _compare(config_heads_wider_than_the_stream(hidden), seq)
    _compare(config_heads_wider_than_the_stream(hidden), seq, interleave=False)


def test_prefill_of_few_rows_takes_the_first_of_equal_logits():
    _first_of_equal_logits(1048, 33)   # a last block of 24 columns


@pytest.mark.parametrize("vocab,seq", TILED_ARGMAX)   # last tiles of 24, 24, 72 and 72 columns
def test_tiles_take_the_first_of_equal_logits(vocab, seq):
    _first_of_equal_logits(vocab, seq)


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


def test_tensors_that_do_not_fit_and_recorded_calls_run_in_the_plain_forward():
    cfg, seq = config_tiny(), 40
    model = _model(cfg, seq).to("cuda:0")
    batch = BatchState(input_ids=torch.randint(0, 1000, (1, seq), device="cuda:0"), position_ids=torch.arange(seq, device="cuda:0"))
    hidden = model(batch).hidden_states
    bound = math.sqrt(12 * cfg.num_hidden_layers) * 2.0**-9
    compiled = torch.compile(lambda: model(batch).hidden_states, backend="eager", fullgraph=True)()
    assert float((compiled.double() - hidden.double()).norm() / hidden.double().norm()) <= bound
    model.config.vocab_size = 1016   # the plain forward goes by the tensors
    out = model(batch)
    assert float((out.hidden_states.double() - hidden.double()).norm() / hidden.double().norm()) <= bound
    model.config.vocab_size, model.config.num_hidden_layers = 1024, 3
    with pytest.raises(IndexError):
        model(batch)


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


@pytest.mark.parametrize("seq", [300, 1100])
def test_wide_forward_in_a_captured_graph(seq):
    cfg = config_1b_slice(layers=1, vocab=1024)
    model = _model(cfg, seq).to("cuda:0")
    batch = BatchState(input_ids=torch.randint(0, cfg.vocab_size, (1, seq), device="cuda:0"), position_ids=torch.arange(seq, device="cuda:0"))
    expected = model(batch)
    hidden, ids = expected.hidden_states.clone(), expected.output_ids.clone()
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
        assert torch.equal(out.hidden_states, hidden) and torch.equal(out.output_ids, ids) and bool(model.stacked_kv_cache[0].any())
        assert torch.equal(model(batch).hidden_states, hidden)


def test_argmax_takes_the_first_maximum_and_nan_above_all():
    lib = prefill.load_library()
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
    lib = prefill.load_library()
    for field, value in (("head_dim", 96), ("num_attention_heads", 16), ("hidden_size", 516), ("seq", 0), ("vocab_size", 1001)):
        shape = prefill.Shape(1, 5, 8, 2, 64, 512, 1024, 1024, 8, 8, 1, 1e-5)
        setattr(shape, field, value)
        assert lib.mk_prefill_argmax(ctypes.byref(shape), None, None, None) < 0
        assert lib.mk_prefill_last_error()
