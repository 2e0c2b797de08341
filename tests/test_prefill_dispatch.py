"""Which calls the HIP prompt forward takes.  Its kernels get bare addresses and sizes, so a call that does not fit must go
to the plain PyTorch forward; decided on the host, and checked here without a GPU and without a launch."""

import ctypes

import pytest
import torch

from helpers import config_tiny
from megakernels_amd import prefill
from megakernels_amd.llama import LlamaForCausalLM
from megakernels_amd.model_types import BatchState, ExtraModelConfig


class _OnGpu:
    """What ``covers`` asks of the ids, said of ids on a GPU."""

    is_cuda, device, dtype = True, torch.device("cpu"), torch.int64

    def __init__(self, batch, seq):
        self.shape = torch.Size((batch, seq))

    def numel(self):
        return self.shape.numel()

    def get_device(self):
        return -1


def _model(cfg=None, batch=1):
    return LlamaForCausalLM.from_random(cfg or config_tiny(), ExtraModelConfig(max_len_override=32, max_batch_size=batch))


def _covers(model, batch=1, seq=8):
    return prefill.covers(model, _OnGpu(batch, seq), torch.arange(seq))


def _forward(model, seq=8):
    return model(BatchState(input_ids=torch.arange(seq)[None], position_ids=torch.arange(seq)))


def test_models_of_the_constructors_are_taken():
    assert _covers(_model()) and _covers(_model(batch=3), batch=2)
    assert not _covers(_model(), batch=2) and not _covers(_model(), seq=1)


def _set_config(name, value):
    return lambda m: setattr(m.config, name, value)


def _cut_stacked(name, dim):
    def change(m):
        t = getattr(m.stacked_params, name)
        setattr(m.stacked_params, name, t.narrow(dim, 0, t.shape[dim] - 8 if dim else t.shape[dim] - 1).contiguous())
    return change


def _cut_cache(which, dim):
    def change(m):
        caches = list(m.stacked_kv_cache)
        for i in which:
            caches[i] = caches[i].narrow(dim, 0, caches[i].shape[dim] // 2).contiguous()
        m.stacked_kv_cache = tuple(caches)
    return change


def _cut_weight(get, dim, keep):
    def change(m):
        holder = get(m)
        holder.weight = holder.weight.narrow(dim, 0, keep).contiguous()
    return change


MISFITS = {
    "more layers than are stacked": _set_config("num_hidden_layers", 3),
    "no layers": _set_config("num_hidden_layers", 0),
    "a vocabulary larger than the embedding": _set_config("vocab_size", 1032),
    "a vocabulary smaller than the embedding": _set_config("vocab_size", 1016),
    "another intermediate size": _set_config("intermediate_size", 1088),
    "another hidden size": _set_config("hidden_size", 576),
    **{f"{name} of fewer {'layers' if dim == 0 else 'rows' if dim == 1 else 'columns'}": _cut_stacked(name, dim)
       for name, dims in (("qkv_proj", 3), ("o_proj", 3), ("gate_proj", 3), ("up_proj", 3), ("down_proj", 3), ("attn_ln_weight", 2), ("mlp_ln_weight", 2))
       for dim in range(dims)},
    **{f"{'K' if 0 in which else ''}{'V' if 1 in which else ''} cache with half its dimension {dim}": _cut_cache(which, dim)
       for which, dims in (((0,), (0, 1, 2, 3, 4)), ((1,), (0, 1, 2, 3, 4)), ((0, 1), (0, 3, 4))) for dim in dims},
    "a shorter embedding": _cut_weight(lambda m: m.model.embed_tokens, 0, 1000),
    "a narrower embedding": _cut_weight(lambda m: m.model.embed_tokens, 1, 448),
    "a shorter head": _cut_weight(lambda m: m.lm_head.lm_head, 0, 1000),
    "a shorter final norm": _cut_weight(lambda m: m.lm_head.input_norm, 0, 448),
    "a sine table shorter than the cosine's": lambda m: setattr(m.model, "rope_sin", m.model.rope_sin[:100].contiguous()),
    "rotary tables of half the width": lambda m: vars(m.model).update(rope_cos=m.model.rope_cos[:, :32].contiguous(),
                                                                      rope_sin=m.model.rope_sin[:, :32].contiguous()),
    "stacked weights without dimensions": lambda m: vars(m.stacked_params).update({k: torch.ones((), dtype=torch.bfloat16) for k in vars(m.stacked_params)}),
    "a norm weight of another rank": lambda m: setattr(m.stacked_params, "attn_ln_weight", m.stacked_params.attn_ln_weight[0, 0].clone()),
}


@pytest.mark.parametrize("misfit", MISFITS)
def test_tensors_that_do_not_fit_the_configuration_are_not_taken(misfit):
    cfg = config_tiny()
    cfg.tie_word_embeddings = False
    model = _model(cfg, batch=2)
    assert _covers(model)
    MISFITS[misfit](model)
    assert not _covers(model)


def test_what_the_plain_forward_refuses_or_takes_of_them():
    model = _model()
    model.config.num_hidden_layers = 3
    with pytest.raises(IndexError):
        _forward(model)
    model = _model()
    _cut_stacked("gate_proj", 2)(model)
    with pytest.raises(RuntimeError):
        _forward(model)
    model = _model()
    expected = _forward(model)
    model.config.vocab_size = 1016   # the tensors' own sizes count
    assert torch.equal(_forward(model).output_ids, expected.output_ids)


def test_more_stacked_layers_than_are_run_are_taken():
    model = _model(config_tiny(layers=3))
    model.config.num_hidden_layers = 2
    assert _covers(model)


def test_calls_that_are_recorded_are_not_taken():
    """Tracing, compiling and dispatch modes see PyTorch's operations only."""
    from torch.fx.experimental.proxy_tensor import make_fx
    from torch.utils.flop_counter import FlopCounterMode

    model = _model()
    taken = []

    def step(x):
        taken.append(_covers(model))
        return x + 1

    step(torch.zeros(2))
    torch.jit.trace(step, (torch.zeros(2),), check_trace=False)
    make_fx(step)(torch.zeros(2))
    with FlopCounterMode(display=False):
        step(torch.zeros(2))
    step(torch.zeros(2))
    assert taken == [True, False, False, False, True]
    assert torch.equal(torch.compile(lambda x: x + int(_covers(model)), backend="eager", fullgraph=True)(torch.zeros(2)), torch.zeros(2))


def _workspace(rows, hidden, batch=1, inter=None):
    shape = prefill.Shape(batch, rows // batch, 32, 8, 64, hidden, inter or 4 * hidden, 32768, rows, rows, 1, 1e-5)
    return prefill.load_library().mk_prefill_workspace_bytes(ctypes.byref(shape))


@pytest.mark.parametrize("hidden,most", [(2048, 4096), (1024, 4096), (512, 4096), (256, 4096), (64, 4096)])
def test_prompts_beyond_the_measured_crossing_take_the_librarys_products(hidden, most):
    assert _workspace(most, hidden) > 0 and _workspace(most, hidden, batch=2) > 0
    assert _workspace(most + 1, hidden) == 0 and _workspace(8192, hidden, batch=4) == 0
    assert _workspace(40, 4096) == 0 and _workspace(40, hidden + 8) == 0
    # what wide tiles do not take
    inter, limit = (1 << 20) + 64, min(4096, (1 << 21) // hidden)
    assert _workspace(limit, hidden, inter=inter) > 0 and _workspace(limit + 1, hidden, inter=inter) == 0


@pytest.mark.parametrize("rows,hidden", [(257, 256), (1000, 2048), (4096, 1024), (513, 4096), (700, 8192)])
def test_one_entry_chooses_between_the_tilings(rows, hidden):
    assert _workspace(rows, hidden) == _wide_workspace(rows, hidden, max_len=rows) > 0
    for product in range(5):
        assert _plan(product, rows, hidden) == _wide_plan(product, rows, hidden)


def _plan(product, rows, hidden=2048, inter=8192, heads=32, kv_heads=8, head_dim=64, vocab=128256):
    shape = prefill.Shape(1, rows, heads, kv_heads, head_dim, hidden, inter, vocab, rows, rows, 1, 1e-5)
    plan = (ctypes.c_int32 * 4)()
    assert prefill.load_library().mk_prefill_tile_plan(ctypes.byref(shape), product, plan) == 0
    return product, plan[0], plan[3]


def test_the_gpu_tests_reach_every_tiling_of_the_1b_layers_and_every_instance():
    import test_gpu_prefill as gpu

    layers, head, square = range(4), 4, 3
    reached = {_plan(product, rows, vocab=8192) for rows in gpu.TILED_1B for product in layers}
    reached |= {_plan(head, rows, vocab=vocab) for vocab, rows in gpu.TILED_HEAD}
    reached |= {_plan(head, rows, 512, 1024, 8, 2, vocab=vocab) for vocab, rows in gpu.WIDE_HEAD}
    reached |= {_plan(product, rows, vocab=1024) for rows in gpu.WIDE_1B for product in range(5)}
    assert {_plan(product, rows) for rows in range(65, 4097) for product in range(5)} <= reached
    # up to 256 rows these plans are of the narrow tiles, which the sizes up to there reach by themselves
    short = {_plan(product, rows, vocab=8192) for rows in gpu.TILED_1B if rows <= 256 for product in layers}
    assert all(_wide_workspace(rows, 2048) == 0 for rows in (65, 256)) and {_plan(product, rows) for rows in range(65, 257) for product in layers} <= short
    reached |= {_plan(product, rows, hidden, 1024, head_dim=128) for hidden, rows in gpu.TILED_WIDE_HEADS + gpu.TILED_NARROW for product in layers}
    reached |= {_plan(head, rows, 512, 1024, 8, 2, vocab=vocab) for vocab, rows in gpu.TILED_ARGMAX}
    epilogue = {0: "rope", 1: "residual", 2: "silu", 3: "residual", 4: "argmax"}
    instances = {(epilogue[product], shape) for product, shape, _ in reached}
    assert instances == {(e, shape) for e in epilogue.values() for shape in range(5)} - {("residual", square)}
    assert {_plan(head, rows, 512, 1024, 8, 2, vocab=vocab)[1] for vocab, rows in gpu.TILED_ARGMAX} == {0, 1, 2, 3}


def _wide_workspace(rows, hidden, batch=1, inter=None, max_len=8192):
    shape = prefill.Shape(batch, rows // batch, 32, 8, 64, hidden, inter or 4 * hidden, 32768, max_len, rows, 1, 1e-5)
    return prefill.load_library().mk_prefill_wide_workspace_bytes(ctypes.byref(shape))


@pytest.mark.parametrize("hidden,least,most", [
    (256, 257, 4096), (1024, 257, 4096), (2048, 257, 4096), (2112, 513, 1024), (3008, 513, 1024), (3072, 513, 2048), (4096, 513, 2048),
    (4160, 513, 1024), (6144, 513, 1024), (6208, 641, 1024), (8192, 641, 1024)])
def test_prompts_that_wide_tiles_take(hidden, least, most):
    assert _wide_workspace(least, hidden) > 0 and _wide_workspace(most, hidden) > 0 and _wide_workspace(most, hidden, batch=2) > 0
    assert _wide_workspace(least - 1, hidden) == 0 and _wide_workspace(most + 1, hidden) == 0
    assert _wide_workspace(most, hidden - 8) == 0 and _wide_workspace(most, hidden, inter=1000) == 0
    assert _wide_workspace(most, hidden, batch=2, max_len=1 << 30) == 0
    assert _wide_workspace(1000, 192) == 0


def _wide_plan(product, rows, hidden=2048, inter=8192, heads=32, kv_heads=8, head_dim=64, vocab=128256):
    shape = prefill.Shape(1, rows, heads, kv_heads, head_dim, hidden, inter, vocab, rows, rows, 1, 1e-5)
    plan = (ctypes.c_int32 * 4)()
    assert prefill.load_library().mk_prefill_wide_plan(ctypes.byref(shape), product, plan) == 0
    return product, plan[0], plan[3]


def test_the_gpu_tests_reach_every_wide_tiling_of_the_1b_and_8b_layers():
    import test_gpu_prefill as gpu

    head, of_8b = 4, dict(hidden=4096, inter=14336, head_dim=128)
    reached = {_wide_plan(product, rows, vocab=1024) for rows in gpu.WIDE_1B for product in range(5)}
    assert {_wide_plan(product, rows) for rows in range(257, 4097) for product in range(4)} <= reached
    reached |= {_wide_plan(product, rows, vocab=4096, **of_8b) for rows in gpu.WIDE_8B for product in range(5)}
    assert {_wide_plan(product, rows, **of_8b) for rows in range(513, 2049) for product in range(4)} <= reached
    of_heads = {_wide_plan(head, rows, 512, 1024, 8, 2, vocab=vocab) for vocab, rows in gpu.WIDE_HEAD}
    assert {shape for _, shape, _ in of_heads} >= {3, 4}   # 256 x 256 and 128 x 256, each with a last tile of 8 columns
    reached |= of_heads
    assert {_wide_plan(head, rows) for rows in range(257, 4097)} <= reached
    # products that K is not split for run in 128 x 256 and 256 x 256, the residual ones in 128 x 256
    flat, square = 4, 3
    assert {(product, shape) for product, shape, _ in reached if shape >= square} == {
        (0, flat), (0, square), (1, flat), (2, flat), (2, square), (3, flat), (head, flat), (head, square)}


def test_tile_plans_are_refused_where_nothing_is_tiled():
    lib = prefill.load_library()
    plan = (ctypes.c_int32 * 4)()
    for rows, hidden, product in ((64, 2048, 0), (4097, 2048, 0), (100, 4096, 0), (100, 2048, 5), (100, 2048, -1)):
        shape = prefill.Shape(1, rows, 32, 8, 64, hidden, 8192, 32768, rows, rows, 1, 1e-5)
        assert lib.mk_prefill_tile_plan(ctypes.byref(shape), product, plan) < 0 and lib.mk_prefill_last_error()


def test_wide_plans_and_forwards_are_refused_where_there_are_none():
    lib = prefill.load_library()
    plan = (ctypes.c_int32 * 4)()
    for rows, hidden, product in ((256, 2048, 0), (4097, 2048, 0), (512, 4096, 0), (2049, 4096, 0), (1000, 2048, 5), (1000, 2048, -1)):
        shape = prefill.Shape(1, rows, 32, 8, 64, hidden, 8192, 32768, rows, rows, 1, 1e-5)
        assert lib.mk_prefill_wide_plan(ctypes.byref(shape), product, plan) < 0 and lib.mk_prefill_last_error()
    shape = prefill.Shape(1, 1000, 32, 8, 64, 2048, 8192, 32768, 1000, 1000, 1, 1e-5)
    assert lib.mk_prefill_wide_plan(ctypes.byref(shape), 0, None) < 0
    assert lib.mk_prefill_wide_forward(ctypes.byref(shape), None, None, None, None, None, None, None) < 0 and lib.mk_prefill_last_error()


@pytest.mark.parametrize("rows,hidden", [(256, 256), (129, 256), (1000, 256), (200, 2048)])
def test_gate_and_up_of_more_columns_than_32_bits_address_run_in_narrow_tiles(rows, hidden):
    """256 x 256 tiles address gate and up's output, 256 rows of it, with 32 bits: the forward that takes intermediate sizes
    beyond 2^20 must not run it in them."""
    square, up = 3, 2
    assert _plan(up, rows, hidden, 1 << 20)[1] == square
    for inter in ((1 << 20) + 64, 4194368, 8388672, (1 << 25) + 64):   # 8388672: 256 rows are 2^32 bytes and a little
        assert _workspace(rows, hidden, inter=inter) > 0 and _wide_workspace(rows, hidden, inter=inter) == 0
        assert _plan(up, rows, hidden, inter)[1] < square


def test_rotation_is_not_planned_for_halves_of_tiles_that_it_does_not_have():
    """Two whole rounds of 256 x 256 tiles take longer than two of 128 x 256, which one and a half would not."""
    flat, qkv = 4, 0
    assert {_wide_plan(qkv, rows, head_dim=128)[1] for rows in range(2689, 4097)} == {flat}   # 6144 columns


def test_plans_count_the_rounds_of_the_xcd_with_the_most_column_tiles():
    """Column tile n is XCD n % 8's, of 32 CUs with one block of these shapes each: a plan must not need a second round there
    while another shape needs one that is less than twice as long."""
    qkv, o, down, medium, two_a_cu, flat = 0, 1, 3, 1, 2, 4
    # 12 tiles of 128 columns and 20 row tiles: two rounds of 40 tiles a XCD, where 128 x 256 has one of 20
    for rows in (2049, 2300, 2500):
        shape = dict(hidden=1536, inter=6144, heads=24, kv_heads=6)
        assert _wide_plan(o, rows, **shape)[1:] == (flat, 1) and _wide_plan(down, rows, **shape)[1:] == (flat, 1)
        # 12 tiles of 256 columns of the 1B architecture, 17 to 20 row tiles
        assert _wide_plan(qkv, rows)[1:] == (two_a_cu, 1)
    # K in four parts only where all of them are in one round
    assert _wide_plan(down, 560, hidden=2304, inter=9216, heads=20, kv_heads=5, head_dim=128)[1:] == (medium, 2)
