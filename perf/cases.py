"""What a user of this package has it do, as cases that can be timed and compared.

Three kinds of work, each through the public entry points:

* ``decode``: ``MK_Generator.generate`` - greedy batch-1 decode of ``ntok`` tokens behind ``context`` cached positions,
  as ``scripts/generate.py`` and ``bench.py`` run it: one megakernel launch for the whole run of steps.
* ``prefill``: the model's forward over a prompt of ``context`` tokens, which fills the KV cache and yields the hidden
  state and the greedy token of every position - what every script runs before it decodes.
* ``turn``: one turn of ``scripts/llama_repl.py``: prefill of the conversation so far, then ``generate_with_eos`` in
  chunks of 16 tokens with the end-of-sequence check on the host after each chunk.

The models are the two architectures that the package's configurations name, at full size and in bf16.
"""

import math

import torch

from megakernels_amd.demos.latency.scheduler import LatencyScheduleBuilder, pick_num_attention_partitions
from megakernels_amd.dispatch import make_mk_interpreter
from megakernels_amd.generators import MK_Generator
from megakernels_amd.llama import LlamaConfig, LlamaForCausalLM
from megakernels_amd.model_types import BatchState, ExtraModelConfig
from megakernels_amd.scheduler import assign_to_sms, tensorize_instructions

DEVICE = "cuda:0"
EOS_CHECK_INTERVAL = 16  # tokens between two looks for an end-of-sequence id, as in scripts/llama_repl.py
ARCHITECTURES = {"1b": LlamaConfig.llama_1b, "8b": LlamaConfig.llama_8b}


def listed():
    def case(name, kind, arch, context, ntok=0):
        return {"name": name, "kind": kind, "arch": arch, "context": context, "ntok": ntok}

    return [
        # a program that shows every token as it comes: one token per call, right after a short prompt
        case("decode_1b_single", "decode", "1b", 45, 1),
        # a chunk of an answer some way into a chat; a context that is no multiple of anything
        case("decode_1b_chat", "decode", "1b", 437, 16),
        # the benchmark's headline workload: 4096 cached positions
        case("decode_1b_4k", "decode", "1b", 4096, 16),
        # the longest context of the scripts' default cache (max_len_override = 16384 and what follows it)
        case("decode_1b_16k", "decode", "1b", 16384, 16),
        # the larger model behind a short prompt
        case("decode_8b_short", "decode", "8b", 32, 16),
        # the larger model behind a long document: split KV with the reduction tree
        case("decode_8b_32k", "decode", "8b", 32768, 8),
        # a one-line prompt: latency of the forward, launches count
        case("prefill_1b_prompt", "prefill", "1b", 32),
        # a page of text, odd length
        case("prefill_1b_page", "prefill", "1b", 777),
        # a long document
        case("prefill_1b_4k", "prefill", "1b", 4096),
        # the larger model: a one-line prompt, and a few pages
        case("prefill_8b_prompt", "prefill", "8b", 32),
        case("prefill_8b_2k", "prefill", "8b", 2048),
        # a chat turn: the conversation so far prefilled, then four chunks of the answer
        case("turn_1b", "turn", "1b", 253, 64),
    ]


def draw(rng):
    """A case of the same ranges: sizes spread over their logarithm, odd ones as likely as even ones."""
    def size(low, high):
        return min(high, int(math.exp(rng.uniform(math.log(low), math.log(high + 1)))))

    kind = rng.choice(["decode", "decode", "decode", "prefill", "prefill", "turn"])
    arch = rng.choice(["1b", "1b", "8b"])
    if kind == "decode":
        return {"kind": kind, "arch": arch, "context": size(16, 16384 if arch == "1b" else 32768), "ntok": size(1, 16 if arch == "1b" else 8)}
    if kind == "prefill":
        return {"kind": kind, "arch": arch, "context": size(8, 4096 if arch == "1b" else 2048), "ntok": 0}
    return {"kind": kind, "arch": arch, "context": size(16, 2048 if arch == "1b" else 512), "ntok": size(17, 64) if arch == "1b" else size(4, 10)}


def _model(arch, max_len, seed):
    """A randomly initialised model with two properties of a trained one.  Its residual stream is carried, not swamped, by
    the layers: embedding rows of unit size, matrices that keep the size of what they multiply, and the projections into
    the stream scaled by 1 / sqrt(2 L) as training starts from.  Its next-token distribution is peaked: the LM head favours one successor for every token.  (With independent
    random rows the two best of 128256 logits lie within a bf16 rounding of each other in one position of twenty, and
    greedy tokens say nothing.)"""
    config = ARCHITECTURES[arch]()
    config.tie_word_embeddings = False
    unit = config.hidden_size ** -0.5
    model = LlamaForCausalLM.from_random(config, ExtraModelConfig(interleave_rope=True, max_len_override=max_len), seed=seed,
                                         device=DEVICE, std=unit, draw_device=DEVICE)
    embed = model.model.embed_tokens.weight
    embed.mul_(1 / unit)
    for residual in (model.stacked_params.o_proj, model.stacked_params.down_proj):
        residual.mul_((2 * config.num_hidden_layers) ** -0.5)
    model.lm_head.lm_head.weight.copy_(embed.roll(1, 0)).mul_(unit)
    return model


def _generator(model, context, ntok):
    c = model.config
    partitions = pick_num_attention_partitions(context, ntok, DEVICE, c.num_key_value_heads, c.head_dim)
    schedule = LatencyScheduleBuilder.build(model, num_attention_partitions=partitions)
    tensorize_instructions(schedule.globs, assign_to_sms("rr", schedule=schedule))
    return MK_Generator(model, make_mk_interpreter("latency"), schedule)


@torch.no_grad()
def prepare(case, seed):
    """The model with its weights and KV cache, the schedule, and the tokens: resident on the GPU, as in a program that
    has answered before.  For ``decode`` the cached positions hold N(0, 1) rows, as rotated keys and values roughly do."""
    torch.cuda.set_device(DEVICE)
    kind, context, ntok = case["kind"], case["context"], case["ntok"]
    model = _model(case["arch"], context + ntok + 16, seed)
    gen = torch.Generator(device=DEVICE).manual_seed(seed + 1)
    state = {"kind": kind, "context": context, "ntok": ntok, "model": model}
    if kind != "decode":
        state["input_ids"] = torch.randint(0, model.config.vocab_size, (1, context), generator=gen, device=DEVICE)
    else:
        for cache in model.stacked_kv_cache:
            for layer in range(cache.shape[0]):
                cache[layer, :, :context] = torch.randn(cache[layer, :, :context].shape, generator=gen, device=DEVICE).to(cache.dtype)
    if kind != "prefill":
        state["tokens"] = torch.zeros(1, ntok + 1, device=DEVICE, dtype=torch.long)
        state["tokens"][0, 0] = torch.randint(0, model.config.vocab_size, (), generator=gen, device=DEVICE)
        state["generator"] = _generator(model, context, ntok)
    return state


@torch.no_grad()
def run(state):
    model, context, ntok = state["model"], state["context"], state["ntok"]
    k_cache, v_cache = model.stacked_kv_cache
    if state["kind"] != "decode":
        out = model(BatchState(input_ids=state["input_ids"], position_ids=torch.arange(context, device=DEVICE)))
        if state["kind"] == "prefill":
            return {"hidden_states": out.hidden_states, "output_ids": out.output_ids, "k_cache": k_cache, "v_cache": v_cache}
    generator, tokens = state["generator"], state["tokens"]
    globs = generator.schedule.globs
    result = {"tokens": tokens, "logits": globs.logits, "hidden_states": globs.hidden_states, "k_cache": k_cache, "v_cache": v_cache}
    if state["kind"] == "decode":
        generator.generate(tokens, prompt_len=context, ntok=ntok)
        return result
    tokens[:, 0] = out.output_ids[:, -1]
    # ids outside the vocabulary: the answer never ends by itself, so every pass does the same work
    end, generated = generator.generate_with_eos(tokens, prompt_len=context, ntok=ntok + 1,
                                                 eos_token_check_interval=EOS_CHECK_INTERVAL, eos_token_ids=[-1])
    return {**result, "prompt_hidden_states": out.hidden_states, "end": end, "generated": generated}


def work(case):
    c = ARCHITECTURES[case["arch"]]()
    L, hid, inter, vocab = c.num_hidden_layers, c.hidden_size, c.intermediate_size, c.vocab_size
    H, KVH, D = c.num_attention_heads, c.num_key_value_heads, c.head_dim
    context, ntok = case["context"], case["ntok"]
    layers = L * ((H + 2 * KVH) * D * hid + hid * H * D + 3 * inter * hid)
    matrices, norms, kv_row = layers + vocab * hid, (2 * L + 1) * hid, L * 2 * KVH * D
    nbytes = flops = 0
    if case["kind"] != "decode":
        # every matrix once; per position an embedding row in, a hidden state, a K and V row and a token out; causal attention
        nbytes += 2 * (matrices + norms + context * (2 * hid + kv_row)) + 16 * context
        flops += 2 * context * matrices + L * 2 * H * D * context * (context + 1)
    if case["kind"] != "prefill":
        for pos in range(context, context + ntok):
            # every matrix once, the cached rows in, one row and the logits out
            nbytes += 2 * (matrices + norms + kv_row * (pos + 1) + kv_row + vocab + hid)
            flops += 2 * matrices + L * 4 * H * D * (pos + 1)
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    # Decode follows a fixed order of summation that the package's tests compare bit for bit with a CPU restatement.
    # The forward rounds the residual stream to bf16 twice a layer: against the same forward with attention in fp32 and
    # every product summed in two halves, hidden states differ by 1.0 % (1b) to 1.5 % (8b) of their norm and by at most
    # 0.1 of a value; keys and values by less; no token differs.
    return "exact" if case["kind"] == "decode" else {"rel": 0.03, "max": 0.5, "differ": 0.01}
