"""The work that a user of this library has it do, as cases to time and to compare.

The library runs a decoder from token ids to logits: whole prompts in one step, then one token a sequence and step,
through `Engine.step` (and, in the generation loop, the sampler and `Engine.step_from`). The cases are such steps at the
layer sizes that the repository's benchmark and tests name, from a toy model whose steps are all launches to prompts of
8192 tokens. Every layer of a model does the same work, so the large models run here with fewer layers of their sizes:
what a layer costs against the output head stays visible, and making the inputs stays quick.
"""
import math

import torch

from xeno_rt_amd.config import architecture, parse_config
from xeno_rt_amd.engine import Engine
from xeno_rt_amd.sampling import Sampler, SamplerConfig

_LARGE = dict(num_attention_heads=32, num_key_value_heads=8, head_dim=128, tie_word_embeddings=False, hidden_act="silu", torch_dtype="bfloat16",
              max_position_embeddings=16384)
MODELS = {
    "tiny-llama": dict(architectures=["LlamaForCausalLM"], vocab_size=256, hidden_size=64, intermediate_size=176, num_hidden_layers=2,
                       num_attention_heads=4, num_key_value_heads=2, head_dim=16, rms_norm_eps=1e-5, rope_theta=10000.0,
                       max_position_embeddings=128, tie_word_embeddings=False),
    "tiny-qwen3": dict(architectures=["Qwen3ForCausalLM"], vocab_size=384, hidden_size=96, intermediate_size=256, num_hidden_layers=3,
                       num_attention_heads=6, num_key_value_heads=3, head_dim=32, rms_norm_eps=1e-6, rope_theta=1000000.0,
                       max_position_embeddings=256, tie_word_embeddings=True),
    "qwen3-0.6b": dict(_LARGE, architectures=["Qwen3ForCausalLM"], vocab_size=151936, hidden_size=1024, num_attention_heads=16,
                       intermediate_size=3072, num_hidden_layers=28, rms_norm_eps=1e-6, rope_theta=1000000.0, tie_word_embeddings=True),
    "llama32-1b": dict(_LARGE, architectures=["LlamaForCausalLM"], vocab_size=128256, hidden_size=2048, head_dim=64, intermediate_size=8192,
                       num_hidden_layers=16, rms_norm_eps=1e-5, rope_theta=500000.0, tie_word_embeddings=True),
    "llama3-8b": dict(_LARGE, architectures=["LlamaForCausalLM"], vocab_size=128256, hidden_size=4096, intermediate_size=14336,
                      num_hidden_layers=32, rms_norm_eps=1e-5, rope_theta=500000.0),
    "qwen3-8b": dict(_LARGE, architectures=["Qwen3ForCausalLM"], vocab_size=151936, hidden_size=4096, intermediate_size=12288,
                     num_hidden_layers=36, rms_norm_eps=1e-6, rope_theta=1000000.0),
    "qwen3-32b": dict(_LARGE, architectures=["Qwen3ForCausalLM"], vocab_size=151936, hidden_size=5120, num_attention_heads=64,
                      intermediate_size=25600, num_hidden_layers=64, rms_norm_eps=1e-6, rope_theta=1000000.0),
}


def _case(model, kind, sequences, shortest, longest, layers=None, dtype="bfloat16", cached=0, steps=0, all_logits=False):
    """kind "decode": one token for each of `sequences` that hold shortest .. longest tokens; "prompts": that many prompts (or, with
    `cached`, continuations of sequences that hold so many tokens) of shortest .. longest tokens in one step, logits of every last
    token or of all; "generate": prompts, then `steps` greedy steps."""
    return {"model": model, "layers": layers or MODELS[model]["num_hidden_layers"], "dtype": dtype, "kind": kind, "sequences": sequences,
            "shortest": shortest, "longest": longest, "cached": cached, "steps": steps, "all_logits": all_logits}


def listed():
    named = {
        # a toy model's whole request in true float32: prompts of 5 to 17 tokens and eight greedy steps, all launches and host work
        "tiny-generate": _case("tiny-llama", "generate", 3, 5, 17, dtype="float32", steps=8),
        # one user chatting with a small model: a decode step of 28 small layers with head norms, an odd context
        "small-decode-1": _case("qwen3-0.6b", "decode", 1, 333, 333),
        # one user and an 8B model at a context of 4096: a step that reads every weight once
        "8b-decode-1": _case("llama3-8b", "decode", 1, 4095, 4095, layers=6),
        # eight sequences at 4096: what the benchmark is quoted on
        "8b-decode-8": _case("llama3-8b", "decode", 8, 4095, 4095, layers=6),
        # a busy server: 61 sequences of unequal lengths, where the cache weighs as much as the weights
        "8b-decode-61": _case("llama3-8b", "decode", 61, 1027, 4095, layers=4),
        # 32 sequences of a 32B model: wider layers, eight query heads to a key/value head, head norms
        "32b-decode-32": _case("qwen3-32b", "decode", 32, 1500, 2500, layers=3),
        # one prompt of 2048 tokens: what the benchmark quotes as prefill
        "8b-prompt-2048": _case("llama3-8b", "prompts", 1, 2048, 2048, layers=6),
        # a long document: attention weighs more
        "8b-prompt-8192": _case("llama3-8b", "prompts", 1, 8192, 8192, layers=4),
        # eight prompts of 64 to 2048 tokens that start together, head norms
        "8b-prompts-unequal": _case("qwen3-8b", "prompts", 8, 64, 2048, layers=6),
        # the next turn of a conversation: 333 tokens on 3001 that are cached
        "8b-continue-333": _case("llama3-8b", "prompts", 1, 333, 333, layers=6, cached=3001),
        # scoring a sentence: the logits of all of its 100 tokens, heads of 64, tied head
        "1b-score-100": _case("llama32-1b", "prompts", 1, 100, 100, all_logits=True),
        # the true float32 path at real sizes, an odd prompt
        "1b-float32-prompt": _case("llama32-1b", "prompts", 1, 777, 777, layers=8, dtype="float32"),
    }
    return [dict(case, name=name) for name, case in named.items()]


def draw(rng):
    def spread(low, high):
        return min(high, max(low, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))

    kind = rng.choice(["tiny", "decode", "decode", "decode", "prompts", "prompts", "prompts", "continue", "score", "float32"])
    if kind == "tiny":
        model = rng.choice(["tiny-llama", "tiny-qwen3"])
        most = rng.randint(4, 30)
        return _case(model, "generate", rng.randint(1, 8), rng.randint(1, most), most, dtype=rng.choice(["float32", "bfloat16"]), steps=rng.randint(4, 8))
    if kind == "float32":
        longest = spread(16, 777)
        return _case("llama32-1b", "prompts", 1, longest, longest, layers=rng.randint(2, 8), dtype="float32")
    model, layers = rng.choice([("qwen3-0.6b", 28), ("llama32-1b", 16), ("llama3-8b", rng.randint(3, 6)), ("llama3-8b", rng.randint(3, 6)),
                                ("qwen3-8b", rng.randint(3, 6)), ("qwen3-32b", rng.randint(2, 3))])
    if kind == "decode":
        sequences, longest = spread(1, 64), spread(64, 4095)
        return _case(model, "decode", sequences, max(1, int(longest * rng.uniform(0.3, 1.0))), longest, layers=min(layers, 4) if sequences > 16 else layers)
    if kind == "score":
        longest = spread(16, 256)
        return _case(model, "prompts", 1, longest, longest, layers=layers, all_logits=True)
    if kind == "continue":
        longest = spread(2, 1024)
        return _case(model, "prompts", rng.randint(1, 4), max(1, longest // 2), longest, layers=layers, cached=spread(64, 4000))
    sequences = spread(1, 8)
    longest = spread(32, 8192 // sequences)
    return _case(model, "prompts", sequences, max(1, int(longest * rng.uniform(0.1, 1.0))), longest, layers=min(layers, 8192 * 4 // (sequences * longest)) if
                 sequences * longest > 4096 else layers)


# ---- a case's numbers ----------------------------------------------------------------------------------------------------------------

def _config(case):
    return dict(MODELS[case["model"]], num_hidden_layers=case["layers"])


def _lengths(case):
    """The lengths of the case's sequences, spread evenly from the shortest to the longest."""
    n, low, high = case["sequences"], case["shortest"], case["longest"]
    return [high] if n == 1 else [low + (high - low) * i // (n - 1) for i in range(n)]


def _sizes(case):
    c = _config(case)
    d = c["head_dim"]
    return c, c["hidden_size"], c["num_attention_heads"] * d, c["num_key_value_heads"] * d, c["intermediate_size"], c["vocab_size"]


def _tensors(case, seed):
    """The model's tensors by checkpoint name: matrices ~ N(0, 0.02) in the compute dtype, gains around 1."""
    c, h, q, kv, ff, vocab = _sizes(case)
    g = torch.Generator(device="cuda").manual_seed(seed)
    dtype = torch.bfloat16 if case["dtype"] == "bfloat16" else torch.float32

    def matrix(rows, columns):
        return torch.empty(rows, columns, dtype=dtype, device="cuda").normal_(0.0, 0.02, generator=g)

    def gain(n):
        return 1.0 + 0.1 * torch.randn(n, generator=g, device="cuda")

    out = {"model.embed_tokens.weight": matrix(vocab, h), "model.norm.weight": gain(h)}
    if not c["tie_word_embeddings"]:
        out["lm_head.weight"] = matrix(vocab, h)
    for i in range(c["num_hidden_layers"]):
        p = f"model.layers.{i}."
        out.update({p + "input_layernorm.weight": gain(h), p + "post_attention_layernorm.weight": gain(h),
                    p + "self_attn.q_proj.weight": matrix(q, h), p + "self_attn.k_proj.weight": matrix(kv, h), p + "self_attn.v_proj.weight": matrix(kv, h),
                    p + "self_attn.o_proj.weight": matrix(h, q),
                    p + "mlp.gate_proj.weight": matrix(ff, h), p + "mlp.up_proj.weight": matrix(ff, h), p + "mlp.down_proj.weight": matrix(h, ff)})
        if c["architectures"] == ["Qwen3ForCausalLM"]:
            out.update({p + "self_attn.q_norm.weight": gain(c["head_dim"]), p + "self_attn.k_norm.weight": gain(c["head_dim"])})
    return out


def _ids(case, seed):
    """(what every sequence holds in the cache beforehand, the tokens that the pass brings)."""
    g = torch.Generator().manual_seed(seed + 1)
    vocab = MODELS[case["model"]]["vocab_size"]
    draw_ids = lambda n: torch.randint(0, vocab, (n,), generator=g).tolist()  # noqa: E731
    if case["kind"] == "decode":
        return [draw_ids(n) for n in _lengths(case)], [draw_ids(1) for _ in _lengths(case)]
    return [draw_ids(case["cached"]) for _ in _lengths(case)], [draw_ids(n) for n in _lengths(case)]


def prepare(case, seed):
    config = parse_config(_config(case))
    held, new = _ids(case, seed)
    totals = [len(a) + len(b) + case["steps"] for a, b in zip(held, new)]
    engine = Engine(architecture(config.architecture).build(config), _tensors(case, seed), dtype=case["dtype"],
                    max_tokens=sum((n + 63) // 64 * 64 for n in totals), max_slots=len(totals), max_context=max(totals))
    state = {"case": case, "engine": engine, "new": new, "held": [len(ids) for ids in held]}
    if case["kind"] == "generate":
        state["sampler"] = Sampler(engine.ops, engine.device)
        state["greedy"] = [SamplerConfig(temperature=0.0, top_k=0, top_p=1.0, repetition_penalty=1.0)] * len(totals)
    if any(held):
        # the sequences' earlier tokens, up to 8192 of them a step
        state["slots"] = [engine.alloc_slot() for _ in totals]
        step, count = [], 0
        for slot, ids in zip(state["slots"], held):
            if step and count + len(ids) > 8192:
                engine.step(step)
                step, count = [], 0
            step.append((slot, ids, []))
            count += len(ids)
        engine.step(step)
    return state


def run(state):
    case, engine = state["case"], state["engine"]
    if case["kind"] == "generate":
        slots = [engine.alloc_slot() for _ in state["new"]]
        logits = [engine.step([(slot, ids, [len(ids) - 1]) for slot, ids in zip(slots, state["new"])])]
        tokens = []
        rows = [(slot, row) for row, slot in enumerate(slots)]
        for _ in range(case["steps"]):
            tokens.append(state["sampler"].launch(logits[-1], state["greedy"], [[]] * len(slots), [0.0] * len(slots)))
            logits.append(engine.step_from(tokens[-1], rows))
        for slot in slots:
            engine.free_slot(slot)
        return {"logits": logits, "tokens": tokens}
    if any(state["held"]):
        slots = state["slots"]
        for slot, length in zip(slots, state["held"]):
            engine.cache.truncate(slot, length)
    else:
        slots = [engine.alloc_slot() for _ in state["new"]]
    logits = engine.step([(slot, ids, list(range(len(ids))) if case["all_logits"] else [len(ids) - 1]) for slot, ids in zip(slots, state["new"])])
    if not any(state["held"]):
        for slot in slots:
            engine.free_slot(slot)
    return logits


def work(case):
    """Every weight of the layers and the head read once, every cached key and value that is seen read once, those of the new tokens
    written once, the logits written once; the products' operations and causal attention's."""
    c, h, q, kv, ff, vocab = _sizes(case)
    element = 2 if case["dtype"] == "bfloat16" else 4
    per_layer = (q + 2 * kv) * h + h * q + 3 * ff * h
    layers = case["layers"]
    if case["kind"] == "generate":
        steps = [[(0, n) for n in _lengths(case)]] + [[(n + i, 1) for n in _lengths(case)] for i in range(case["steps"])]
    elif case["kind"] == "decode":
        steps = [[(n, 1) for n in _lengths(case)]]
    else:
        steps = [[(case["cached"], n) for n in _lengths(case)]]
    size = flops = 0
    for step in steps:
        tokens = sum(n for _, n in step)
        rows = tokens if case["all_logits"] else len(step)
        keys = sum(before * n + n * (n + 1) // 2 for before, n in step)
        size += (layers * per_layer + vocab * h) * element + layers * 2 * kv * element * sum(before + n for before, n in step) + rows * vocab * 4
        flops += 2 * layers * per_layer * tokens + layers * 4 * q * keys + 2 * vocab * h * rows
    return {"bytes": size, "flops": flops}


def tolerance(case):
    return {"rel": 3e-2, "max": 0.2} if case["dtype"] == "bfloat16" else {"rel": 1e-5, "max": 1e-4, "differ": 0.0}


# ---- the same in 64 bits -------------------------------------------------------------------------------------------------------------

def _norm(x, gain, eps):
    return x * torch.rsqrt((x * x).mean(dim=-1, keepdim=True) + eps) * gain.double()


def _turn(x, base):
    """Pairs (i, i + half) of every head turned by position / base^(2i / size); the angles are those of 32-bit arithmetic, which define them."""
    half = x.shape[-1] // 2
    theta = torch.tensor(base, dtype=torch.float32) ** (2.0 * torch.arange(half, dtype=torch.float32) / float(2 * half))
    angle = (torch.arange(x.shape[0], dtype=torch.float32)[:, None] / theta[None, :]).double().to(x.device)[:, None, :]
    a, b = x[..., :half], x[..., half:]
    return torch.cat([a * angle.cos() - b * angle.sin(), a * angle.sin() + b * angle.cos()], dim=-1)


def _forward(case, w, sequences, tails):
    """Logits in 64 bits of the last `tails[i]` tokens of each whole sequence, one after another."""
    c, h, q_width, kv_width, ff, vocab = _sizes(case)
    heads, groups, d, eps, base = c["num_attention_heads"], c["num_key_value_heads"], c["head_dim"], c["rms_norm_eps"], c["rope_theta"]
    lengths = [len(s) for s in sequences]
    x = w["model.embed_tokens.weight"][torch.tensor(sum(sequences, []), device="cuda")].double()
    for i in range(c["num_hidden_layers"]):
        p = f"model.layers.{i}."
        get = lambda name: w[p + name].double()  # noqa: E731
        y = _norm(x, get("input_layernorm.weight"), eps)
        q, k, v = (y @ get(f"self_attn.{n}_proj.weight").T for n in "qkv")
        outs = []
        for qs, ks, vs in zip(q.split(lengths), k.split(lengths), v.split(lengths)):
            qs, ks, vs = qs.view(-1, heads, d), ks.view(-1, groups, d), vs.view(-1, groups, d)
            if c["architectures"] == ["Qwen3ForCausalLM"]:
                qs, ks = _norm(qs, get("self_attn.q_norm.weight"), eps), _norm(ks, get("self_attn.k_norm.weight"), eps)
            qs, ks = _turn(qs, base) / math.sqrt(d), _turn(ks, base)
            n = qs.shape[0]
            later = torch.ones(n, n, dtype=torch.bool, device="cuda").triu(1)
            out = torch.empty(n, heads, d, dtype=torch.float64, device="cuda")
            for head in range(heads):
                g = head // (heads // groups)
                scores = (qs[:, head].contiguous() @ ks[:, g].T.contiguous()).masked_fill_(later, -math.inf)
                out[:, head] = torch.softmax(scores, dim=-1) @ vs[:, g].contiguous()
            outs.append(out.view(n, q_width))
        x = x + torch.cat(outs) @ get("self_attn.o_proj.weight").T
        wanted = i + 1 == c["num_hidden_layers"]
        if wanted:                                  # behind the last attention only the wanted tokens count
            x = torch.cat([part[-tail:] for part, tail in zip(x.split(lengths), tails)])
        parts = []
        for rows in x.split(16384):
            y = _norm(rows, get("post_attention_layernorm.weight"), eps)
            gate = y @ get("mlp.gate_proj.weight").T
            parts.append(rows + (gate * torch.sigmoid(gate) * (y @ get("mlp.up_proj.weight").T)) @ get("mlp.down_proj.weight").T)
        x = torch.cat(parts)
    head = w["model.embed_tokens.weight" if c["tie_word_embeddings"] else "lm_head.weight"]
    return _norm(x, w["model.norm.weight"], eps) @ head.double().T


def exact(case, seed):
    w = _tensors(case, seed)
    held, new = _ids(case, seed)
    if case["kind"] == "generate":
        sequences, logits, tokens = [list(ids) for ids in new], [], []
        for step in range(case["steps"] + 1):
            logits.append(_forward(case, w, sequences, [1] * len(sequences)))
            if step < case["steps"]:
                tokens.append(logits[-1].argmax(dim=1).to(torch.int32))
                sequences = [ids + [token] for ids, token in zip(sequences, tokens[-1].tolist())]
        return {"logits": logits, "tokens": tokens}
    tokens = sum(len(a) + len(b) for a, b in zip(held, new))
    c, h, q, kv, ff, vocab = _sizes(case)
    if tokens * case["layers"] * 2.0 * ((q + 2 * kv) * h + h * q + 3 * ff * h) > 6e14:         # about 20 seconds in 64 bits
        return None
    return _forward(case, w, [a + b for a, b in zip(held, new)], [len(b) if case["all_logits"] else 1 for b in new])
