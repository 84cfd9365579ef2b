"""The layers of a plain dense decoder launched by one call (csrc/dense_blocks.hip) at sizes whose products, norms and attention take the
kernels that the tiny models of test_engine_gpu.py are too small for."""
import ctypes
from types import SimpleNamespace

import pytest
import torch

from helpers import assert_logits, token_ids

pytestmark = pytest.mark.gpu
DTYPES = ["float32", "bfloat16"]
# heads of 64 without head norms, heads of 128 with them
WIDE = {"llama": dict(architectures=["LlamaForCausalLM"], num_attention_heads=16, num_key_value_heads=4, head_dim=64, rms_norm_eps=1e-5, tie_word_embeddings=False),
        "qwen3": dict(architectures=["Qwen3ForCausalLM"], num_attention_heads=8, num_key_value_heads=4, head_dim=128, rms_norm_eps=1e-6, tie_word_embeddings=True)}


def wide_engine(name, dtype, sizes=None, **options):
    from xeno_rt_amd.config import parse_config
    from xeno_rt_amd.engine import Engine
    raw = {**WIDE[name], **dict(vocab_size=1000, hidden_size=1024, intermediate_size=3072, num_hidden_layers=2, rope_theta=10000.0,
                                max_position_embeddings=4096, hidden_act="silu"), **(sizes or {})}
    return Engine.random(parse_config(raw), seed=5, dtype=dtype, std=0.05, gain_std=0.2, **dict(dict(max_tokens=64 * 64, max_slots=4, graphs=False), **options))


def one_by_one(engine, step):
    """The same step with its layers launched part by part, from the same state of the cache."""
    held = [(slot, engine.length(slot)) for slot, _, _ in step]
    engine.model.one_call = False
    try:
        logits = engine.step(step)
    finally:
        engine.model.one_call = True
    for slot, length in held:
        engine.cache.truncate(slot, length)
    return logits


# ---- one call against part by part ---------------------------------------------------------------------------------------------------------

@pytest.mark.parametrize("pack", ["always", False])
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("name", ["llama", "qwen3"])
def test_layers_of_real_widths_launched_by_one_call(name, dtype, pack, monkeypatch):
    """All logits of a step, to the bits: products cut along k whose second kernel does the norm, or the heads of q, k and v; attention of prompts, cut by keys and
    not, of float32 prompts, of decode steps with a merge, without, and finishing q and k itself. Every kernel of a step lays its workspace behind what is still
    read of the step's memory."""
    engine = wide_engine(name, dtype, pack_weights=pack)
    if dtype == "bfloat16":
        from test_kernels_gpu import parts_of
        assert parts_of(engine.ops, 100, 1024, 3072, "add", True)[2] > 1 and parts_of(engine.ops, 333, 2048, 1024, "store")[2] > 1
        assert bool(engine.ops.lib.xrt_attention_finishes_qkv(1, 8, 4, 128, 0, 1, 128, 4096, 1100))
    ids = token_ids(engine.vocab_size, 2200, seed=3)
    slots = [engine.alloc_slot() for _ in range(4)]
    one_call, taken = engine.ops.dense_blocks, []
    monkeypatch.setattr(engine.ops, "dense_blocks", lambda *arguments, **more: (taken.append(1), one_call(*arguments, **more))[1])
    held = [0] * 4

    def check(counts):
        step = [(slot, ids[at:at + count], list(range(count))) for slot, at, count in zip(slots, held, counts) if count]
        want, before = one_by_one(engine, step), len(taken)
        got = engine.step(step)
        assert len(taken) == before + 1 and torch.isfinite(got).all() and torch.equal(got, want), counts
        held[:] = [at + count for at, count in zip(held, counts)]

    for counts in ([40, 0, 0, 0], [60, 0, 0, 0], [0, 333, 0, 0], [0, 0, 700, 0], [1, 1, 1, 0], [17, 1, 64, 300], [1, 1, 1, 1], [0, 0, 1200, 0], [100, 0, 40, 0], [1, 1, 1, 1],
                   [0, 0, 1, 0]):
        check(counts)
    engine.cache.check()


# ---- the rows that somebody wants, behind the last attention ---------------------------------------------------------------------------

# (heads, key/value heads, dims, tokens, sequences, tokens held before, wanted rows, whether their attention runs alone); measured: the comment at the rule
ALONE = [(32, 8, 128, 2048, 1, 0, 1, True), (32, 8, 128, 8192, 1, 0, 1, True), (32, 8, 128, 333, 1, 3001, 1, True), (32, 8, 128, 8192, 1, 0, 256, True),
         (32, 8, 128, 8192, 1, 0, 2048, False), (32, 8, 128, 8192, 1, 16000, 1024, False), (32, 8, 128, 1000, 1, 16000, 250, False),
         (16, 8, 128, 2048, 1, 4000, 512, False), (64, 8, 128, 2048, 1, 0, 128, True), (32, 8, 64, 17, 1, 16000, 4, True),
         (32, 8, 128, 320, 16, 8000, 16, True), (32, 8, 128, 20, 20, 4000, 5, True), (32, 8, 128, 66000 * 4, 66000, 0, 66000, False),
         (32, 8, 96, 8192, 1, 0, 2048, True)]
ALONE_FLOAT = [(32, 8, 64, 777, 1, 0, 1, True), (32, 8, 64, 2048, 1, 0, 64, True), (32, 8, 64, 2048, 1, 0, 65, False), (32, 8, 64, 2048, 512, 0, 512, True),
               (32, 8, 96, 2048, 1, 0, 512, True)]


@pytest.mark.parametrize("dtype,table", [(0, ALONE_FLOAT), (1, ALONE)])
def test_wanted_rows_go_through_the_attention_alone_where_that_takes_less(dtype, table):
    from xeno_rt_amd.ops import load_ops
    from xeno_rt_amd.ops.hip import DenseLayer, _DenseStep
    lib = load_ops().lib
    for heads, kv_heads, dims, tokens, sequences, held, rows, alone in table:
        layer = DenseLayer(n_heads=heads, n_kv_heads=kv_heads, head_dim=dims)
        count = tokens // sequences
        step = _DenseStep(dtype=dtype, tokens=tokens, hidden=4096, n_seqs=sequences, max_count=count, max_context=held + count, fewest=count)
        assert bool(lib.xrt_dense_wanted_alone(ctypes.byref(layer), ctypes.byref(step), rows)) == alone, (heads, kv_heads, dims, tokens, sequences, held, rows)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("name", ["llama", "qwen3"])
def test_any_number_of_wanted_rows_gives_what_the_whole_step_gives(name, dtype):
    """700 tokens behind 500, some hundred behind none, of which one to a quarter are wanted: their attention alone, and with all of the step's."""
    engine = wide_engine(name, dtype)
    slots = [engine.alloc_slot() for _ in range(3)]
    ids = token_ids(engine.vocab_size, 1200, seed=3)
    engine.step([(slots[0], ids[:500], [])])
    for rows in (1, 3, 20, 70, 175):
        wanted = [699 - 4 * i for i in range(rows)]
        step = [(slots[0], ids[500:], wanted)]
        want = one_by_one(engine, step)
        got = engine.step(step)
        engine.cache.truncate(slots[0], 500)
        assert_logits(got, want.cpu(), dtype, f"{name}, {rows} of 700 rows wanted")
        assert dtype != "float32" or torch.equal(got, want), f"{name}: float32 bits depend on how many rows are wanted"
    step = [(slots[1], ids[:400], list(range(0, 400, 4))), (slots[2], ids[100:333], [5, 232])]
    want = one_by_one(engine, step)
    got = engine.step(step)
    assert_logits(got, want.cpu(), dtype, f"{name}, 102 of 633 rows wanted")
    assert dtype != "float32" or torch.equal(got, want)
    engine.cache.check()


def test_more_wanted_rows_than_a_decode_step_has_sequences(monkeypatch):
    """A decode step has 65535 sequences at most; a step of prompts may want more rows than that."""
    from xeno_rt_amd.parts.attention import Attention
    monkeypatch.setattr(Attention, "WANTED_FROM", 0)
    engine = wide_engine("llama", "bfloat16", dict(hidden_size=64, intermediate_size=64, num_attention_heads=1, num_key_value_heads=1, vocab_size=64,
                                                   num_hidden_layers=1), max_tokens=1024 * 320, max_slots=1024)
    slots = [engine.alloc_slot() for _ in range(1024)]
    ids = token_ids(64, 257 + 1024, seed=4)
    step = [(slot, ids[i:i + 257], [4 * j + 1 for j in range(64)]) for i, slot in enumerate(slots)]
    got = engine.step(step)                                                # 263168 tokens, 65536 of them wanted
    assert got.shape == (65536, 64) and bool(torch.isfinite(got).all())
    for slot in slots:
        engine.free_slot(slot)
    for i in (0, 511, 1023):
        slot = engine.alloc_slot()
        want = engine.step([(slot, step[i][1], list(range(257)))])[step[i][2]]
        engine.free_slot(slot)
        assert_logits(got[64 * i:64 * i + 64], want.cpu(), "bfloat16", f"sequence {i}")


# ---- what `DecoderModel.forward` is given ------------------------------------------------------------------------------------------------

def forward(engine, slot, ids, wanted, without=(), cache=None, **changes):
    """The model on a step of one sequence from its first token, its batch without the fields named."""
    from xeno_rt_amd.engine.batch import build_batch
    engine.cache.reserve(slot, len(ids))
    engine.cache.sync()
    batch = vars(build_batch([slot], [ids], [0], [wanted], "cuda:0"))
    try:
        return engine.model.forward(SimpleNamespace(**{**{name: value for name, value in batch.items() if name not in without}, **changes}), cache or engine.cache)
    finally:
        engine.cache.cancel(slot)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("name", ["llama", "qwen3"])
def test_batches_that_say_less_of_themselves(name, dtype):
    """What a batch need not say: its counts on the host, how its tokens fall into sequences."""
    engine = wide_engine(name, dtype)
    slot, ids = engine.alloc_slot(), token_ids(engine.vocab_size, 150, seed=3)
    want = forward(engine, slot, ids, [0, 70, 149])
    sequences = ("sequence_offsets", "sequence_slots", "sequence_starts", "n_sequences", "max_count", "max_context", "is_decode")
    on_host = ("host_counts", "host_slots", "host_starts")
    for without, changes in ((on_host, {}), (sequences + on_host, {}), (on_host, {"max_count": 0}), (on_host, {"max_context": 0})):
        got = forward(engine, slot, ids, [0, 70, 149], without, **changes)
        assert_logits(got, want.cpu(), dtype, f"{name} without {without} {changes}")
        assert dtype != "float32" or torch.equal(got, want), (without, changes)


class OtherCache:
    """A cache whose last layer's keys and values are not what the model's layers write."""

    def __init__(self, cache, **changes):
        self.cache, self.changes, self.last = cache, changes, len(cache.needs) - 1

    def layer_cache(self, call):
        from dataclasses import replace
        layer = self.cache.layer_cache(call)
        if call != self.last:
            return layer
        return replace(layer, kv=replace(layer.kv, **{name: change(getattr(layer.kv, name)) for name, change in self.changes.items()}))


@pytest.mark.parametrize("dtype", DTYPES)
def test_what_a_layer_is_made_of_is_looked_at_before_anything_runs(dtype, monkeypatch):
    """Caches, weights and norms of another type, size, layout or device are refused, as they are by the parts one by one."""
    from xeno_rt_amd.ops.hip import KernelError, PackedMatrix
    engine = wide_engine("qwen3", dtype)
    slot, ids = engine.alloc_slot(), token_ids(engine.vocab_size, 40, seed=3)
    other = torch.bfloat16 if dtype == "float32" else torch.float32
    want = forward(engine, slot, ids, [39])
    launched = []
    before = engine.ops.lib.xrt_dense_blocks
    monkeypatch.setattr(engine.ops.lib, "xrt_dense_blocks", lambda *arguments: (launched.append(1), before(*arguments))[1])

    def spread(t):                                               # the same elements, each row twice as far from the next
        return torch.stack([t, t], dim=-2).flatten(-3, -2)[..., ::2, :] if t.dim() > 1 else torch.stack([t, t], dim=-1)[..., 0]

    changes = {"another type": lambda t: t.to(torch.float16), "the host": lambda t: t.cpu(), "not contiguous": spread, "fewer rows": lambda t: t[..., :-1].contiguous()}
    for what, change in changes.items():
        for name in ("k", "v"):
            with pytest.raises(KernelError, match="key cache" if name == "k" else "value cache"):
                forward(engine, slot, ids, [39], cache=OtherCache(engine.cache, **{name: change}))
    for change in (lambda t: t.to(other), lambda t: t[:, :2].contiguous()):            # the other compute type; fewer heads
        with pytest.raises(KernelError, match="key cache"):
            forward(engine, slot, ids, [39], cache=OtherCache(engine.cache, k=change, v=change))
    with pytest.raises(KernelError, match="value cache"):
        forward(engine, slot, ids, [39], cache=OtherCache(engine.cache, v=lambda t: t[:-1]))
    for change in (lambda t: t.long(), lambda t: t.cpu(), lambda t: t.reshape(-1), lambda t: t[:, ::2]):
        with pytest.raises(KernelError, match="block table"):
            forward(engine, slot, ids, [39], cache=OtherCache(engine.cache, block_table=change))
    layer = engine.model.spec.layers[-1]
    mixer, feed_forward = layer.mixer, layer.feed_forward
    places = [(mixer, "w_qkv"), (mixer, "w_o"), (feed_forward, "w_gate_up"), (feed_forward, "w_down"), (mixer, "q_norm"), (mixer, "k_norm"),
              (layer.mixer_norm, "weight"), (layer.feed_forward_norm, "weight"), (mixer.position, "theta"), (mixer.position, "table")]
    for part, name in places:
        held = getattr(part, name)
        if held is None:
            continue
        for what, change in changes.items():
            if isinstance(held, PackedMatrix):
                if what == "fewer rows":
                    changed = PackedMatrix(held.data, held.shape[0] - 16, held.shape[1], held.packing)
                else:
                    changed = PackedMatrix(change(held.data), *held.shape, held.packing)
            else:
                changed = change(held)
            with monkeypatch.context() as patch:
                patch.setattr(part, name, changed)
                with pytest.raises(KernelError):
                    forward(engine, slot, ids, [39])
    assert not launched
    assert torch.equal(forward(engine, slot, ids, [39]), want) and len(launched) == 2
