"""Layers whose launches are those of the layer before with other tensors: the same bits as layer by layer."""
import pytest
import torch

from tiny import random_tokens

pytestmark = pytest.mark.gpu

WIDE = dict(architectures=["Qwen2ForCausalLM"], model_type="qwen2", hidden_act="silu", num_hidden_layers=6, hidden_size=896,
            num_attention_heads=14, num_key_value_heads=2, intermediate_size=1216, vocab_size=600, rope_theta=1000000.0,
            rms_norm_eps=1e-6, max_position_embeddings=2048, tie_word_embeddings=True, use_sliding_window=False)
ODD = dict(WIDE, num_hidden_layers=5, hidden_size=200, num_attention_heads=9, num_key_value_heads=3, head_dim=48,
           intermediate_size=232, tie_word_embeddings=False)


def build(raw, dtype, seed=3):
    from minfer_amd import DecoderModel, config_from_dict
    config = config_from_dict(raw)
    model = DecoderModel(config.model_spec(), dtype, "cuda:0")
    gen = torch.Generator(device="cuda").manual_seed(seed)

    def get(name):
        shape = tuple(model.expected_tensors()[name].shape)
        t = torch.randn(shape, generator=gen, device="cuda") * (0.1 if len(shape) > 1 else 0.3)
        return (t + (1.0 if "norm" in name else 0.0)).to(torch.bfloat16).to(dtype)
    model.load(get)
    return model


def walk(model, steps):
    """Logits of the steps, each a list of (sequence, new tokens), then of one decode step of every sequence."""
    from minfer_amd import Engine
    eng = Engine(model, max_tokens=4096, max_seqs=4)
    slots, out = [eng.new_sequence() for _ in range(3)], []
    for i, step in enumerate(steps):
        ids = [slots[s] for s, _ in step]
        out.append(eng.step(ids, [random_tokens(600, n, 17 * i + s) for s, n in step], "last").clone())
    out.append(eng.step(slots, [[5], [6], [7]], "last").clone())
    return out


@pytest.mark.parametrize("raw", [WIDE, ODD], ids=["896", "odd"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_the_same_bits(monkeypatch, raw, dtype):
    """Steps of at most 16 rows, of 17 to 64, of more, from a context and of several sequences; every size class has kernels (and
    norms prepared ahead) of its own."""
    from minfer_amd.engine import alike
    from minfer_amd.kernels import ops
    model = build(raw, dtype)
    steps = [[(0, 37)], [(1, 5), (0, 2)], [(2, 130)], [(0, 65), (1, 300), (2, 1)], [(1, 64)], [(0, 16)], [(2, 17)], [(1, 1), (0, 2)]]
    again = []
    checked = ops.check_recorded
    monkeypatch.setattr(ops, "check_recorded", lambda rc: (again.append(rc), checked(rc)))
    got = walk(model, steps)
    # every step makes the launches of all layers but the first two and the last from the record
    assert len(again) >= len(steps) * (raw["num_hidden_layers"] - 3) and not any(again)
    monkeypatch.setattr(alike.AlikeLayers, "forward", lambda self, block, h, ctx, e, w: block.forward(h, ctx, e, w))
    want = walk(model, steps)
    for i, (a, b) in enumerate(zip(got, want)):
        assert torch.isfinite(b).all() and torch.equal(a, b), i


def test_layers_that_are_not_alike(monkeypatch):
    """A layer with another constant, a layer of another type and one whose matrix has no tiled copy take the general path."""
    from minfer_amd.engine import alike
    from minfer_amd.kernels import ops
    from minfer_amd.parts.attention import GQAttention

    class Other(GQAttention):
        def forward(self, x, h, ctx, entry, writes_cache):
            super().forward(x, h, ctx, entry, writes_cache)
            ops.add_rows(h, torch.full_like(h, 0.25))

    model = build(dict(WIDE, num_hidden_layers=9), torch.bfloat16)
    model.blocks[3].mixer.scale *= 1.5
    model.blocks[5].mixer.__class__ = Other
    model.blocks[7].mixer.o.tiled = None
    again = []
    checked = ops.check_recorded
    monkeypatch.setattr(ops, "check_recorded", lambda rc: (again.append(rc), checked(rc)))
    got = walk(model, [[(0, 40)], [(1, 100), (2, 3)]])
    few = len(again)
    monkeypatch.setattr(alike.AlikeLayers, "forward", lambda self, block, h, ctx, e, w: block.forward(h, ctx, e, w))
    want = walk(model, [[(0, 40)], [(1, 100), (2, 3)]])
    assert 0 < few <= 8 and all(torch.equal(a, b) for a, b in zip(got, want))


def test_only_short_steps_are_recorded(monkeypatch):
    """A record holds all scratch of its layer: long steps have none."""
    from minfer_amd import Engine
    from minfer_amd.engine import alike
    from minfer_amd.kernels import ops
    model = build(WIDE, torch.bfloat16)
    eng = Engine(model, max_tokens=8192, max_seqs=2)
    made, record = [], ops.record_launches
    monkeypatch.setattr(ops, "record_launches", lambda: (made.append(1), record())[1])
    most = alike.MOST_VALUES // WIDE["hidden_size"]
    for n, recorded in ((most, True), (most + 1, False)):
        slots = [eng.new_sequence(), eng.new_sequence()]
        eng.step(slots, [random_tokens(600, n - 1000, n), random_tokens(600, 1000, n)], "last")
        assert bool(made) == recorded
        made.clear()
        for slot in slots:
            eng.end_sequence(slot)


def test_the_record_is_gone_before_the_last_block(monkeypatch):
    """As much memory is allocated when the last block begins, and at most as much when the head does, as layer by layer."""
    from minfer_amd import Engine
    from minfer_amd.engine import alike
    model = build(WIDE, torch.bfloat16)
    eng = Engine(model, max_tokens=4096, max_seqs=2)
    last, head, seen = model.blocks[-1].forward, model.head.forward, []

    def at(fn):
        def call(*args, **kw):
            seen.append(torch.cuda.memory_allocated())
            return fn(*args, **kw)
        return call
    monkeypatch.setattr(model.blocks[-1], "forward", at(last))
    monkeypatch.setattr(model.head, "forward", at(head))
    got = []
    for general in (False, True, False, True):                  # (the first two settle what is kept between steps)
        with monkeypatch.context() as m:
            if general:
                m.setattr(alike.AlikeLayers, "forward", lambda self, block, h, ctx, e, w: block.forward(h, ctx, e, w))
            slot = eng.new_sequence()
            seen.clear()
            eng.step([slot], [random_tokens(600, 900, 1)], "last")
            got.append(tuple(seen))
            eng.end_sequence(slot)
    assert len(got[2]) == 2 and got[2] == got[3]


def test_a_recorded_launch_that_fails_raises_the_kernels_error():
    """(`test_host_call.py`: it ends the layer's launches and the step.)"""
    from minfer_amd.kernels import ops
    ops.check_recorded(0)
    with pytest.raises(ops.KernelError):
        ops.check_recorded(1)
