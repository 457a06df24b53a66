"""What a decoder session launches, seen through a stand-in for the device (no GPU)."""
from dataclasses import replace

import numpy as np
import pytest

from karume_amd import decoder
from karume_amd.decoder import LlamaConfig, LlamaDecoderSession, random_weights
from karume_amd.runtime import ExecutionError, GpuOutOfMemoryError
from stand_in_gpu import StandInGpu

CONFIG = LlamaConfig(layers=2, d_model=128, ffn=256, heads=2, kv_heads=1, head_dim=64, vocab=64,
                     group_size=64, max_position=256)


def make_session(gpu, seed, config=CONFIG):
    return LlamaDecoderSession(gpu, random_weights(config, seed=seed), chunk_length=8)


def one_row(session, context, past):
    return session.run(np.array([[1]], dtype=np.int32), np.array([[past]], dtype=np.int32), 0,
                       context=context, query_length=1)


# ---- recorded steps belong to the session that recorded them -----------------------------------

@pytest.mark.parametrize("through", ["run", "decode_tokens"])
def test_a_session_on_another_sessions_context_launches_its_own_weights(through):
    gpu = StandInGpu()
    a, b = make_session(gpu, 1), make_session(gpu, 2)
    context = a.create_generation_context(capacity=64, chunk_length=8)
    b.create_generation_context(capacity=64, chunk_length=8)

    def step(session, past):
        if through == "run":
            one_row(session, context, past)
        else:
            session.decode_tokens(context, 1, 1)
            context.past = past + 1   # (the stand-in's lengths read back as zeros)
    for past, (session, other) in enumerate([(a, b), (a, b), (b, a), (b, a), (a, b), (b, a)]):
        gpu.clear()
        step(session, past)
        for name in ("q", "o", "down"):
            assert not gpu.mentions(other.layers[0][name].w), (past, name)
        assert gpu.mentions(session.layers[1]["down"].w)
        assert gpu.mentions(session.lm_head.w) and not gpu.mentions(other.lm_head.w)
        assert gpu.mentions(session.buf["logits"]) and not gpu.mentions(other.buf["logits"])
    # the context's own session keeps its step; the other runs by plain launches
    assert gpu.open_graphs() == 1
    b.close()
    assert gpu.open_graphs() == 1
    context.dispose()
    a.close()
    assert gpu.open_graphs() == 0


def test_a_closed_session_refuses_every_call_and_launches_nothing():
    gpu = StandInGpu()
    session = make_session(gpu, 3)
    context = session.create_generation_context(capacity=64, chunk_length=8)
    for past in range(3):
        one_row(session, context, past)      # the second and third replay a recorded step
    session.decode_tokens(context, 1, 2)
    context.past = 5
    session.close()
    assert gpu.open_graphs() == 0
    gpu.clear()
    calls = [lambda: one_row(session, context, 5), lambda: session.decode_tokens(context, 1, 1),
             lambda: session.run(np.zeros((1, 8), np.int32), np.zeros((1, 8), np.int32), 7,
                                 context=context, query_length=8),
             lambda: session.create_generation_context(capacity=64, chunk_length=8)]
    for call in calls:
        with pytest.raises(ExecutionError, match="closed"):
            call()
    assert gpu.log == [] and not context.poisoned and context.past == 5
    context.dispose()                        # what is left is the context's own memory
    session.close()
    assert gpu.live == {}


# ---- contexts that are not the session's own ---------------------------------------------------

def test_a_context_on_another_stream_is_not_stepped_through_a_recorded_step():
    """The words of a recorded step travel on the stream of the context's own memory; a session
    whose launches go to another stream must not replay between them."""
    mine, other = StandInGpu(), StandInGpu()
    a, b = make_session(other, 4), make_session(mine, 5)
    context = a.create_generation_context(capacity=64, chunk_length=8)
    b.create_generation_context(capacity=64, chunk_length=8)
    for past in range(4):
        other.clear()
        one_row(b, context, past)
        assert other.log == [], past     # ids and positions went up on b's own stream
    assert mine.open_graphs() == other.open_graphs() == 0
    mine.clear()
    b.decode_tokens(context, 1, 3)
    assert [name for name, _ in other.log] == ["krm_buf_download"]    # the lengths, at the end
    assert mine.open_graphs() == 0


def test_a_replayed_decode_longer_than_the_contexts_own_history():
    gpu = StandInGpu()
    short = make_session(gpu, 6, replace(CONFIG, max_position=16))
    long = make_session(gpu, 7)
    context = short.create_generation_context(capacity=64, chunk_length=8)
    long.create_generation_context(capacity=64, chunk_length=8)
    assert context.memory.history_len == 16
    assert len(long.decode_tokens(context, 1, 40)) == 40


def test_a_context_larger_than_the_sessions_own_needs_no_workspace_ahead():
    """A session that never made a context of this capacity has no workspace, or a smaller one: a
    run is sized for its own columns, not for those that a recorded step would be kept for."""
    gpu = StandInGpu()
    a, b = make_session(gpu, 8), make_session(gpu, 9)
    context = a.create_generation_context(capacity=200, chunk_length=8)
    for past in range(3):
        gpu.clear()
        one_row(b, context, past)
        assert [args[14] for name, args in gpu.log if name == "krm_attention_state"] == [past] * 2
        assert not any(name == "krm_attention_state_lengths" for name, _ in gpu.log)


# ---- memory kept from a retired context ---------------------------------------------------------

def used(gpu):
    return sum(gpu.live.values())


def test_a_session_keeps_one_retired_contexts_memory_and_gives_it_back(monkeypatch):
    gpu = StandInGpu()
    session = make_session(gpu, 10)
    make = lambda: session.create_generation_context(capacity=64, chunk_length=8)  # noqa: E731
    make().dispose()
    with_one, one = used(gpu), session._spare_memory.buffer.nbytes
    first, second = make(), make()
    one_row(session, first, 0), one_row(session, first, 1)
    assert used(gpu) == with_one + one and gpu.open_graphs() == 1
    second.dispose(), first.dispose()              # the second one finds the place taken
    assert used(gpu) == with_one and gpu.open_graphs() == 0
    session.release_spare_memory()
    assert used(gpu) == with_one - one
    session.release_spare_memory()
    monkeypatch.setattr(decoder, "MAX_SPARE_BYTES", one - 1)
    make().dispose()                               # larger than what is worth keeping
    assert used(gpu) == with_one - one


def test_an_allocation_without_room_takes_the_kept_memory_back():
    gpu = StandInGpu()
    session = make_session(gpu, 11)
    make = lambda: session.create_generation_context(capacity=64, chunk_length=8)  # noqa: E731
    make().dispose()
    one = session._spare_memory.buffer.nbytes
    gpu.memory = used(gpu) + one - 1
    buffer = gpu.alloc(one)
    assert session._spare_memory is None
    with pytest.raises(GpuOutOfMemoryError):
        gpu.alloc(one)
    buffer.free()
