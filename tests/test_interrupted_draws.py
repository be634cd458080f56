"""A draw whose consumer uses the model between two of its tokens: its tokens, and what the session then says the caches hold,
are those of a draw that nothing came between; and whatever it uses it on, a stream of its own too, is behind the step that a draw
leaves running.  Device-free: the versions are the graph's host reference, also stood in as captured ones (the first step
launched behind the prompt, the rest replayed), or compiled ones whose streams and graphs only take notes."""

import dataclasses
import functools

import numpy as np
import pytest

import oracle
from iron_amd.applications.llama import Llama
from iron_amd.applications.tilarax import Tilarax
from iron_amd.common import graph
from iron_amd.lm import Sampler
from iron_amd.lm.batched import BatchedOnHost, _HostBatchVersion
from iron_amd.lm.causal import OnHost, _HostVersion
from iron_amd.lm.session import Session
from tests.llama_support import SCALED, weights
from tests.tilarax_support import built as tilarax

oracle.install()

CONFIG = dataclasses.replace(SCALED, prefill_chunk=16, max_seq_len=48, num_hidden_layers=1)
RING = dataclasses.replace(CONFIG, max_seq_len=192, sliding_window=5)


class Captured(_HostVersion):
    """A captured version's contract: ``start`` sets the words, ``replay`` goes on from what the last run carried."""

    captured = True
    hands = True

    def start(self, **values):
        *_, self.words = self(**values)

    def replay(self, n=1):
        for _ in range(n):
            self.start(**self.words)

    def hands_over(self, to):
        return self.hands

    def run_and_start(self, to, *tensors, **values):
        *_, carried = self(*tensors, **values)
        to.start(**carried)
        return carried


class Eager(OnHost, Llama):
    pass


class Replayed(OnHost, Llama):
    def load_versions(self, **_):
        self.use(Captured(self, False), Captured(self, True))


class Started(Replayed):
    """As captured versions that cannot hand over."""

    def load_versions(self, **_):
        super().load_versions()
        self.prompt_chunk.hands = False


def loaded(cls, config):
    model = cls(config, weights(config))
    model.load_versions()
    return model


def other(model, token):
    return (int(token) + 1) % model.config.vocab_size


def another_token(model, prompt, drawn):
    model.logits([*prompt, *drawn[:-1], other(model, drawn[-1])])


def another_token_and_a_step(model, prompt, drawn):
    foreign = [*prompt, *drawn[:-1], other(model, drawn[-1])]
    model.logits(foreign)
    model.logits([*foreign, 3])


def another_history(model, prompt, drawn):
    model.logits(prompt[::-1])


def another_draw(model, prompt, drawn):
    given_up = model.session.draw(prompt[:5], 6, Sampler(1.5, 20, seed=9))
    next(given_up), next(given_up)
    given_up.close()


def another_greedy_draw(model, prompt, drawn):
    assert len(list(model.session.draw(prompt[:5], 6))) == 6


def another_session(model, prompt, drawn):
    Session(model).logits(prompt[3:])


def a_call_of_its_own(model, prompt, drawn):
    model(token=7, position=2)


def versions_loaded_anew(model, prompt, drawn):
    model.load_versions()


def versions_loaded_anew_and_not_captured(model, prompt, drawn):
    OnHost.load_versions(model)


BETWEEN = [versions_loaded_anew, versions_loaded_anew_and_not_captured, another_token, another_token_and_a_step, another_history, another_draw, another_greedy_draw, another_session, a_call_of_its_own]


@functools.cache
def alone(config, sampler, cls, each):
    """A prompt, what is drawn behind it, and the logits behind that."""
    prompt = np.random.default_rng(4).integers(0, config.vocab_size, 21).tolist()
    model = loaded(cls, config)
    tokens = list(model.session.draw(prompt, 4, sampler(), each=each))
    return prompt, tokens, model.logits([*prompt, *tokens])


def sampled():
    return Sampler(1.5, 50, seed=2)


def greedy():
    return None


@pytest.mark.parametrize("between", BETWEEN, ids=lambda f: f.__name__)
@pytest.mark.parametrize("config, sampler, cls, each", [(CONFIG, sampled, Eager, False), (CONFIG, sampled, Replayed, False), (CONFIG, greedy, Replayed, False),
                                                        (CONFIG, sampled, Replayed, True), (CONFIG, sampled, Started, False), (RING, greedy, Replayed, False),
                                                        (RING, greedy, Eager, False)])
def test_what_a_consumer_does_between_two_tokens_changes_nothing(config, sampler, cls, each, between):
    prompt, tokens, behind = alone(config, sampler, cls, each)
    model = loaded(cls, config)
    for places in ((1,), (1, 3), (4,)):
        model.session.forget(0)
        drawn = []
        for token in model.session.draw(prompt, 4, sampler(), each=each):
            drawn.append(token)
            if len(drawn) in places:
                between(model, prompt, drawn)
        assert drawn == tokens, places
        # Whatever the session now takes the caches to hold is there (rows made by a chunk and by steps differ by roundings).
        got = model.logits([*prompt, *tokens])
        assert np.abs(got - behind).max() <= 0.02 * np.abs(behind).max(), places


@pytest.mark.parametrize("cls", [Eager, Replayed, Started])
def test_two_draws_of_one_session_taken_in_turn(cls):
    prompts = [np.random.default_rng(s).integers(0, CONFIG.vocab_size, n).tolist() for s, n in ((4, 21), (5, 9))]
    want = [list(loaded(cls, CONFIG).session.draw(p, 5)) for p in prompts]
    model = loaded(cls, CONFIG)
    assert list(zip(*(model.session.draw(p, 5) for p in prompts))) == list(zip(*want))


def test_a_draw_that_nothing_came_between_runs_nothing_twice():
    model, runs = loaded(Replayed, CONFIG), []
    prompt = np.random.default_rng(4).integers(0, CONFIG.vocab_size, 21).tolist()
    call = Captured.__call__
    for version in (model.decode_step, model.prompt_chunk):
        version.__class__ = type("Counted", (Captured,), {"__call__": lambda self, *t, **v: (runs.append(v["position"]), call(self, *t, **v))[1]})
    assert len(list(model.session.draw(prompt, 5))) == 5
    assert runs == [15, 20, 21, 22, 23, 24]
    assert model.session.cached.size == 25


def test_versions_stood_in_by_what_is_called_started_and_replayed_alone():
    """``use`` takes versions that hold no more than a session needs of them: they run, and none is asked to hand over."""
    whole = loaded(Replayed, CONFIG)

    class Called:
        def __init__(self, version, **more):
            self.version = version
            vars(self).update(more)

        def __call__(self, *tensors, **values):
            return self.version(*tensors, **values)

    model = Llama(CONFIG, weights(CONFIG))
    step = whole.decode_step
    model.use(Called(step, captured=True, start=step.start, replay=step.replay, write=step.write, read=lambda resident: step.read(whole.drawn)), Called(whole.prompt_chunk))
    prompt, tokens, behind = alone(CONFIG, greedy, Replayed, False)
    assert list(model.session.draw(prompt, 4)) == tokens
    assert np.array_equal(model.logits([*prompt, *tokens]), behind)


# ---------------------------------------------------------------- a conversation as one request of a batched model
class ReplayedBatch(_HostBatchVersion):
    captured = True

    def start(self):
        self()

    def replay(self, n=1):
        for _ in range(n):
            self()


class EagerTilarax(BatchedOnHost, Tilarax):
    pass


class ReplayedTilarax(BatchedOnHost, Tilarax):
    def load_versions(self, **_):
        self.use(ReplayedBatch(self), ReplayedBatch(self, "ids"), ReplayedBatch(self, "picks"))


def batched(cls):
    model, _ = tilarax("mixed", cls, activations=np.float32, max_seq_len=64, prefill_chunk=16, slots=2)
    model.load_versions()
    return model


def a_batch_of_others(model, prompt, drawn):
    model.generate_batch([prompt[:3]], 3, [Sampler(1.5, 20, seed=9)])


def everything_forgotten(model, prompt, drawn):
    model.session.forget(0)
    assert len(model.generate_batch([prompt[:3], prompt[:4]], 2)) == 2


@functools.cache
def alone_in_a_batch(cls, each):
    model = batched(cls)
    prompt = np.random.default_rng(4).integers(0, model.config.vocab_size, 21).tolist()
    tokens = list(model.session.draw(prompt, 4, Sampler(1.5, 20, seed=2), each=each))
    return prompt, tokens, model.logits([*prompt, *tokens])


@pytest.mark.parametrize("between", [another_token, another_token_and_a_step, another_history, another_draw, another_greedy_draw, a_batch_of_others, everything_forgotten],
                         ids=lambda f: f.__name__)
@pytest.mark.parametrize("cls, each", [(EagerTilarax, False), (ReplayedTilarax, False), (ReplayedTilarax, True)])
def test_what_a_consumer_does_between_two_tokens_of_a_request_changes_nothing(cls, each, between):
    prompt, tokens, behind = alone_in_a_batch(cls, each)
    model = batched(cls)
    for places in ((1,), (1, 3), (4,)):
        model.session.forget(0)
        drawn = []
        for token in model.session.draw(prompt, 4, Sampler(1.5, 20, seed=2), each=each):
            drawn.append(token)
            if len(drawn) in places:
                between(model, prompt, drawn)
        assert drawn == tokens, places
        got = model.logits([*prompt, *tokens])
        assert np.abs(got - behind).max() <= 1e-4 * np.abs(behind).max(), places   # (float32 states, in whatever portions)
    pair = [list(batched(cls).session.draw(p, 4)) for p in (prompt, prompt[7:15])]
    assert list(zip(*(model.session.draw(p, 4) for p in (prompt, prompt[7:15])))) == list(zip(*pair))


class Notes:
    """Streams, events and graphs that note, a stream each, what would be put on it."""

    def __init__(self, monkeypatch):
        import torch

        self.on = {"own": [], "other": [], "host": []}
        self.stream = "own"
        notes = self

        class Event:
            def record(self):
                pass

            def synchronize(self):
                pass

        class Stream:
            def __init__(self):
                self.name = notes.stream

            def wait_stream(self, other):
                notes.on[self.name].append(("behind", other.name))

            def synchronize(self):
                notes.on["host"].append(("behind", self.name))

        monkeypatch.setattr(torch.cuda, "Event", Event)
        monkeypatch.setattr(torch.cuda, "current_stream", Stream)
        monkeypatch.setattr(graph, "current_stream", lambda: notes.stream)
        monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
        monkeypatch.setattr(torch.Tensor, "record_stream", lambda tensor, stream: notes.put("held"))

    def put(self, what):
        self.on[self.stream].append(what)

    def replay(self):   # a captured graph's
        self.put("graph")


USES = {
    "a call": lambda model, prompt: prompt.run(np.zeros(CONFIG.prefill_chunk, np.int32), token=1, position=0, start=0, rows=1, rope_start=0),
    "a start": lambda model, prompt: model.decode_step.start(token=1, position=3),
    "a replay": lambda model, prompt: model.decode_step.replay(2),
    "a write": lambda model, prompt: model.decode_step.write(model.draws, np.zeros((CONFIG.max_seq_len, 4), np.int32)),
    "a read": lambda model, prompt: model.decode_step.read(model.drawn),
}


@pytest.mark.parametrize("use", [*USES, "a release"])
def test_the_step_that_a_draw_leaves_running_is_ahead_of_whatever_comes_next(monkeypatch, use):
    import torch

    from iron_amd import kernels
    from iron_amd.common.graph import WORD_SLOTS, CompiledGraph

    model = Llama(CONFIG, weights(CONFIG))
    decode, prompt = (model.compile(capture=True, **shapes) for shapes in model.shapes())
    model.use(decode, prompt)
    notes = Notes(monkeypatch)
    arena = model.arena
    arena.load("cpu")
    monkeypatch.setattr(CompiledGraph, "load", lambda self: self)
    monkeypatch.setattr(kernels, "copy_rows", lambda *a, **k: notes.put("token"))
    pinned_empty = torch.empty
    monkeypatch.setattr(torch, "empty", lambda *shape, pin_memory=False, **kw: pinned_empty(*shape, **kw))
    monkeypatch.setattr(torch.Tensor, "pin_memory", lambda tensor: tensor)
    for version in (decode, prompt):
        version.words = arena.view(arena.resident_offsets[id(version._words_resident)], (WORD_SLOTS,), np.int32)
        version.host_words = torch.zeros(WORD_SLOTS, dtype=torch.int32)
        version._host_words_np, version._staging, version._graph = version.host_words.numpy(), {}, notes
        version.input_tensors = [version._tensor(h) for h in version.recording.inputs]
        version.output_tensors = [version._tensor(h) for h in version.recording.outputs]
    assert prompt.hands_over(decode)
    *_, (inputs, words) = model.session.chunk_calls([1, 2, 3])
    prompt.run_and_start(decode, *inputs, **words)
    assert notes.on["own"] == ["held", "graph", "token", "graph"]   # the memory is this stream's too; the portion, its token's way into the words, the step
    notes.stream = "other"
    if use == "a release":
        model.release()
        assert notes.on["host"][-1] == ("behind", "own") and decode._graph is None
        return
    USES[use](model, prompt)
    assert notes.on["other"][:2] == [("behind", "own"), "held"] and notes.on["other"].count(("behind", "own")) == 1
    notes.stream = "own"
    USES[use](model, prompt)
    assert ("behind", "other") in notes.on["own"]
