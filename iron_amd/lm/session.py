"""A conversation's view of a loaded ``CausalLM``: which tokens' keys and values the caches
hold, and how a longer history becomes launches.

The interface is the reference's (iron/lm/session.py:25-229: ``logits``, ``draw``, ``forget``,
``resume``, ``prompt_ids``).  The mechanics are this build's: a history is turned into a short
*plan* of launches -- eager prompt chunks under a row bound, then either one host-started decode
step or a run of replays of the captured step, whose token and position stay on the device -- and
the plan is refused as a whole before its first launch if any of it would leave the caches.
"""

from __future__ import annotations

import dataclasses
from collections.abc import Iterator

import numpy as np

from ..operators.sample import ROW_WORDS


@dataclasses.dataclass(frozen=True)
class ChunkCall:
    """One launch of the prompt version: the padded ids and the per-call words."""

    ids: np.ndarray
    values: dict

    def __iter__(self):
        # Unpacks as ``(inputs, values)``, the shape a version is called with.
        yield (self.ids,)
        yield self.values


def _common_prefix(a: np.ndarray, b: np.ndarray) -> int:
    n = min(a.size, b.size)
    differs = np.flatnonzero(a[:n] != b[:n])
    return int(differs[0]) if differs.size else n


class Session:
    def __init__(self, lm):
        self.lm = lm
        self.cached = np.empty(0, dtype=np.int64)   # tokens whose cache rows are current

    # ------------------------------------------------------------------ what the caches hold
    def _claim(self) -> None:
        """The model's caches serve one session at a time; taking them over empties the view."""
        if self.lm.holder is not self:
            self.lm.holder = self
            self.cached = self.cached[:0]

    def _checked(self, tokens) -> np.ndarray:
        ids = np.asarray(tokens, dtype=np.int64).ravel()
        vocab = self.lm.config.vocab_size
        bad = ids[(ids < 0) | (ids >= vocab)]
        if bad.size:
            raise IndexError(f"tokens {bad} are outside [0, {vocab})")
        return ids

    def _reusable(self, ids: np.ndarray) -> int:
        """Leading tokens of ``ids`` already in the caches.  The last token always runs: its
        logits are what the caller is after."""
        return min(_common_prefix(ids, self.cached), ids.size - 1)

    def forget(self, position: int) -> None:
        """Drop everything from ``position`` on (and, for a ring, back to where it can restart)."""
        keep = min(max(position, 0), self.cached.size)
        self.cached = self.cached[: self.resume(keep)]

    def resume(self, held: int) -> int:
        """Where a run must start so that ``held`` leading tokens stay valid: ``held`` itself unless
        some state cannot be rewound to it (a ring cache restarts at a chunk boundary its rows
        still cover, ``KVCache.restart``)."""
        ran = self.cached.size
        starts = [state.restart(held, ran) for state in self.lm.recurrent]
        return min(starts + [held])

    # ------------------------------------------------------------------ planning
    def prompt_ids(self, tokens) -> np.ndarray:
        """``tokens`` as a prompt launch takes them: ``prefill_chunk`` int32 ids, zero past the last
        (the row bound keeps the padding unread)."""
        chunk = np.zeros(self.lm.config.prefill_chunk, dtype=np.int32)
        piece = np.asarray(tokens).ravel()
        chunk[: piece.size] = piece
        return chunk

    def chunk_calls(self, tokens, start: int = 0) -> list[ChunkCall]:
        """The prompt launches that run ``tokens[start:]``, a chunk each."""
        ids = np.asarray(tokens, dtype=np.int64).ravel()
        width = self.lm.config.prefill_chunk
        calls = []
        for first in range(start, ids.size, width):
            last = min(first + width, ids.size)      # one past the chunk's final token
            words = {"token": int(ids[last - 1]), "position": last - 1, "start": first,
                     "rows": last - first, "rope_start": first}
            calls.append(ChunkCall(self.prompt_ids(ids[first:last]), words))
        return calls

    def _fits(self, count: int, more: int = 0) -> None:
        rows = self.lm.config.max_seq_len
        if count <= 0 or count + more > rows:
            extra = f" and {more + 1} more to draw" if more else ""
            raise ValueError(f"{count} tokens{extra} do not fit {rows} rows")

    # ------------------------------------------------------------------ running
    def logits(self, tokens) -> np.ndarray:
        """The logits after the last of ``tokens`` (the whole history), ``(vocab_size,)``.

        A history one token longer than the cached one is a single decode step; any other runs
        prompt chunks from the first token the caches lack.

        Raises:
            ValueError: no token, or more than ``max_seq_len``.
            IndexError: a token outside the vocabulary (nothing has been launched).
        """
        ids = self._checked(tokens)
        self._fits(ids.size)
        self._claim()
        model = self.lm
        shared = self._reusable(ids)
        if shared == self.cached.size == ids.size - 1:
            row = model.run(token=int(ids[-1]), position=ids.size - 1)
        else:
            begin = self.resume(shared)
            self.cached = ids[:begin]
            row = None
            for inputs, words in self.chunk_calls(ids, begin):
                row = model.run(*inputs, **words)
        self.cached = ids
        # The output buffer is the arena's and the next launch reuses it: hand out a copy, without
        # the columns that only pad an odd vocabulary.
        return np.array(row.numpy()).ravel()[: model.config.vocab_size]

    def draw(self, tokens, max_tokens: int, sampler=None, each: bool = False) -> Iterator[int]:
        """Yield ``max_tokens`` tokens drawn on the device after ``tokens``.

        ``sampler`` (``generation.Sampler``) fixes every draw ahead of time as one row per position;
        without one the draws are greedy.  The first token comes from the prompt's last chunk.  The
        rest are replays of the captured decode step with nothing read back in between (the drawn
        tokens are collected from the device's record afterwards), unless ``each`` asks for every
        token as soon as its step has run, or the step is not captured: then the host starts each
        step from the last one's carried values.

        Between two tokens the model may be called, also by other draws: what that replaced in the
        caches and the draw rows is put back before the next token, and the tokens are the same.

        Raises:
            ValueError: the history and the draws do not fit the caches.
            RuntimeError: the model's versions are not loaded.
        """
        model, ids = self.lm, self._checked(tokens)
        if max_tokens <= 0:
            raise ValueError(f"{ids.size} tokens and {max_tokens} more to draw do not fit {model.config.max_seq_len} rows")
        self._fits(ids.size, max_tokens - 1)
        if model.prompt_chunk is None or model.decode_step is None:
            raise RuntimeError(f"{type(model).__name__}: load_versions() first")
        self._claim()
        prompt_len = ids.size
        table = self._draw_rows(sampler, prompt_len, max_tokens)
        self._stage_draw_rows(table)
        begin = self.resume(self._reusable(ids))
        # Until the run is over nobody knows how far it got (the caller may stop iterating).
        self.cached = self.cached[:0]
        remaining, step = max_tokens - 1, model.decode_step
        *chunks, (inputs, words) = self.chunk_calls(ids, begin)
        for others, at in chunks:
            model.run(*others, **at)
        replayed = bool(remaining) and step.captured and not each
        hands_over = getattr(model.prompt_chunk, "hands_over", None)
        started = replayed and hands_over is not None and hands_over(step)   # (the first step behind the prompt, while its token is on its way here)
        if started:
            carried = model.prompt_chunk.run_and_start(step, *inputs, **words)
        else:
            _, carried = model(*inputs, **words)
        out = [int(carried["token"])]
        ran = model.launched
        yield out[0]
        if replayed and self._interrupted(ran):
            self._regain(ids, [], table)
            step, started, ran = model.decode_step, False, model.launched
            replayed = step.captured
        if replayed:
            if not started:
                step.start(**carried)
            step.replay(remaining - 1)
            record = step.read(model.drawn)       # position p holds the token drawn at p
            ran = model.launched
            for token in record[prompt_len : prompt_len + remaining].tolist():
                out.append(token)
                yield token
        else:
            for _ in range(remaining):
                if self._interrupted(ran):
                    self._regain(ids, out[:-1], table)
                _, carried = model(**carried)
                out.append(int(carried["token"]))
                ran = model.launched
                yield out[-1]
        if not self._interrupted(ran):
            # Every drawn token but the last has been through a step and has its cache rows.
            self.cached = np.concatenate([ids, np.asarray(out[:-1], dtype=np.int64)])

    def _interrupted(self, ran) -> bool:
        """Whether anything of the model ran since ``ran`` was its count of launches."""
        return self.lm.holder is not self or self.lm.launched != ran

    def _regain(self, prompt: np.ndarray, drawn, table) -> None:
        """Draw rows and caches as a draw had them behind ``prompt`` and the ``drawn`` tokens: what another run left of them
        stays, the rest is run again, a prompt's rows by chunks and a drawn token's by its step."""
        model = self.lm
        if model.prompt_chunk is None or model.decode_step is None:
            raise RuntimeError(f"{type(model).__name__}: load_versions() first")
        self._claim()
        self._stage_draw_rows(table)
        ids = np.concatenate([prompt, np.asarray(drawn, dtype=np.int64)])
        begin = self.resume(_common_prefix(ids, self.cached))
        self.cached = self.cached[:0]
        for inputs, words in self.chunk_calls(prompt, begin):
            model.run(*inputs, **words)
        for position in range(max(begin, prompt.size), ids.size):
            model.run(token=int(ids[position]), position=position)

    def _draw_rows(self, sampler, prompt_len: int, count: int) -> np.ndarray | None:
        """The draw rows of ``count`` tokens from position ``prompt_len - 1`` on; none for a greedy run."""
        if sampler is None:
            return None
        table = np.zeros((self.lm.config.max_seq_len, ROW_WORDS), dtype=np.int32)
        table[prompt_len - 1 : prompt_len - 1 + count] = sampler.rows(count, self.lm.k_max)
        return table

    def _stage_draw_rows(self, table: np.ndarray | None) -> None:
        """Write the draw rows; all-zero rows draw greedily.  A greedy run after a greedy run finds
        the table already zero and writes nothing."""
        model = self.lm
        if table is None and not model.sampled:
            return
        model.decode_step.write(model.draws, np.zeros((model.config.max_seq_len, ROW_WORDS), np.int32) if table is None else table)
        model.sampled = table is not None
