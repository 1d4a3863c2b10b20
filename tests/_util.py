"""Shared helpers of the test-suite (not a test module)."""

from __future__ import annotations

import numpy as np
import torch

from bpdecode_amd.grammar.ir import Alt, CharSet, Concat, Empty, Opt, Plus, Ref
from bpdecode_amd.ops import FsaTensors
from bpdecode_amd.tokenizer import Vocabulary
from oracle import dense as OD

TOY_VOCAB = Vocabulary.from_tokens(
    ["a", "b", "c", "ab", "ba", "0", "1", "12", "-", ".", "aa", "", "caf", "\xc3", "\xe9", "é", "<eos>"],
    eos_id=16,
)
TOY_PATTERNS = ["[01]+", "a+b*", "(ab)+", "-?[0-9]+(\\.[0-9]+)?", "a|bc|12", "[a-c]*", "caf(e|é)"]

PDA_VOCAB = Vocabulary.from_tokens(
    ["(", ")", "x", "y", "{", "}", "a", "b", ":", "0", "1", ",", "<eos>", "((", "x)", "", "{a", ":0,",
     "\"", "[1", "[", "]", "tr", "ue", "nul", "l", "-", "2.5", "e9", " ", "\"ab\"", "\\n"],
    eos_id=12,
)


def oracle_table(fsa: FsaTensors) -> np.ndarray:
    """tok_next from the oracle's restatement of build_token_transitions."""
    return OD.build_token_transitions(
        fsa.trans.cpu().numpy(), fsa.accept.cpu().numpy(), fsa.live.cpu().numpy(), fsa.num_symbols,
        fsa.offsets.cpu().numpy(), fsa.symbols.cpu().numpy(), fsa.eos_id,
    )


def bits_of(t: torch.Tensor) -> np.ndarray:
    return t.cpu().contiguous().view(torch.int16 if t.element_size() == 2 else torch.int32).numpy().copy()


class OracleWalk:
    """One sequence walked through the oracle's tok_next table of a regex
    bundle: the allowed token ids, the commit, and completeness (EOS
    allowed)."""

    def __init__(self, fsa: FsaTensors) -> None:
        self.fsa = fsa
        self.rows: dict[int, np.ndarray] = {}  # oracle tok_next rows, built as states are met
        self.accept = fsa.accept.cpu().numpy().astype(bool)
        self.state = fsa.start

    def _row(self, s: int) -> np.ndarray:
        if s not in self.rows:
            f = self.fsa
            self.rows[s] = OD.build_token_transitions(
                f.trans.cpu().numpy(), f.accept.cpu().numpy(), f.live.cpu().numpy(), f.num_symbols,
                f.offsets.cpu().numpy(), f.symbols.cpu().numpy(), f.eos_id, rows=[s])[0]
        return self.rows[s]

    def allowed(self) -> set[int]:
        if self.state < 0:
            return set()
        return set(np.nonzero(self._row(self.state) != -1)[0].tolist())

    def advance(self, token: int) -> None:
        if self.state >= 0:
            self.state = int(OD.advance(self._row(self.state)[None], [0], [token])[0])

    def is_complete(self) -> bool:
        return self.state >= 0 and bool(self.accept[self.state])


def random_bundle(S: int, M: int, V: int, seed: int, max_len: int = 40) -> FsaTensors:
    """A bundle of arbitrary tables: targets outside the table, symbol ids at
    and above M, empty tokens, tokens longer than 16 symbols, EOS inside the
    vocabulary and a live set that need not be closed (``dead`` live in half
    of them)."""
    g = np.random.default_rng(seed)
    trans = g.integers(-2, S + 2, size=S * M).astype(np.int32)
    keep = g.random(S * M) < 0.9
    trans[keep] = g.integers(0, S, size=int(keep.sum()))
    dead = int(g.integers(0, S))
    live = (g.random(S) < 0.7).astype(np.uint8)
    live[dead] = seed % 2
    lens = g.integers(0, max_len + 1, size=V)
    lens[g.random(V) < 0.7] //= 8
    off = np.zeros(V + 1, dtype=np.int32)
    np.cumsum(lens, out=off[1:])
    sym = g.integers(0, M, size=int(off[-1]))
    bad = g.random(sym.size) < 0.01
    sym[bad] = np.minimum(M + g.integers(0, 4, size=int(bad.sum())), 255)
    t = torch.from_numpy
    return FsaTensors(trans=t(trans), accept=t((g.random(S) < 0.3).astype(np.uint8)), live=t(live), num_symbols=M,
                      dead=dead, offsets=t(off), symbols=t(sym.astype(np.int32)), eos_id=int(g.integers(0, V)))


def walked_allowed(fsa: FsaTensors, states) -> np.ndarray:
    """[rows, vocab]: the tokens that mask.hpp's walk allows from each state,
    restated in numpy for arbitrary tables: a walk fails on a symbol id at or
    above ``num_symbols``, on a target outside the table and on a step into
    ``dead``, and must end on a live state; EOS where the state accepts;
    nothing from a state below 0 or past the table."""
    S, M, V = fsa.num_states, fsa.num_symbols, fsa.vocab_size
    trans, live, accept, off, sym = (t.cpu().numpy().astype(np.int64) for t in
                                     (fsa.trans, fsa.live, fsa.accept, fsa.offsets, fsa.symbols))
    st = np.asarray(states, dtype=np.int64)
    inside = (st >= 0) & (st < S)
    cur = np.repeat(np.where(inside, st, -1)[:, None], V, axis=1)
    lens = off[1:] - off[:-1]
    for k in range(int(lens.max())):
        t = np.nonzero(lens > k)[0]
        c, at = sym[off[t] + k], cur[:, t]
        nxt = trans[np.clip(at, 0, None) * M + np.minimum(c, M - 1)[None, :]]
        ok = (at >= 0) & (c < M)[None, :] & (nxt >= 0) & (nxt < S) & (nxt != fsa.dead)
        cur[:, t] = np.where(ok, nxt, -1)
    allowed = (cur >= 0) & (live[np.clip(cur, 0, None)] != 0)
    if fsa.eos_id is not None and 0 <= fsa.eos_id < V:
        allowed[:, fsa.eos_id] = inside & (accept[np.clip(st, 0, S - 1)] != 0)
    return allowed


def reachable(tok_next: np.ndarray, start: int) -> list[int]:
    seen, todo = {start}, [start]
    while todo:
        for d in np.unique(tok_next[todo.pop()]):
            if d >= 0 and int(d) not in seen:
                seen.add(int(d))
                todo.append(int(d))
    return sorted(seen)


def member(grammar, text):
    """Is ``text`` in the language of ``grammar``?  An independent recursive
    matcher over the grammar IR (no NFA, no PDA): the set of end positions."""
    rules = grammar.rules
    busy = set()

    def m(e, pos):
        if isinstance(e, Empty):
            return {pos}
        if isinstance(e, CharSet):
            return {pos + 1} if pos < len(text) and e.matches(ord(text[pos])) else set()
        if isinstance(e, Ref):
            key = (e.name, pos)
            if key in busy:
                return set()
            busy.add(key)
            try:
                return m(rules[e.name], pos)
            finally:
                busy.discard(key)
        if isinstance(e, Concat):
            cur = {pos}
            for p in e.parts:
                cur = set().union(*(m(p, q) for q in cur)) if cur else set()
            return cur
        if isinstance(e, Alt):
            return set().union(*(m(o, pos) for o in e.options))
        if isinstance(e, Opt):
            return {pos} | m(e.node, pos)
        reached = set() if isinstance(e, Plus) else {pos}
        frontier = {pos}
        while frontier:
            nxt = set()
            for p in frontier:
                for q in m(e.node, p):
                    if q not in reached:
                        reached.add(q)
                        nxt.add(q)
            frontier = nxt
        return reached

    return len(text) in m(rules[grammar.root], 0)
