"""Soft lookahead on the device against the float64 oracle (relative error
1e-5 with an absolute floor of 1e-5 near 0; -inf pattern exact)."""

from __future__ import annotations

from dataclasses import replace

import numpy as np
import pytest
import torch

from bpdecode_amd import _lib, ops, synth
from bpdecode_amd._lib import check, lib, stream_of
from bpdecode_amd.batch import ConstraintBatch
from bpdecode_amd.ops import FsaTensors
from bpdecode_amd.tokenizer import Vocabulary
from oracle import soft as OS
from tests._util import TOY_PATTERNS, TOY_VOCAB

pytestmark = pytest.mark.gpu

RTOL, ATOL = 1e-5, 1e-5


def close(got: np.ndarray, want: np.ndarray) -> bool:
    inf_ok = np.array_equal(np.isneginf(got), np.isneginf(want))
    fin = np.isfinite(want)
    return inf_ok and bool(np.all(np.abs(got[fin] - want[fin]) <= RTOL * np.abs(want[fin]) + ATOL))


@pytest.mark.parametrize("pattern", TOY_PATTERNS)
@pytest.mark.parametrize("k", [1, 2, 3, 5])
def test_build_lookahead_toy(dev, pattern, k):
    fsa = FsaTensors.build(pattern, TOY_VOCAB).to(dev)
    la = ops.build_lookahead(fsa, k).cpu().numpy()
    want = OS.build_lookahead(fsa.tok_next.cpu().numpy(), fsa.live.cpu().numpy(),
                              fsa.accept.cpu().numpy(), fsa.eos_id, k)
    assert close(la, want)


def test_build_lookahead_email_serving(dev):
    vocab = synth.serving_vocab(151_936, seed=1)
    fsa = FsaTensors.build(synth.EMAIL, vocab).to(dev)
    la = ops.build_lookahead(fsa, 4).cpu().numpy()
    want = OS.build_lookahead(fsa.tok_next.cpu().numpy(), fsa.live.cpu().numpy(),
                              fsa.accept.cpu().numpy(), fsa.eos_id, 4)
    assert close(la, want)


@pytest.mark.parametrize("S,V", [(1, 1), (2, 4097), (63, 4095), (65, 1000), (512, 4097), (513, 4097),
                                 (1, 6144), (2, 6143), (63, 8191), (65, 8193), (512, 6145), (513, 6145)])
@pytest.mark.parametrize("k", [1, 2, 4])
def test_build_lookahead_state_counts(dev, S, V, k):
    """Rounds from (state, next) counts up to 512 states and from 6,144
    tokens on, from the table elsewhere; chunk edges, entries outside the table, states without tokens."""
    g = np.random.default_rng(S + k)
    tn = g.integers(0, S, size=(S, V)).astype(np.int32)
    tn[g.random((S, V)) < 0.9] = -1
    tn[g.random((S, V)) < 0.01] = S + 3  # outside the table: rejected
    tn[S // 2] = -1
    live, accept = (g.random(S) < 0.8).astype(np.uint8), (g.random(S) < 0.3).astype(np.uint8)
    eos = V - 1
    out = torch.empty((S, V), dtype=torch.float32, device=dev)
    need = int(lib().bpd_soft_workspace_bytes(0, S, k))
    ws = torch.empty(need, dtype=torch.uint8, device=dev)
    d = [torch.from_numpy(a).to(dev) for a in (tn, accept, live)]
    want = OS.build_lookahead(np.where(tn < S, tn, -1), live, accept, eos, k)
    for size in (need, 8 * S):  # the two vectors alone: the table-reading rounds
        out.fill_(7.0)
        check(lib().bpd_soft_build_lookahead(d[0].data_ptr(), S, V, d[1].data_ptr(), d[2].data_ptr(), eos, k,
                                             out.data_ptr(), ws.data_ptr(), size, stream_of(dev)))
        assert close(out.cpu().double().numpy(), want)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("alpha", [0.0, 1.0, -0.5, 2.0])
def test_apply_soft(dev, dtype, alpha):
    fsa = FsaTensors.build("a[012]+|b0", TOY_VOCAB).with_lookahead(3).to(dev)
    st = torch.tensor([0, 1, 2, -1, -2, 0], dtype=torch.int32)
    base = torch.randn(6, TOY_VOCAB.size).to(dtype)
    batch = ConstraintBatch(fsa, capacity=6, device=dev)
    for i in range(6):
        batch.add(i)
    batch._state[:6] = st.to(dev)
    got = base.to(dev)
    batch.apply_soft(list(range(6)), got, alpha)
    want = OS.apply_soft(base.float().numpy(), fsa.lookahead.cpu().numpy().astype(np.float64), st.numpy(), alpha)
    host = base.clone()
    ops.apply_soft_(host, fsa.to("cpu"), st, alpha)
    assert torch.equal(got.cpu().view(torch.uint8), host.view(torch.uint8))
    g = got.cpu().float().numpy().astype(np.float64)
    if dtype == torch.float32:
        assert close(g, want)
    else:
        assert np.array_equal(np.isneginf(g), np.isneginf(want))
        fin = np.isfinite(want)
        assert np.all(np.abs(g[fin] - want[fin]) <= 1e-2 * np.abs(want[fin]) + 1e-2)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows,vocab,pad", [(1, 1, 0), (3, 7, 0), (5, 4095, 1), (2, 2049, 3), (9, 8192, 0),
                                            (300, 8193, 5), (300, 16384, 0), (67, 40_001, 8)])
def test_apply_soft_row_shapes(dev, dtype, rows, vocab, pad):
    """Rows of any stride, start alignment and length around the block's
    4096- and 8192-element spans, on the one- and the two-group grid: the
    same words as the library's host entry point.  float16: the device fuses
    the multiply, the add and the conversion (one rounding, where the host
    rounds to float first), so the words are those of the float64 value."""
    g = torch.Generator().manual_seed(rows * 31 + vocab)
    S = 5
    la = torch.randn(S, vocab, generator=g) * 4
    la[torch.rand(S, vocab, generator=g) < 0.8] = -torch.inf
    st = torch.randint(-2, S + 1, (rows,), generator=g, dtype=torch.int32)  # S: out of range, masked
    wide = (torch.randn(rows, vocab + pad, generator=g) * 3).to(dtype)
    got = wide.to(dev)
    off = min(1, pad)
    ops.soft_apply_(got[:, off:off + vocab], la.to(dev), st.to(dev), alpha=0.75)
    want = wide.clone()
    ops.soft_apply_(want[:, off:off + vocab], la, st.where(st < S, -1), alpha=0.75)
    if dtype == torch.float16:
        bias = la.double()[st.clamp(0, S - 1).long()].numpy()
        v = wide[:, off:off + vocab].double().numpy() + 0.75 * bias
        keep = np.isfinite(want[:, off:off + vocab].float().numpy())
        want[:, off:off + vocab] = torch.from_numpy(np.where(keep, v, -np.inf).astype(np.float16))
    assert torch.equal(got.cpu().view(torch.uint8), want.view(torch.uint8))


def test_apply_soft_carries_queued_writes(dev):
    """add / evict / reset before apply_soft: the mask launch applies them,
    and the pool holds them for the next commit."""
    fsa = FsaTensors.build("a[012]+|b0", TOY_VOCAB).with_lookahead(3).to(dev)
    batch = ConstraintBatch(fsa, capacity=8, device=dev)
    for i in range(6):
        batch.add(i)
    tok = TOY_VOCAB.token_bytes.index(b"a")
    batch.commit(list(range(6)), torch.full((6,), tok, dtype=torch.int64, device=dev))
    batch.evict(1)
    batch.evict(4)
    batch.add(7)
    batch.reset(2)
    ids = [7, 0, 2, 3, 5]
    after = int(fsa.tok_next[fsa.start, tok])
    states = [fsa.start, after, fsa.start, after, after]
    x = torch.randn(5, TOY_VOCAB.size)
    got = x.to(dev)
    batch.apply_soft(ids, got, 0.5)
    want = x.clone()
    ops.apply_soft_(want, fsa.to("cpu"), torch.tensor(states, dtype=torch.int32), 0.5)
    assert torch.equal(got.cpu(), want)
    assert [batch.state_of(i) for i in ids] == states
    nxt = batch.commit(ids, torch.full((5,), tok, dtype=torch.int64, device=dev)).tolist()
    assert nxt == [int(fsa.tok_next[s, tok]) if s >= 0 else -1 for s in states]


@pytest.mark.parametrize("rows", [1, 9])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_apply_soft_of_an_empty_vocabulary_makes_queued_writes(dev, rows, dtype):
    """No logits to change, but the pool writes that travel with the call are
    made."""
    pool = torch.arange(12, dtype=torch.int32, device=dev)
    la = torch.empty(3, 0, device=dev)
    x = torch.empty(rows, 0, dtype=dtype, device=dev)
    slots = torch.arange(rows, dtype=torch.int64, device=dev)
    pending = torch.tensor([2, 7, 11, 1, -1, 2], dtype=torch.int64, device=dev)  # three slots, three values
    code = {torch.float32: _lib.DTYPE_F32, torch.bfloat16: _lib.DTYPE_BF16}[dtype]
    want = pool.clone()
    for n in (0, 3):
        check(lib().bpd_soft_apply_queued(x.data_ptr(), code, rows, 0, 0, la.data_ptr(), 3, pool.data_ptr(),
                                          slots.data_ptr(), pending.data_ptr(), n, 0.5, None, stream_of(dev)))
        if n:
            want[pending[:3]] = pending[3:].to(torch.int32)
        assert torch.equal(pool, want), n


@pytest.mark.parametrize("vocab", ["v17", "v20"])
@pytest.mark.parametrize("stats", ["list", "wave", "members", "classes", "pieces"])
def test_prior_carries_queued_writes(dev, vocab, stats, monkeypatch):
    """add / evict / reset before apply_soft_prior: its first launch makes
    them, its rows read them, and the pool holds them for the next commit."""
    if stats == "pieces":
        monkeypatch.setenv("BPD_SOFT_PRIOR_PIECES", "1")
    else:
        monkeypatch.setenv("BPD_SOFT_STATS", stats)
    voc = TOY_VOCAB if vocab == "v17" else TOY_VOCAB20
    fsa = FsaTensors.build("a[012]+|b0", voc).densify().to(dev)
    batch = ConstraintBatch(fsa, capacity=300, device=dev)
    ids = list(range(290))
    for i in ids:
        batch.add(i)
    tok = voc.token_bytes.index(b"a")
    batch.commit(ids, torch.full((290,), tok, dtype=torch.int64, device=dev))
    after = int(fsa.tok_next[fsa.start, tok])
    states = [after] * 290
    # 14 fit a launch's arguments, 15 and 250 one upload, 290 are flushed first
    for queued in (3, 14, 15, 250, 290):
        for i in range(queued):
            batch.reset(ids[i])
        states[:queued] = [fsa.start] * queued
        batch.evict(ids[-1])
        batch.add(("new", queued))
        ids[-1], states[-1] = ("new", queued), fsa.start
        x = torch.randn(290, voc.size, generator=torch.Generator().manual_seed(queued)) * 3
        got = x.to(dev)
        batch.apply_soft_prior(ids, got, 3, 0.5)
        want = x.clone()
        ops.apply_soft_prior_(want, fsa.to("cpu"), torch.tensor(states, dtype=torch.int32), 3, 0.5)
        assert torch.equal(torch.isneginf(got.cpu()), torch.isneginf(want))
        assert torch.allclose(got.cpu(), want, rtol=1e-5, atol=1e-5)
        states = batch.commit(ids, torch.full((290,), tok, dtype=torch.int64, device=dev)).tolist()
        assert states == [batch.state_of(i) for i in ids]
        batch.commit(ids, torch.full((290,), voc.token_bytes.index(b"0"), dtype=torch.int64, device=dev))
        states = [int(fsa.tok_next[s, voc.token_bytes.index(b"0")]) if s >= 0 else -1 for s in states]


# ------------------------------------------------------- prior-weighted --
# The toy vocabulary with three more tokens: V = 20, a multiple of 4, so the
# vectorised kernels apply (V = 17 takes the scalar ones).
TOY_VOCAB20 = Vocabulary.from_tokens(list(TOY_VOCAB.token_bytes) + [b"d", b"e0", b"bb"],
                                     eos_id=TOY_VOCAB.eos_id)


@pytest.mark.parametrize("pattern", TOY_PATTERNS)
@pytest.mark.parametrize("k", [1, 2, 4])
@pytest.mark.parametrize("alpha", [0.0, 1.0, -0.5])
@pytest.mark.parametrize("vocab", ["v17", "v20"])
def test_prior_toy(dev, pattern, k, alpha, vocab):
    fsa = FsaTensors.build(pattern, TOY_VOCAB if vocab == "v17" else TOY_VOCAB20).densify()
    S, V = fsa.tok_next.shape
    st = torch.tensor(list(range(S)) + [-1, 0], dtype=torch.int32)
    g = torch.Generator().manual_seed(k * 13 + len(pattern))
    x = torch.randn(len(st), V, generator=g) * 3
    got = x.to(dev)
    ops.apply_soft_prior_(got, fsa.to(dev), st.to(dev), k, alpha)
    want = OS.prior_lookahead(x.double().numpy(), fsa.tok_next.numpy(), fsa.live.numpy(),
                              fsa.accept.numpy(), fsa.eos_id, st.numpy(), k, alpha)
    assert close(got.cpu().double().numpy(), want)


@pytest.mark.parametrize("vocab", ["v17", "v20"])
def test_prior_batch_slots_and_errors(dev, vocab):
    fsa = FsaTensors.build("a[012]+|b0", TOY_VOCAB if vocab == "v17" else TOY_VOCAB20).densify().to(dev)
    S, V = fsa.tok_next.shape
    batch = ConstraintBatch(fsa, capacity=8, device=dev)
    for i in range(6):
        batch.add(i)
    pool = torch.tensor([0, 1, 2, -1, 0, 2, -2, -2], dtype=torch.int32)
    batch._state[:] = pool.to(dev)
    ids = [4, 2, 0, 3, 1]
    x = torch.randn(5, V) * 3
    got = x.to(dev)
    batch.apply_soft_prior(ids, got, k=3, alpha=0.5)
    want = OS.prior_lookahead(x.double().numpy(), fsa.tok_next.cpu().numpy(), fsa.live.cpu().numpy(),
                              fsa.accept.cpu().numpy(), fsa.eos_id, pool[ids].numpy(), 3, 0.5)
    assert close(got.cpu().double().numpy(), want)
    batch.check_errors()
    batch._state[0] = S  # out-of-range state: -inf row and the device error flag
    got = x.to(dev)
    batch.apply_soft_prior([0], got[:1], k=3, alpha=0.5)
    assert torch.isneginf(got[0]).all()
    with pytest.raises(IndexError):
        batch.check_errors()


def test_prior_unaligned_vocab(dev):
    # V = 17 (not a multiple of 4) and a strided row view take the scalar kernels
    fsa = FsaTensors.build("[a-c]*", TOY_VOCAB).densify()
    S, V = fsa.tok_next.shape
    wide = torch.randn(4, V + 3, generator=torch.Generator().manual_seed(17)) * 3
    st = torch.tensor([0, 0, -1, 0], dtype=torch.int32)
    want = OS.prior_lookahead(wide[:, :V].double().numpy(), fsa.tok_next.numpy(), fsa.live.numpy(),
                              fsa.accept.numpy(), fsa.eos_id, st.numpy(), 4, 1.0)
    w = wide.to(dev)
    ops.apply_soft_prior_(w[:, :V], fsa.to(dev), st.to(dev), 4, 1.0)
    assert close(w[:, :V].cpu().double().numpy(), want)
    assert torch.equal(w[:, V:].cpu(), wide[:, V:])


@pytest.mark.parametrize("rows,vocab,pad,offset", [
    (1, 4095, 0, 0), (3, 4096, 1, 1), (2, 4097, 2, 3), (5, 8191, 0, 2), (1, 8193, 3, 0), (600, 4099, 0, 0),
    (60, 20_003, 1, 3), (256, 8100, 0, 1), (257, 4095, 0, 0),
])
@pytest.mark.parametrize("eos", [0, 4094, -1])
def test_prior_row_shapes(dev, rows, vocab, pad, offset, eos):
    """Member-list kernels at the edges of their chunks (4096 tokens a stage,
    8192 a statistics block), at every alignment of the rows, with more rows
    than blocks in flight, chunks that the blocks of a row share unevenly and
    rows at and above the CUs; nothing outside the rows' columns is written."""
    S, C = 6, 9
    rng = np.random.default_rng(vocab + rows)
    columns = rng.integers(-1, S, size=(S, C + 1))
    columns[:, C] = -1  # tokens rejected everywhere: most of them, at most 1024 a chunk are not
    tn = columns[:, np.where(rng.random(vocab) < 0.1, rng.integers(0, C, size=vocab), C)]
    tn[:, eos] = np.where(np.arange(S) % 2 == 0, np.arange(S), -1)
    fsa = FsaTensors.build("a", TOY_VOCAB).densify()
    fsa = replace(fsa, tok_next=torch.from_numpy(tn).to(torch.int32), trans=torch.zeros(S, dtype=torch.int32),
                  accept=(torch.arange(S) % 2 == 0).to(torch.uint8), live=torch.ones(S, dtype=torch.uint8),
                  num_symbols=1, eos_id=eos % vocab, allow_bits=None, soft_classes=None)
    st = torch.from_numpy(rng.integers(-1, S, size=rows)).to(torch.int32)
    flat = torch.randn(offset + rows * (vocab + pad), generator=torch.Generator().manual_seed(rows)) * 3
    flat[rng.random(flat.numel()) < 0.01] = -float("inf")
    view = flat[offset:].view(rows, vocab + pad)[:, :vocab]
    want = OS.prior_lookahead(view.double().numpy(), tn, np.ones(S, dtype=np.uint8), np.arange(S) % 2 == 0,
                              eos % vocab, st.numpy(), 3, 0.5)
    got = flat.to(dev)
    fd = fsa.to(dev)
    assert fd.ensure_soft_classes().chunk_cap > 0
    out = got[offset:].view(rows, vocab + pad)[:, :vocab]
    ops.apply_soft_prior_(out, fd, st.to(dev), 3, 0.5)
    assert close(out.cpu().double().numpy(), want)
    view.copy_(out.cpu())
    assert torch.equal(got.cpu(), flat)


@pytest.fixture(scope="module")
def email_serving():
    """B=128, V=151,936, k=4 over the email DFA, logits N(0, 3),
    rows at random reachable states; the float64 oracle of every row,
    computed once with the rows split over host threads (numpy releases the
    interpreter lock in its array loops)."""
    from concurrent.futures import ThreadPoolExecutor

    vocab = synth.serving_vocab(151_936, seed=1)
    fsa = FsaTensors.build(synth.EMAIL, vocab).densify()
    tn = fsa.tok_next.numpy()
    st = synth.random_walk_states(fsa.tok_next, fsa.start, fsa.eos_id, 128, 40, seed=5).to(torch.int32)
    x = synth.logits(128, tn.shape[1], std=3.0, dtype=torch.float32, seed=11)
    xd = x.double().numpy()
    live, acc, stn = fsa.live.numpy(), fsa.accept.numpy(), st.numpy()
    with ThreadPoolExecutor(16) as ex:
        rows = list(ex.map(lambda b: OS.prior_lookahead(xd[b:b + 1], tn, live, acc, fsa.eos_id,
                                                         stn[b:b + 1], 4, 1.0), range(128)))
    return fsa, st, x, np.concatenate(rows)


@pytest.mark.parametrize("stats", ["list", "wave", "members", "classes"])
def test_prior_email_serving(dev, stats, monkeypatch, email_serving):
    """B=128, V=151,936, k=4 over the email DFA: every row against the
    float64 oracle and against the alpha-free identity (alpha = 0 leaves
    log_softmax on tokens whose k-1 lookahead is finite); class statistics
    with wave shifts over 8192-token chunks from the chunk member lists (and
    the member-list output pass) or from the class map, and over
    4096-token chunks from the member lists and from the class map."""
    monkeypatch.setenv("BPD_SOFT_STATS", stats)
    fsa, st, x, want = email_serving
    fd = fsa.to(dev)
    assert fd.ensure_soft_classes().chunk_cap in (256, 512, 1024)
    got = x.to(dev)
    ops.apply_soft_prior_(got, fd, st.to(dev), 4, 1.0)
    got = got.cpu().double().numpy()
    assert close(got, want)
    zero = x.to(dev)
    ops.apply_soft_prior_(zero, fd, st.to(dev), 4, 0.0)
    ls = torch.log_softmax(x.double(), dim=1).numpy()
    fin = np.isfinite(got)
    assert np.array_equal(np.isfinite(zero.cpu().numpy()), fin)
    z = zero.cpu().double().numpy()
    assert np.all(np.abs(z[fin] - ls[fin]) <= RTOL * np.abs(ls[fin]) + ATOL)


@pytest.mark.parametrize("pattern", ["a[012]+|b0", "[a-c]*"])
def test_prior_pieces_path(dev, pattern, monkeypatch):
    """The gather-over-class-pieces statistics (taken above 1024 token
    classes; forced here) give the same results."""
    monkeypatch.setenv("BPD_SOFT_PRIOR_PIECES", "1")
    fsa = FsaTensors.build(pattern, TOY_VOCAB).densify()
    S, V = fsa.tok_next.shape
    st = torch.tensor(list(range(S)) + [-1], dtype=torch.int32)
    x = torch.randn(len(st), V) * 3
    got = x.to(dev)
    ops.apply_soft_prior_(got, fsa.to(dev), st.to(dev), 4, 0.7)
    want = OS.prior_lookahead(x.double().numpy(), fsa.tok_next.numpy(), fsa.live.numpy(),
                              fsa.accept.numpy(), fsa.eos_id, st.numpy(), 4, 0.7)
    assert close(got.cpu().double().numpy(), want)


def test_prior_pieces_path_email(dev, monkeypatch):
    vocab = synth.serving_vocab(151_936, seed=1)
    fsa = FsaTensors.build(synth.EMAIL, vocab).densify()
    st = synth.random_walk_states(fsa.tok_next, fsa.start, fsa.eos_id, 16, 40, seed=9).to(torch.int32)
    x = synth.logits(16, 151_936, std=3.0, dtype=torch.float32, seed=12)
    fd = fsa.to(dev)
    a = x.to(dev)
    ops.apply_soft_prior_(a, fd, st.to(dev), 4, 1.0)
    monkeypatch.setenv("BPD_SOFT_PRIOR_PIECES", "1")
    b = x.to(dev)
    ops.apply_soft_prior_(b, fd, st.to(dev), 4, 1.0)
    a, b = a.cpu().double().numpy(), b.cpu().double().numpy()
    assert close(b, a)


@pytest.mark.parametrize("vocab", ["v17", "v20"])
def test_prior_wide_class_map_and_extreme_logits(dev, monkeypatch, vocab):
    """Every statistics path gives the oracle's results: wave shifts over the
    member lists (with the member-list output pass) and over the uint16
    class map (the -1e4 logits sit far below their wave's maximum, so those
    blocks take the exact per-class maximum), the 4096-token chunk member
    lists, the uint16 class map and the int32 one.  Rows mixing -inf, very negative
    and large logits keep every class sum exact."""
    fsa = FsaTensors.build("-?[0-9]+(\\.[0-9]+)?", TOY_VOCAB if vocab == "v17" else TOY_VOCAB20).densify()
    S, V = fsa.tok_next.shape
    st = torch.tensor(list(range(S)) * 2, dtype=torch.int32)
    g = torch.Generator().manual_seed(3)
    x = torch.randn(len(st), V, generator=g) * 3
    x[1::2, ::3] = -1.0e4
    x[2::4, 1::5] = float("-inf")
    x[3::4, 2] = 60.0
    want = OS.prior_lookahead(x.double().numpy(), fsa.tok_next.numpy(), fsa.live.numpy(),
                              fsa.accept.numpy(), fsa.eos_id, st.numpy(), 4, 0.8)
    fd = fsa.to(dev)
    sc = fd.ensure_soft_classes()
    assert sc.token_class16 is not None
    a = x.to(dev)
    ops.apply_soft_prior_(a, fd, st.to(dev), 4, 0.8)
    assert close(a.cpu().double().numpy(), want)
    for stats in ("wave", "members", "classes"):
        monkeypatch.setenv("BPD_SOFT_STATS", stats)
        m = x.to(dev)
        ops.apply_soft_prior_(m, fd, st.to(dev), 4, 0.8)
        assert close(m.cpu().double().numpy(), want), stats
    monkeypatch.setenv("BPD_SOFT_STATS", "classes")
    sc.token_class16, sc._c = None, None
    b = x.to(dev)
    ops.apply_soft_prior_(b, fd, st.to(dev), 4, 0.8)
    assert close(b.cpu().double().numpy(), want)


@pytest.mark.parametrize("pattern", ["[a-c]*", "a[012]+|b0"])
@pytest.mark.parametrize("vocab", ["v17", "v20"])
def test_prior_error_stays_near_float32_rounding(dev, pattern, vocab):
    """Across seeded draws the device result stays at float32 rounding level
    of the float64 oracle at k = 4: within 2e-6 + 2e-7 * max|x| per row (the
    exponentials take x - max before scaling, so a large row maximum costs
    no precision beyond the rounding of the inputs themselves)."""
    fsa = FsaTensors.build(pattern, TOY_VOCAB if vocab == "v17" else TOY_VOCAB20).densify()
    S, V = fsa.tok_next.shape
    fd = fsa.to(dev)
    g = torch.Generator().manual_seed(23)
    worst = 0.0
    for _ in range(12):
        x = torch.randn(6, V, generator=g) * 3 + 20.0 * torch.rand(1, generator=g)
        st = torch.tensor([min(i, S - 1) for i in range(5)] + [-1], dtype=torch.int32)
        want = OS.prior_lookahead(x.double().numpy(), fsa.tok_next.numpy(), fsa.live.numpy(),
                                  fsa.accept.numpy(), fsa.eos_id, st.numpy(), 4, 1.0)
        got = x.to(dev)
        ops.apply_soft_prior_(got, fd, st.to(dev), 4, 1.0)
        got = got.cpu().double().numpy()
        assert np.array_equal(np.isneginf(got), np.isneginf(want))
        tol = 2e-6 + 2e-7 * x.abs().amax(dim=1, keepdim=True).double().numpy()
        fin = np.isfinite(want)
        err = np.zeros_like(want)
        err[fin] = np.abs(got[fin] - want[fin])
        worst = max(worst, float((err / tol).max()))
    assert worst <= 1.0, worst
