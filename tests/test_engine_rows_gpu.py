"""Logits rows of an engine step in the caller's memory.  They go to pageable memory through
the engine's ring of eight pinned pieces of 1 MiB, to memory that the runtime knows by its
copy.  Both hold the same bytes."""
import ctypes

import numpy as np
import pytest

import _layer_stack as T

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def eng(gpu, tmp_path_factory):
    import engine
    cfg = T.config([(T.attn(), None)], vocab=5003)
    folder = T.save(tmp_path_factory.mktemp("model"), cfg, T.weights(cfg, 3))
    with engine.Engine(folder, dtype="float32", max_seqs=4, max_tokens=1024,
                       max_step_tokens=128) as e:
        yield e


def step(eng, entries, out):
    from llm_capi import EngineEntry
    arr, keep = (EngineEntry * len(entries))(), []
    for i, (seq, tok, want) in enumerate(entries):
        t, w = np.asarray(tok, np.int32), np.asarray(want, np.int32)
        keep.append((t, w))
        arr[i] = EngineEntry(seq, t.ctypes.data, t.size, w.ctypes.data, w.size)
    eng._check(eng.lib.llm_engine_step(eng._h, arr, len(entries), ctypes.c_void_p(out)))


def check(eng, lens, pick):
    import torch
    rng = np.random.default_rng(len(lens) + lens[0])
    toks = [rng.integers(0, eng.vocab, n) for n in lens]
    wants = [{None: list(range(n)), "odd": list(range(1, n, 2)), "back": list(range(n))[::-1],
              "none": []}[pick] for n in lens]
    rows = sum(map(len, wants))
    pinned = torch.full((max(rows, 1), eng.vocab), -7.0, pin_memory=True)
    plain = np.full((max(rows, 1), eng.vocab), 7.0, np.float32)
    for out in (pinned.data_ptr(), plain.ctypes.data):
        seqs = [eng.open_seq() for _ in lens]
        step(eng, [(s, t, w) for s, t, w in zip(seqs, toks, wants)], out)
        for s in seqs:
            eng.close_seq(s)
    if rows:
        np.testing.assert_array_equal(plain, pinned.numpy())


# rows of 20,012 bytes: one; 52 and 53: the last in one piece and the first in two; 105 and
# 128: three pieces; 127 in gaps, and a batch of two passes whose rows lie apart
@pytest.mark.parametrize("lens,pick", [
    ([1], None), ([26], None), ([52], None), ([53], None), ([105], None), ([128], None),
    ([60, 67], "odd"), ([100, 90], "back"), ([3], "none"),
])
def test_rows_by_both_ways(eng, lens, pick):
    check(eng, lens, pick)


@pytest.fixture(scope="module")
def wide(gpu, tmp_path_factory):
    import engine
    cfg = T.config([(T.attn(), None)], vocab=40009)
    folder = T.save(tmp_path_factory.mktemp("wide"), cfg, T.weights(cfg, 4))
    with engine.Engine(folder, dtype="float32", max_seqs=4, max_tokens=1024,
                       max_step_tokens=128) as e:
        yield e


# rows of 160,036 bytes: 6 and 7 on both sides of a piece; 52 just fill the ring's 8 MiB, 53
# use a piece again, 105 (over 16 MiB) and 128 a piece for the third time; in gaps and back
# to front, and 190 rows of two passes
@pytest.mark.parametrize("lens,pick", [
    ([6], None), ([7], None), ([52], None), ([53], None), ([105], None), ([128], None),
    ([64, 64], "odd"), ([70, 58], "back"), ([100, 90], "back"), ([100, 90], None),
])
def test_pieces_used_again(wide, lens, pick):
    check(wide, lens, pick)


@pytest.mark.parametrize("tokens,want", [
    (np.array([5, 6, 7], np.int32), [2, 0]), ([5, 6, 7], (1,)), ((5, 6, 7), range(3)),
    (np.array([5, 9, 6, 9, 7, 9], np.int32)[::2], np.array([[1], [2]])),
    (np.array([5, 6, 7]), np.array([0, 2], np.int32)), (np.array([5.0, 6.0, 7.0]), []),
    ([np.int64(5), 6, 7], [True])])
def test_entries_of_every_kind(eng, tokens, want):
    """Entries that the native way takes and those it leaves to the general one."""
    def run(entries):
        s = eng.open_seq()
        try:
            return eng.step([(s, *entries)])
        finally:
            eng.close_seq(s)
    places = [int(p) for p in np.asarray(want, np.int32).reshape(-1)]
    all_rows = run((np.array([5, 6, 7], np.int32), np.array([0, 1, 2], np.int32)))
    got = run((tokens, want))
    assert got.shape == (len(places), eng.vocab) and got.dtype == np.float32
    np.testing.assert_array_equal(got, all_rows[places])


@pytest.mark.parametrize("bad", [([5], [1]), ([1 << 20], [0]), ([], []), ([5], [-1])])
def test_refused_entries(eng, bad):
    s = eng.open_seq()
    with pytest.raises(Exception, match="engine step"):
        eng.step([(s, *bad)])
    assert eng.seq_len(s) == 0
    eng.close_seq(s)
    with pytest.raises(Exception, match="not open"):
        eng.step([(s, [5], [0])])


def test_without_the_extension_module(eng, tmp_path, monkeypatch):
    """The C library alone, or a module built for another Python: steps go the general way."""
    import sys

    import engine
    import llm_capi
    cfg = T.config([(T.attn(), None)], vocab=5003)
    T.save(tmp_path / "m", cfg, T.weights(cfg, 3))

    def step(e):
        seq = e.open_seq()
        out = e.step([(seq, np.array([5, 6, 7], np.int32), [0, 2])])
        e.close_seq(seq)
        return out
    want = step(eng)
    with engine.Engine(tmp_path / "m", dtype="float32", max_tokens=256, lib=llm_capi.load()) as e:
        assert e._native_step  # the default library, named or not
        np.testing.assert_array_equal(step(e), want)
    monkeypatch.setitem(sys.modules, "llm_decoder", None)
    with engine.Engine(tmp_path / "m", dtype="float32", max_tokens=256) as e:
        assert not e._native_step
        np.testing.assert_array_equal(step(e), want)


def test_returned_rows_stay(gpu, tmp_path):
    """Arrays of one step stay as they are through the next ones, past the 64 MiB that are pinned
    at most, and past the engine; from several threads at once."""
    import threading
    import engine
    cfg = T.config([(T.attn(), None)], vocab=5003)
    folder = T.save(tmp_path, cfg, T.weights(cfg, 3))
    held, lock = [], threading.Lock()

    def serve(seed):
        rng = np.random.default_rng(seed)
        with engine.Engine(folder, dtype="float32", max_seqs=2, max_tokens=512) as e:
            for n in [3, 4] + [200] * 12:  # 60,036 and 80,048 bytes; 4.0 MB
                s = e.open_seq()
                toks = rng.integers(0, e.vocab, n)
                out = e.step([(s, toks, list(range(n)))])
                e.close_seq(s)
                plain = np.empty_like(out)
                s = e.open_seq()
                step(e, [(s, toks, list(range(n)))], plain.ctypes.data)
                e.close_seq(s)
                with lock:
                    held.append((out, plain))

    threads = [threading.Thread(target=serve, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert len(held) == 28
    for out, plain in held:
        assert out.flags.writeable and out.flags.c_contiguous
        np.testing.assert_array_equal(out, plain)


@pytest.mark.parametrize("dtype", ["bfloat16", "float32"])
@pytest.mark.parametrize("vocab", [5003, 40000])
@pytest.mark.parametrize("rows", [1, 9, 16, 17, 33])
def test_decode_rows_in_turns(gpu, tmp_path, rows, vocab, dtype):
    """One captured step whose rows go to pinned memory, to pageable memory and to a buffer
    that begins at any float, in turns: the same bytes; nothing behind the rows is written."""
    import engine
    import torch
    cfg = T.config([(T.attn(), None)], vocab=vocab)
    folder = T.save(tmp_path, cfg, T.weights(cfg, 3))
    n = rows * vocab
    with engine.Engine(folder, dtype=dtype, max_seqs=2 * rows, max_tokens=32 * 2 * rows) as e:
        rng = np.random.default_rng(rows)
        toks = rng.integers(0, vocab, (6, rows))
        plain, pinned = np.empty(n, np.float32), torch.empty(n + 8, pin_memory=True)
        want = []
        for places in ["plain"] * 6, ["aligned", "plain", "odd", "aligned", "plain", "odd"]:
            seqs = [e.open_seq() for _ in range(rows)]
            for i, place in enumerate(places):
                pinned.fill_(-7.0)
                at = {"aligned": 0, "odd": 3}.get(place)
                out = plain.ctypes.data if at is None else pinned.data_ptr() + 4 * at
                step(e, [(s, [t], [0]) for s, t in zip(seqs, toks[i])], out)
                got = (plain if at is None else pinned.numpy()[at:at + n]).copy()
                if len(want) < 6:
                    want.append(got)
                np.testing.assert_array_equal(got, want[i])
                if at is not None:
                    assert (pinned[:at] == -7.0).all() and (pinned[at + n:] == -7.0).all()
            for s in seqs:
                e.close_seq(s)


def test_returned_rows_resize_in_place(gpu, tmp_path):
    """A step's array owns its rows, in pinned memory or not: it resizes in place, grows and shrinks,
    and later steps' rows are theirs."""
    import engine
    cfg = T.config([(T.attn(), None)], vocab=5003)
    with engine.Engine(T.save(tmp_path, cfg, T.weights(cfg, 3)), dtype="float32", max_seqs=2, max_tokens=512) as e:
        for n in (3, 4, 60):  # 60,036 and 80,048 bytes; 1.2 MB
            outs = []
            for _ in range(3):
                s = e.open_seq()
                outs.append(e.step([(s, np.arange(n), list(range(n)))]))
                e.close_seq(s)
            want = outs[0].copy()
            assert outs[0].flags.owndata and outs[0].base is None
            outs[0].resize((2 * n, e.vocab), refcheck=False)
            outs[1].resize((n - 2, e.vocab), refcheck=False)
            outs[1].resize((n - 1, e.vocab), refcheck=False)
            np.testing.assert_array_equal(outs[0][:n], want)
            assert not outs[0][n:].any() and not outs[1][n - 2:].any()
            np.testing.assert_array_equal(outs[1][:n - 2], want[:n - 2])
            np.testing.assert_array_equal(outs[2], want)
            assert np.zeros(100000).flags.owndata  # (other arrays are as ever)
