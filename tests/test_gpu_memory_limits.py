"""Calls whose buffers cannot be had (the limits are forced on the handle or batch): they take the other form and
return the same bits, as they did before there was a choice of forms; and the spread form's memory, which the
handles of a device share."""
import ctypes as C
import gc
import threading

import numpy as np
import pytest

from periodsearch_amd import FIT_DTYPE, Batch, lib
from tests.test_gpu_spread_rule import passes, prepared, spread

pytestmark = pytest.mark.gpu


ALL = C.c_size_t(-1).value


def limit(ps, arena=ALL, pinned=ALL):
    fn = lib().ps_test_limits
    fn.argtypes, fn.restype = [C.c_void_p, C.c_size_t, C.c_size_t], None
    fn(ps._handle(), arena, pinned)


def batch_limit(b, arena):
    fn = lib().ps_test_batch_limits
    fn.argtypes, fn.restype = [C.c_void_p, C.c_size_t], None
    fn(b._b, arena)


def batch_spread(b):
    fn = lib().ps_test_batch_spread
    fn.argtypes, fn.restype = [C.c_void_p], C.c_int
    return fn(b._b)


def same(a, b, what):
    for k in FIT_DTYPE.names:
        assert np.array_equal(a[k], b[k], equal_nan=True), (what, k)


def test_a_later_piece_larger_than_the_first():
    """Long fits fill the first piece, many short ones the second: their normal equations take more memory."""
    searches = [prepared(passes(6, 6, 24)), prepared(passes(3, 4, 2))]
    try:
        conw = np.array([s.info()["conw_r0"] for s in searches])
        prob = np.repeat([0, 1], [336, 4000])
        pole = np.arange(len(prob)) % 10 + 1
        freq = np.concatenate([searches[0].freq(1 + np.arange(336) // 10), searches[1].freq(1 + np.arange(4000) // 10 % 50)])
        with Batch(searches) as b:
            free = b.run(conw, prob, freq, pole)
            assert batch_spread(b) == len(prob), "the case means two pieces"
        with Batch(searches) as b:
            batch_limit(b, 300 << 20)  # the first piece needs 220 MB, the second 380
            got = b.run(conw, prob, freq, pole)
            assert batch_spread(b) == 0
        same(got, free, "limited")
        few = np.arange(330, 350)
        for i, s in enumerate(searches):
            sel = few[prob[few] == i]
            same(free[sel], s.fit_batch(freq[sel], pole[sel], conw[i]), i)
    finally:
        for s in searches:
            s.close()


def test_no_room_to_spread():
    text = passes(6, 6, 10)
    a, b = prepared(text), prepared(text)
    try:
        conw = a.info()["conw_r0"]
        freq, pole = a.freq(1 + np.arange(20) // 10), 1 + np.arange(20) % 10
        limit(b, 1 << 20)
        want, got = a.fit_batch(freq, pole, conw), b.fit_batch(freq, pole, conw)
        assert (spread(a), spread(b)) == (20, 0)
        same(got, want, "fits")
        vec = np.zeros((9, a.info()["ma"]))
        nc = a.info()["ncoef"]
        vec[:, :nc], vec[:, nc] = a.geometry()["cg_first"], np.linspace(0.5, 2.5, 9)
        vec[:, nc + 2] = 2 * np.pi * 24 * a.freq(1)
        vec[:, nc + 3:] = 0.5, 0.1, -0.5, -2.0, 1.0
        want, got = a.eval(vec, conw, raw=True), b.eval(vec, conw, raw=True)
        assert (spread(a), spread(b)) == (9, 0)
        for k in want:
            assert np.array_equal(got[k], want[k]), k
    finally:
        a.close()
        b.close()


def test_evaluations_without_pinned_memory():
    """Short lists and lists in chunks, all outputs and some of them."""
    text = passes(3, 4, 2)
    a, b = prepared(text), prepared(text)
    try:
        limit(b, pinned=0)
        conw = a.info()["conw_r0"]
        n = 2 * a.info()["slots"] + 3
        vec = np.zeros((n, a.info()["ma"]))
        nc = a.info()["ncoef"]
        vec[:, :nc], vec[:, nc] = a.geometry()["cg_first"], np.linspace(0.5, 2.5, n)
        vec[:, nc + 2] = 2 * np.pi * 24 * a.freq(1)
        vec[:, nc + 3:] = 0.5, 0.1, -0.5, -2.0, 1.0
        for m, raw in ((1, True), (9, False), (n, True), (n, False)):
            want, got = a.eval(vec[:m], conw, raw=raw), b.eval(vec[:m], conw, raw=raw)
            for k in want:
                assert np.array_equal(got[k], want[k]), (m, k)
    finally:
        a.close()
        b.close()


def arenas():
    fn = lib().ps_test_arenas
    fn.argtypes, fn.restype = [C.c_int, C.POINTER(C.c_int)], C.c_size_t
    n = C.c_int()
    return fn(0, C.byref(n)), n.value


def test_open_handles_share_the_spread_memory():
    """Handles that stay open after a spread call hold none of its memory; what waits for the next call is
    bounded and goes with the last handle."""
    gc.collect()
    others = arenas()[1]
    text = passes(6, 6, 20)
    searches = [prepared(text) for _ in range(6)]
    try:
        conw = searches[0].info()["conw_r0"]
        freq, pole = searches[0].freq(1 + np.arange(100) // 10), 1 + np.arange(100) % 10
        want = None
        for s in searches:
            got = s.fit_batch(freq, pole, conw)
            assert spread(s) == 100
            want = got if want is None else want
            same(got, want, "another handle's arena")
        one = 100 * 20 * 24576  # the Gram blocks of one call
        assert arenas()[1] == others + 6
        if others == 0:
            assert one <= arenas()[0] < 2 * one
        assert arenas()[0] < 3 * (200 << 20)
    finally:
        for s in searches:
            s.close()
    assert arenas()[1] == others
    if others == 0:
        assert arenas()[0] == 0


def test_threads_with_handles_of_their_own():
    """Calls that overlap on streams of their own never share an arena."""
    shapes = [passes(6, 6, 12), passes(3, 4, 20), passes(6, 8, 10), passes(4, 5, 16)]
    searches = [prepared(t) for t in shapes]
    try:
        jobs = []
        for s in searches:
            n = 1 + np.arange(60)
            jobs.append((s, s.freq(1 + n // 10), 1 + n % 10, s.info()["conw_r0"]))
        want = [s.fit_batch(f, p, c) for s, f, p, c in jobs]
        got = [[None] * 5 for _ in jobs]

        def work(i):
            s, f, p, c = jobs[i]
            for r in range(5):
                m = 60 - 10 * r  # arenas of several sizes
                got[i][r] = s.fit_batch(f[:m], p[:m], c)

        threads = [threading.Thread(target=work, args=(i,)) for i in range(len(jobs))]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        for i, w in enumerate(want):
            for r in range(5):
                same(got[i][r], w[:60 - 10 * r], (i, r))
    finally:
        for s in searches:
            s.close()
