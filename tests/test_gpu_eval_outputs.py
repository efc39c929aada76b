"""The outputs of ps_eval on their way out (periodsearch_amd/csrc/ps_device.hip, ps_fit2.h), bit for bit: raw rows
of passes whose last point group is part filled, from one workgroup and from passes spread over many, and
long lists, which are computed in chunks and copied in pieces by several threads, against the same vectors
in short calls.  What is computed is mrqcof.c:16-148 and bright.c:14-126 (against the oracle:
test_gpu_orbits.py)."""
import numpy as np
import pytest

from periodsearch_amd import PS_KERNEL_JFREE, PeriodSearch
from periodsearch_amd import _lib as L
from tests import oracle_binding as ob
from tests.test_gpu_orbits import problem

pytestmark = pytest.mark.gpu

KEYS = ("alpha", "beta", "chisq", "ymod", "dyda")


def prepared(*args, **kw):
    ps = PeriodSearch.from_text(problem(*args, **kw)).prepare(device=0)
    ps.set_kernel(PS_KERNEL_JFREE)
    return ps


def vectors(ps, n):
    rng = np.random.default_rng(11)
    info = ps.info()
    a = np.zeros((n, info["ma"]))
    nc = info["ncoef"]
    a[:, :nc] = ps.geometry()["cg_first"] + rng.normal(0, 0.05, (n, nc)) / (1 + np.arange(nc))
    a[:, nc] = rng.uniform(0.3, 2.8, n)
    a[:, nc + 1] = rng.uniform(0, 6.0, n)
    a[:, nc + 2] = 2 * np.pi * 24 * ps.freq(1)
    a[:, nc + 3:nc + 6] = 0.5, 0.1, -0.5
    a[:, nc + 6], a[:, nc + 7] = np.log(0.1), 1.0
    return a


@pytest.mark.parametrize("shape", [
    (5, 5, 5, 6, 56, 0),    # 7 tiles a pass: the second group's last 16 lanes are the next pass's first points
    (6, 6, 6, 4, 72, 0),    # 5 tiles: 48 of them
    (3, 3, 6, 5, 70, 300),  # calibrated points in the passes' tails
], ids=str)
def test_raw_rows_of_part_filled_passes(shape):
    ps = prepared(*shape)
    try:
        conw, n = ps.info()["conw_r0"], ps.info()["slots"] // 2 + 100
        vecs = vectors(ps, n)
        full = ps.eval(vecs, conw, raw=True)  # one workgroup a vector
        for m in (1, 9):  # spread
            got = ps.eval(vecs[:m], conw, raw=True)
            for k in KEYS:
                assert np.array_equal(got[k], full[k][:m]), (m, k)
    finally:
        ps.close()


@pytest.mark.parametrize("cl_free", [False, True])
@pytest.mark.parametrize("cls", [1e45, 1e100, 1e-45])
def test_any_lommel_seeliger_weight(cls, cl_free):
    """The caller's vector may hold any weight of the Lommel-Seeliger term: with raw rows (whose Lambert columns
    keep the weight apart from the areas) as without."""
    text = problem(6, 6, 6, 2, 50, 300, cl_free=cl_free)
    orc = ob.OracleCtx.from_text(text)
    ps = prepared(6, 6, 6, 2, 50, 300, cl_free=cl_free)
    try:
        conw = ps.info()["conw_r0"]
        orc.set_conw(conw)
        vecs = vectors(ps, 3)
        vecs[:, -1] = cls
        got, plain = ps.eval(vecs, conw, raw=True), ps.eval(vecs, conw)
        for k in ("alpha", "beta", "chisq"):
            assert np.array_equal(got[k], plain[k]), k
        arr = ps.input_arrays()
        n = len(arr["tim"])
        for v, a in enumerate(vecs):
            al, be, chi = orc.mrqcof(a)
            assert np.abs(got["alpha"][v] - al).max() <= 1e-11 * np.abs(al).max()
            assert np.abs(got["beta"][v] - be).max() <= 1e-11 * np.abs(be).max()
            assert abs(got["chisq"][v] - chi) <= 1e-12 * chi
            for p in (0, n // 3, n - 1):
                br, dy = orc.bright(a, arr["ee"][p], arr["ee0"][p], arr["tim"][p])
                assert abs(got["ymod"][v, p] - br) <= 1e-13 * abs(br), p
                assert np.abs(got["dyda"][v, p] - dy).max() <= 1e-12 * np.abs(dy).max(), p
    finally:
        ps.close()


def call(ps, vecs, conw, keys):
    """ps_eval with the named outputs only."""
    info, n = ps.info(), len(vecs)
    shape = {"alpha": (n, info["mfit"], info["mfit"]), "beta": (n, info["mfit"]), "chisq": (n,),
             "ymod": (n, info["npts"]), "dyda": (n, info["npts"], info["ma"])}
    out = {k: np.full(shape[k], np.nan) for k in keys}
    ptr = [out[k].ctypes.data_as(L.DP) if k in out else None for k in KEYS]
    L.check(L.lib().ps_eval(ps._handle(), n, vecs.ctypes.data_as(L.DP), float(conw), *ptr), "ps_eval")
    return out


@pytest.mark.parametrize("keys", [KEYS, KEYS[:3], ("alpha",), ("chisq", "ymod", "dyda"), ()], ids=str)
def test_long_lists_match_short_calls(keys):
    """Chunks of whole rounds and a remainder of one, of a few and of none; pieces that cross the arrays' ends."""
    ps = prepared(5, 5, 5, 2, 30, 0)  # 36 KB of outputs a vector: up to three chunks
    try:
        conw, slots = ps.info()["conw_r0"], ps.info()["slots"]
        vecs = vectors(ps, 2 * slots + 3)
        parts = [ps.eval(vecs[i:i + 7], conw, raw=True) for i in range(0, len(vecs), 7)]
        want = {k: np.concatenate([p[k] for p in parts]) for k in KEYS}
        for n in (2 * slots + 3, 2 * slots, slots + 1):
            got = call(ps, vecs[:n], conw, keys)
            for k in keys:
                assert np.array_equal(got[k], want[k][:n]), (n, k)
    finally:
        ps.close()


@pytest.mark.parametrize("n", [1, 2, 3, 5, 7, 8, 9, 30])
def test_results_of_one_to_several_pieces(n):
    ps = prepared(6, 6, 4, 20, 50, 300)  # 0.6 MB of raw rows a vector: results of one piece to eighteen
    try:
        conw = ps.info()["conw_r0"]
        vecs = vectors(ps, n)
        got = call(ps, vecs, conw, KEYS)
        for i in range(n):
            one = call(ps, vecs[i:i + 1], conw, KEYS)
            for k in KEYS:
                assert np.array_equal(got[k][i], one[k][0]), (i, k)
    finally:
        ps.close()
