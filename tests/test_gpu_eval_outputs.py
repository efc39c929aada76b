"""The outputs of ps_eval on their way out (periodsearch_amd/csrc/ps_device.hip, ps_fit2.h), bit for bit: raw rows
of passes whose last point group is part filled, from one workgroup and from passes spread over many, and
long lists, which are computed in chunks and copied in pieces by several threads, against the same vectors
in short calls.  What is computed is mrqcof.c:16-148 and bright.c:14-126 (against the oracle:
test_gpu_orbits.py)."""
import numpy as np
import pytest

from periodsearch_amd import PS_KERNEL_JFREE, PeriodSearch
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
