"""ps_autotune remembers its times per problem shape.  A mesh without the symmetry orbits runs the J-free form
by tiles, at about half the speed: it is a shape of its own and is timed by itself, and so is a problem whose
lightcurves pack into another number of passes."""
import numpy as np
import pytest

from periodsearch_amd import PeriodSearch
from tests.test_gpu_orbits import problem

pytestmark = pytest.mark.gpu


def tuned(text, turned=False):
    ps = PeriodSearch.from_text(text)
    if turned:
        g = ps._geo.contents
        nor = np.ctypeslib.as_array(g.nor, (g.nfac * 3,)).reshape(g.nfac, 3)
        c, s = np.cos(1e-3), np.sin(1e-3)
        nor[:] = nor @ np.array([[1, 0, 0], [0, c, -s], [0, s, c]]).T
    ps.prepare(device=0)
    try:
        return ps.autotune(ps.info()["conw_r0"])
    finally:
        ps.close()


def short(*args):
    lines = problem(*args).split("\n")
    lines[10] = "4"  # iterations
    return "\n".join(lines)


def test_another_form_or_pass_count_is_timed_again():
    text = short(3, 3, 5, 4, 60, 10)
    first = tuned(text)
    other = tuned(text, turned=True)
    assert other[1:] != first[1:], "times of a mesh with orbits given for one without"
    assert tuned(text) == first and tuned(text, turned=True) == other, "remembered"
    # 250 points both: four curves of 60 (two to a pass), or three of 80 (one to a pass)
    packed = tuned(short(3, 3, 5, 3, 80, 10))
    assert packed[1:] != first[1:], "times of another pass count"
