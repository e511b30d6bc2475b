"""The iterations of one large cloth in one launch (vectors on the chip, matrix
streamed) against the kernels of one pass each: the same bits at 2, 3 and 4
groups of rows a workgroup, with uneven last workgroups, stopped, restarted and
warm-started solves, and when one workgroup has to solve alone (mode 2)."""

import numpy as np
import pytest

from chysx import scenes
from chysx.harness import make_sim
from test_gpu_resident import run

pytestmark = pytest.mark.gpu


def wind(w, mode=None, pins=False, **kw):
    def make():
        g = make_sim(scenes.config3(w=w), **kw)
        if pins:
            g.sim.set_pin_projection(True)
        if mode:
            g.sim.set_warm_start_mode(mode)
        return g
    return make


CASES = {
    # 2 groups a workgroup: the fewest rows there are, one of them in the last
    # slice; an owed direction at the end or none; one iteration
    "513": wind(513, tol=0.0, max_iter=25), "513_even": wind(513, tol=0.0, max_iter=24),
    "513_1": wind(513, tol=0.0, max_iter=1), "513_tol": wind(513, tol=1e-6),
    "514_capped": wind(514, tol=1e-6, max_iter=9), "520_projection": wind(520, mode="projection", tol=1e-6),
    "520_pins": wind(520, pins=True, tol=1e-6),
    # the most rows of 2 groups, the fewest of 3, the most of 4, one row too many
    "724": wind(724, tol=0.0, max_iter=9), "725": wind(725, tol=0.0, max_iter=9),
    "1024": wind(1024, tol=1e-6), "1025": wind(1025, tol=0.0, max_iter=9),
}


@pytest.mark.parametrize("name", CASES)
def test_same_bits_as_the_streaming_kernels(cuda, name):
    want, want_stats = run(CASES[name], 0, steps=2)
    assert np.isfinite(want[-1]).all()
    got, got_stats = run(CASES[name], -1, steps=2)
    assert got_stats == want_stats
    for a, b in zip(got, want):
        np.testing.assert_array_equal(a, b)


def test_one_workgroup_alone_gives_the_same_bits(cuda):
    make = wind(513, tol=0.0, max_iter=3)
    want, want_stats = run(make, 0, steps=2)
    got, got_stats = run(make, 2, steps=2)
    assert got_stats == want_stats
    for a, b in zip(got, want):
        np.testing.assert_array_equal(a, b)
