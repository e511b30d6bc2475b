"""The one-launch solves on the shapes where they can go wrong, against the
kernels that stream the matrix: the same bits."""

import time

import numpy as np
import pytest

from chysx import scenes
from chysx.harness import make_batch, make_sim

pytestmark = pytest.mark.gpu


def mesh(w, h=None, crossed=False, seed=None):
    """A w x h cloth hanging from two corners; crossed: diagonals alternate, so
    rows have up to 8 neighbours; seed: vertices in a random order."""
    h = h or w
    j, i = np.meshgrid(np.arange(h), np.arange(w), indexing="ij")
    pos = np.zeros((w * h, 3), np.float32)
    pos[:, 0], pos[:, 2] = (i.reshape(-1) / 100.0).astype(np.float32), (j.reshape(-1) / 100.0).astype(np.float32)
    jj, ii = np.meshgrid(np.arange(h - 1), np.arange(w - 1), indexing="ij")
    v00 = (jj * w + ii).reshape(-1)
    v10, v01, v11 = v00 + 1, v00 + w, v00 + w + 1
    odd = crossed & ((ii + jj) % 2 == 1).reshape(-1)
    tris = np.concatenate([np.stack([v00, v10, np.where(odd, v01, v11)], 1),
                           np.stack([np.where(odd, v10, v00), v11, v01], 1)]).astype(np.int32)
    pins = np.array([(h - 1) * w, h * w - 1], np.int32)
    if seed is not None:
        order = np.random.default_rng(seed).permutation(w * h)
        at = np.empty(w * h, np.int32)
        at[order] = np.arange(w * h)
        pos, tris, pins = pos[order], at[tris], at[pins]
    return scenes.Scene(f"mesh_{w}_{h}", pos, np.zeros_like(pos), np.full(len(pos), 100.0, np.float32), tris, pins,
                        pos[pins].copy(), 1.0e6, 1.0e3, 1.0e3, None, 1.0 / 60.0, 4)


def assert_same_bits(make, steps=2, modes=(-1,)):
    """Positions, velocities and statistics of `steps` steps under mode 0 and the others."""
    out = {}
    for mode in (0, *modes):
        g = make()
        h = g.sim if hasattr(g, "sim") else g.batch
        h.set_resident_solve(mode)
        rows = []
        for _ in range(steps):
            h.step(1.0 / 60.0)
            rows += [g.pos.cpu().numpy(), g.vel.cpu().numpy(),
                     [h.last_solve_stats()] if hasattr(g, "sim") else [h.stats(k) for k in range(h.num_cloths())]]
        assert np.isfinite(rows[-3]).all()
        out[mode] = rows
    for mode in modes:
        for a, b in zip(out[mode], out[0]):
            if isinstance(a, list):
                assert a == b, mode
            else:
                np.testing.assert_array_equal(a, b)


# batches of more workgroups than there are compute units: places in the order
# of starting (cloths of up to 32 workgroups) and by number (larger ones)
BATCHES = {
    "whole_groups_by_start": lambda: [mesh(w) for w in [181] * 8 + [100] * 10 + [33, 20, 5]],
    "whole_groups_by_number": lambda: [mesh(450), mesh(449), mesh(190), mesh(40), mesh(9)],
    "half_groups_by_start": lambda: [mesh(w, crossed=True) for w in [128] * 8 + [70] * 3 + [23, 10]],
    "half_groups_by_number": lambda: [mesh(w, crossed=True) for w in (257, 256, 129, 31)],
}


@pytest.mark.parametrize("name", BATCHES)
def test_batch_beyond_the_compute_units(cuda, name):
    sc = BATCHES[name]()
    assert_same_bits(lambda: make_batch(sc, tol=0.0, max_iter=11))
    b = make_batch(sc, tol=0.0, max_iter=11)
    b.batch.set_blocking_step(True)
    b.batch.step(1.0 / 60.0)
    t = time.perf_counter()
    b.batch.step(1.0 / 60.0)
    # milliseconds; half a second when workgroups wait for ones that cannot start
    assert time.perf_counter() - t < 0.3
