"""The solve in one launch (matrix in registers) against the kernels that
stream the matrix: positions, velocities, the FP64 iterate and the solve's
statistics are the same bits, whatever the mesh, the options and the number of
workgroups; also when an instance is solved by one workgroup alone because the
others did not start in time (mode 2 gives the start-up no time at all)."""

import numpy as np
import pytest

from chysx import scenes
from chysx.harness import make_batch, make_sim

pytestmark = pytest.mark.gpu


def fan(spokes, rings, bend=None):
    """A disc of `rings` rings of `spokes` vertices around a hub of that degree."""
    ang = 2.0 * np.pi * np.arange(spokes) / spokes
    pos = [np.zeros((1, 3))]
    for r in range(1, rings + 1):
        pos.append(np.stack([0.1 * r * np.cos(ang), 0.003 * np.sin(5 * ang), 0.1 * r * np.sin(ang)], 1))
    tris = []
    for k in range(spokes):
        n = (k + 1) % spokes
        tris.append((0, 1 + k, 1 + n))
        for r in range(rings - 1):
            a, b = 1 + r * spokes, 1 + (r + 1) * spokes
            tris += [(a + k, b + k, b + n), (a + k, b + n, a + n)]
    pos = np.concatenate(pos).astype(np.float32)
    idx = np.array([1, 1 + spokes // 2], np.int32)
    return scenes.Scene(f"fan_{spokes}_{rings}", pos, np.zeros_like(pos), np.full(len(pos), 100.0, np.float32),
                        np.array(tris, np.int32), idx, pos[idx].copy(), 1.0e6, 300.0, 300.0, None, 1.0 / 60.0, 4,
                        bend_k=bend)


def wind(w, **kw):
    return lambda: make_sim(scenes.config3(w=w), **kw)


def drape(w, **kw):
    return lambda: make_sim(scenes.drape(w, seed=5), springs_active=False, **kw)


def projected_pins():
    g = make_sim(scenes.config3(w=40), tol=1e-6)
    g.sim.set_pin_projection(True)
    return g


def on_ground():
    g = make_sim(scenes.drape(40), tol=1e-6, springs_active=False)
    g.sim.add_static_plane(np.array([0, 1, 0], np.float32), 0.0)
    g.sim.set_static_contact_thickness(0.002)
    g.sim.set_static_contact_stiffness(2e3)
    g.sim.set_static_contact_friction(0.4)
    return g


def warm(mode):
    def make():
        from chysx.warmstart import load_params
        g = make_sim(scenes.config3(w=48), tol=1e-6)
        g.sim.ws_set_params(load_params()[0])
        g.sim.set_warm_start_mode(mode)
        return g
    return make


def full_blocks(w):
    def make():
        g = make_sim(scenes.config3(w=w), tol=1e-6)
        g.sim.set_launch_config(dict(spmv_symmetric=0))
        return g
    return make


CASES = {
    # one workgroup: less than a slice, whole slices, one row into a slice, a full group
    "wind3": wind(3, tol=1e-6), "wind8": wind(8, tol=0.0, max_iter=50), "wind20_restarts": wind(20, tol=1e-6),
    "wind32": wind(32, tol=1e-6), "wind32_capped": wind(32, tol=1e-6, max_iter=7),
    "wind32_1": wind(32, tol=0.0, max_iter=1), "wind32_2": wind(32, tol=0.0, max_iter=2),
    # many: one row into the second group, uneven last group, more than 64 groups
    "wind33": wind(33, tol=1e-6), "wind47": wind(47, tol=0.0, max_iter=49), "wind300": wind(300, tol=0.0, max_iter=20),
    # 9-float blocks in half groups: one piece, the second piece's first slice, many
    "drape22": drape(22, tol=0.0, max_iter=50), "drape23": drape(23, tol=1e-6, max_iter=200),
    "drape32": drape(32, tol=0.0, max_iter=50), "drape33": drape(33, tol=0.0, max_iter=50),
    "drape120": drape(120, tol=0.0, max_iter=30), "general24": full_blocks(24), "general50": full_blocks(50),
    # wide rows, packed and not; too wide for any variant
    "fan12": lambda: make_sim(fan(12, 9), tol=1e-6), "fan16": lambda: make_sim(fan(16, 90), tol=1e-6),
    "fan12_bending": lambda: make_sim(fan(12, 9, bend=0.01), tol=1e-6),
    "fan30": lambda: make_sim(fan(30, 9), tol=1e-6),
    "projected_pins": projected_pins, "on_ground": on_ground,
    "warm_projection": warm("projection"), "warm_learned": warm("learned"),
    "batch": lambda: make_batch(scenes.config4(count=20, wmin=4, wmax=70, seed=9), tol=1e-6),
    "batch_fixed": lambda: make_batch(scenes.config4(count=7, wmin=6, wmax=32, seed=3), tol=0.0, max_iter=31),
}


def run(make, mode, steps=4):
    g = make()
    h = g.sim if hasattr(g, "sim") else g.batch
    h.set_resident_solve(mode)
    out, stats = [], []
    for _ in range(steps):
        h.step(1.0 / 60.0)
        if hasattr(g, "sim"):
            stats.append([h.last_solve_stats()])
        else:
            stats.append([h.stats(k) for k in range(h.num_cloths())])
        out += [g.pos.cpu().numpy(), g.vel.cpu().numpy()]
    if hasattr(g, "sim"):
        out.append(h.get_dx64())
    return out, stats


@pytest.mark.parametrize("name", CASES)
def test_same_bits_as_the_streaming_kernels(cuda, name):
    want, want_stats = run(CASES[name], 0)
    assert np.isfinite(want[-1]).all()
    for mode in (-1, 2):
        got, got_stats = run(CASES[name], mode)
        assert got_stats == want_stats, mode
        for a, b in zip(got, want):
            np.testing.assert_array_equal(a, b)


def test_not_a_number_stays_in_its_cloth_and_ends(cuda):
    """A cloth with a NaN velocity runs its fixed count and leaves its batch mates as they are."""
    sc = scenes.config4(count=3, wmin=40, wmax=60, seed=2)
    outs = []
    for mode in (0, -1):
        b = make_batch(sc, tol=0.0, max_iter=10)
        b.batch.set_resident_solve(mode)
        b.batch.step(1.0 / 60.0)
        b.vel[b.offsets[1] + 5, 1] = float("nan")
        b.batch.step(1.0 / 60.0)
        outs.append([b.positions(k) for k in range(3)])
        assert [b.batch.stats(k)["iters"] for k in range(3)] == [10, 10, 10]
    for k in range(3):
        np.testing.assert_array_equal(outs[0][k], outs[1][k])
    assert np.isfinite(outs[1][0]).all() and np.isfinite(outs[1][2]).all()


def test_steps_on_two_streams(cuda):
    """Solves of many workgroups enqueued on two streams and the null stream give the same results."""
    import torch
    sc = scenes.config3(w=128)
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    sims = [make_sim(sc, tol=0.0, max_iter=40) for _ in range(3)]
    torch.cuda.synchronize()
    for _ in range(4):
        for g, s in zip(sims[:2], streams):
            g.sim.step(sc.dt, s.cuda_stream)
        sims[2].sim.step(sc.dt)
    torch.cuda.synchronize()
    for g in sims[:2]:
        np.testing.assert_array_equal(g.positions(), sims[2].positions())
