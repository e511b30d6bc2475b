"""The one-launch solves on the shapes where they can go wrong, against the
kernels that stream the matrix: the same bits."""

import time

import numpy as np
import pytest

from chysx import scenes
from chysx.harness import make_batch, make_sim
from test_gpu_resident import CASES as ONE_LAUNCH
from test_gpu_resident import fan
from test_gpu_sweep import CASES as SWEEP

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


def handle(g):
    return g.sim if hasattr(g, "sim") else g.batch


def assert_same_bits(make, form, steps=2, modes=(-1,)):
    """Positions, velocities and statistics of `steps` steps under mode 0 and the
    others, which solve in form `form`."""
    out = {}
    for mode in (0, *modes):
        g = make()
        h = handle(g)
        h.set_resident_solve(mode)
        rows = []
        for _ in range(steps):
            h.step(1.0 / 60.0)
            rows += [g.pos.cpu().numpy(), g.vel.cpu().numpy(),
                     [h.last_solve_stats()] if hasattr(g, "sim") else [h.stats(k) for k in range(h.num_cloths())]]
            assert h.solve_form() == ("streaming" if mode == 0 else form)
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
    assert_same_bits(lambda: make_batch(sc, tol=0.0, max_iter=11), "one_launch")
    b = make_batch(sc, tol=0.0, max_iter=11)
    b.batch.set_blocking_step(True)
    b.batch.step(1.0 / 60.0)
    t = time.perf_counter()
    b.batch.step(1.0 / 60.0)
    # milliseconds; half a second when workgroups wait for ones that cannot start
    assert time.perf_counter() - t < 0.3


@pytest.mark.parametrize("cases, name", [(c, n) for c in (ONE_LAUNCH, SWEEP) for n in c],
                         ids=lambda v: v if isinstance(v, str) else "")
def test_the_form_that_solves(cuda, cases, name):
    """The meshes that are compared with the streaming kernels do take the other forms."""
    h = handle(cases[name]())
    h.step(1.0 / 60.0)
    # too wide (fan12_bending's hub couples to 24 rows), or one row too many
    assert h.solve_form() == ("streaming" if name in ("fan30", "fan12_bending", "1025") else
                              "one_launch" if cases is ONE_LAUNCH else "sweep")


def drape(w):
    return lambda: make_sim(scenes.drape(w, seed=5), tol=0.0, max_iter=9, springs_active=False)


def cloth(*a, tol=0.0, **kw):
    return lambda: make_sim(mesh(*a, **kw), tol=tol, max_iter=9 if tol == 0.0 else 10000)


def training():
    from chysx.warmstart import load_params
    g = make_sim(mesh(48), tol=1e-6)
    g.sim.ws_set_params(load_params()[0])
    g.sim.set_warm_start_mode("learned")
    g.sim.ws_set_training(True, 1e-4)
    return g


SHAPES = {
    # 9-float half groups: z received before the sums (from 61 workgroups), more
    # than 64 groups, more than one round of looks for three values (from 95
    # groups), the most workgroups there are, one row too many
    "drape200": (drape(200), "one_launch"), "drape270": (drape(270), "one_launch"),
    "drape320": (drape(320), "one_launch"), "drape362": (drape(362), "one_launch"),
    "drape363": (drape(363), "streaming"),
    # packed half groups (rows of up to 8 neighbours)
    "crossed23": (cloth(23, crossed=True), "one_launch"), "crossed150": (cloth(150, crossed=True, tol=1e-6), "one_launch"),
    "crossed362": (cloth(362, crossed=True), "one_launch"), "crossed363": (cloth(363, crossed=True), "streaming"),
    # the widest rows of each kind, and wider ones
    "fan16": (lambda: make_sim(fan(16, 5), tol=1e-6), "one_launch"),
    "fan17": (lambda: make_sim(fan(17, 5), tol=1e-6), "streaming"),
    "fan7_bending": (lambda: make_sim(fan(7, 90, bend=0.01), tol=1e-6), "one_launch"),
    "fan8_bending": (lambda: make_sim(fan(8, 9, bend=0.01), tol=1e-6), "streaming"),
    # whole groups: the most workgroups, long and narrow, any numbering
    "512": (cloth(512), "one_launch"), "16x4096": (cloth(16, 4096), "one_launch"),
    "4096x16": (cloth(4096, 16), "one_launch"), "shuffled64": (cloth(64, seed=3, tol=1e-6), "one_launch"),
    "shuffled128": (cloth(128, seed=3), "streaming"),
    # the sweep beyond squares; boundary rows that no longer fit
    "700x1400": (cloth(700, 1400), "sweep"), "300x2000": (cloth(300, 2000, tol=1e-4), "sweep"),
    "1400x700": (cloth(1400, 700), "streaming"), "shuffled520": (cloth(520, seed=3), "streaming"),
    "training": (training, "one_launch"),
}


@pytest.mark.parametrize("name", SHAPES)
def test_same_bits_as_the_streaming_kernels(cuda, name):
    make, form = SHAPES[name]
    assert_same_bits(make, form, steps=3 if name == "training" else 2)


def test_form_of_a_batch_by_its_iterations(cuda):
    """Wide-row cloths that need more workgroups than there are compute units:
    in one launch only from a number of iterations on, and not at all where they leave most compute units unused."""
    def forms(sc, steps=1, **kw):
        b = make_batch(sc, **kw)
        out = []
        for _ in range(steps):
            b.batch.step(1.0 / 60.0)
            out.append(b.batch.solve_form())
        return out
    many = [mesh(128, crossed=True) for _ in range(12)]
    assert forms(many, tol=0.0, max_iter=2) == ["streaming"]
    assert forms(many, tol=0.0, max_iter=50) == ["one_launch"]
    assert forms(many, steps=2, tol=1e-6, max_iter=3) == ["streaming", "streaming"]
    # with a tolerance, by the iterations of the step before: 6 for these cloths
    b = make_batch(many, tol=1e-6)
    before = 10000
    for _ in range(5):
        b.batch.step(1.0 / 60.0)
        assert b.batch.solve_form() == ("one_launch" if before >= 6 else "streaming")
        before = max(b.batch.stats(k)["iters"] for k in range(12))
    assert forms([mesh(257, crossed=True) for _ in range(3)], tol=0.0, max_iter=50) == ["streaming"]
    assert_same_bits(lambda: make_batch(many, tol=0.0, max_iter=50), "one_launch")


def test_wide_and_small_solves_on_several_streams(cuda):
    """A cloth that takes every compute unit beside batches whose cloths span a
    few workgroups, each on a stream of its own: the results of each alone, and
    no start-up wait that runs out (half a second each)."""
    import torch
    small = [mesh(w) for w in [40, 64, 90] * 30]
    makes = [lambda: make_sim(mesh(512), tol=0.0, max_iter=20), lambda: make_batch(small, tol=0.0, max_iter=15),
             lambda: make_sim(mesh(513), tol=0.0, max_iter=10), lambda: make_batch(small[:40], tol=0.0, max_iter=40)]
    alone = []
    for make in makes:
        g = make()
        for _ in range(9):
            handle(g).step(1.0 / 60.0)
        alone.append(g.pos.cpu().numpy())
    gs = [make() for make in makes]
    streams = [torch.cuda.Stream() for _ in gs]
    for g in gs:
        handle(g).step(1.0 / 60.0)
    torch.cuda.synchronize()
    t = time.perf_counter()
    for _ in range(8):
        for g, s in zip(gs, streams):
            handle(g).step(1.0 / 60.0, s.cuda_stream)
    torch.cuda.synchronize()
    assert time.perf_counter() - t < 0.4
    for g, want in zip(gs, alone):
        np.testing.assert_array_equal(g.pos.cpu().numpy(), want)


@pytest.mark.parametrize("w", [60, 530])
def test_storage_changed_behind_an_enqueued_step(cuda, w):
    """A change of the matrix storage waits for the step that was enqueued
    before it, on a stream of its own."""
    import torch
    def run(wait):
        g = make_sim(mesh(w), tol=0.0, max_iter=400)
        s = torch.cuda.Stream()
        torch.cuda.synchronize()
        for storage in (dict(spmv_symmetric=0), dict(spmv_symmetric=1, spmv_packed=1), dict(spmv_symmetric=1, spmv_packed=0)):
            g.sim.step(1.0 / 60.0, s.cuda_stream)
            if wait:
                torch.cuda.synchronize()
            g.sim.set_launch_config(storage)
        g.sim.step(1.0 / 60.0, s.cuda_stream)
        torch.cuda.synchronize()
        return g.pos.cpu().numpy(), g.sim.last_solve_stats()
    (a, sa), (b, sb) = run(False), run(True)
    np.testing.assert_array_equal(a, b)
    assert sa == sb and np.isfinite(a).all()


LOST = {"one_launch": lambda: make_sim(mesh(60), tol=0.0, max_iter=20),
        "one_launch_tol": lambda: make_sim(mesh(60), tol=1e-6),
        "batch": lambda: make_batch([mesh(w) for w in (20, 60, 40)], tol=0.0, max_iter=20),
        "sweep": lambda: make_sim(mesh(520), tol=0.0, max_iter=5),
        "sweep_tol": lambda: make_sim(mesh(520), tol=1e-4)}


@pytest.mark.parametrize("name", LOST)
def test_lost_workgroup_is_reported_and_not_trusted(cuda, name):
    """After a solve that lost a workgroup (mode 4 marks the exchange as such a
    solve leaves it) no further one runs on its words: the error comes from the
    step itself, from the statistics, or from the next step of a caller who asks
    for none; then the streaming kernels take over, until the one-launch form is
    asked for again."""
    import torch
    stats = (lambda h: h.last_solve_stats()) if name != "batch" else (lambda h: h.stats(0))
    for ask in ("stats", "next step"):
        g = LOST[name]()
        h = handle(g)
        form = name.split("_tol")[0].replace("batch", "one_launch")
        h.step(1.0 / 60.0)
        torch.cuda.synchronize()
        assert h.solve_form() == form
        h.set_resident_solve(4)
        with pytest.raises(RuntimeError, match="lost one of its workgroups"):
            h.step(1.0 / 60.0)
            h.step(1.0 / 60.0) if ask == "next step" and not name.endswith("tol") else None
            torch.cuda.synchronize()
            stats(h) if ask == "stats" else h.step(1.0 / 60.0)
        state = g.pos.cpu().numpy(), g.vel.cpu().numpy()
        outs = []
        for mode, want in ((None, "streaming"), (-1, form), (0, "streaming")):
            if mode is not None:
                h.set_resident_solve(mode)
            g.pos.copy_(torch.as_tensor(state[0]))
            g.vel.copy_(torch.as_tensor(state[1]))
            if name != "batch":
                h.set_warm_start(np.zeros((g.scene.n, 3)))
            h.step(1.0 / 60.0)
            stats(h)
            assert h.solve_form() == want
            outs.append(g.pos.cpu().numpy())
        if name != "batch":
            np.testing.assert_array_equal(outs[1], outs[0])
            np.testing.assert_array_equal(outs[2], outs[0])


def learned():
    from chysx.warmstart import load_params
    g = make_sim(mesh(130), tol=1e-6)
    g.sim.ws_set_params(load_params()[0])
    g.sim.set_warm_start_mode("learned")
    return g


# name: what is solved, the form of the step whose workgroups do not meet (one
# workgroup alone where the host does not wait, or in a batch), of the others
NOT_MET = {
    "waits": (lambda: make_sim(mesh(130), tol=1e-6), "streaming", "one_launch"),
    "enqueued": (lambda: make_sim(mesh(130), tol=0.0, max_iter=9), "one_launch", "one_launch"),
    "learned": (learned, "streaming", "one_launch"),
    "batch": (lambda: make_batch([mesh(w) for w in (130, 100, 20)], tol=1e-6), "one_launch", "one_launch"),
    "sweep_waits": (lambda: make_sim(mesh(520), tol=1e-4), "streaming", "sweep"),
    "sweep_enqueued": (lambda: make_sim(mesh(520), tol=0.0, max_iter=3), "sweep", "sweep"),
}


@pytest.mark.parametrize("name", NOT_MET)
def test_workgroups_that_do_not_meet(cuda, name):
    """A start-up wait of no length (mode 3), from the fourth step on: that step
    gives the same bits, the next ones stream, and the one-launch form comes
    back when it is asked for."""
    import torch
    make, missed, form = NOT_MET[name]
    outs = []
    for mode in (0, 3):
        g = make()
        h = handle(g)
        rows, forms = [], []
        for k in range(8):
            if k in (0, 3, 6):
                h.set_resident_solve(0 if mode == 0 else {0: -1, 3: 3, 6: -1}[k])
            h.step(1.0 / 60.0)
            torch.cuda.synchronize()
            forms.append(h.solve_form())
            rows += [g.pos.cpu().numpy(), g.vel.cpu().numpy()]
        outs.append(rows)
        assert forms == (["streaming"] * 8 if mode == 0 else [form] * 3 + [missed] + ["streaming"] * 2 + [form] * 2)
    for a, b in zip(*outs):
        np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("w", [20, 60, 530])
def test_step_on_a_stream_that_is_being_captured(cuda, w):
    """A fixed-count step with nothing enqueued before it runs at once, outside
    the captured graph; one that waits for its solve is refused and changes
    nothing."""
    import torch
    kw = dict(tol=0.0, max_iter=20)
    ref = make_sim(mesh(w), **kw)
    want = []
    for _ in range(4):
        ref.sim.step(1.0 / 60.0)
        want.append(ref.positions())
    g = make_sim(mesh(w), **kw)
    s = torch.cuda.Stream()
    g.sim.step(1.0 / 60.0, s.cuda_stream)
    assert g.sim.last_solve_stats()["iters"] == 20
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        x = torch.zeros(8, device="cuda")
        g.sim.step(1.0 / 60.0, s.cuda_stream)
        x += 1
    torch.cuda.synchronize()
    np.testing.assert_array_equal(g.positions(), want[1])
    assert g.sim.last_solve_stats()["iters"] == 20
    for _ in range(2):
        graph.replay()
        torch.cuda.synchronize()
        assert (x == 1).all()
    np.testing.assert_array_equal(g.positions(), want[1])
    g.sim.step(1.0 / 60.0, s.cuda_stream)
    torch.cuda.synchronize()
    np.testing.assert_array_equal(g.positions(), want[2])
    assert g.sim.last_solve_stats()["iters"] == 20
    g.sim.set_blocking_step(True)
    other = torch.cuda.CUDAGraph()
    with torch.cuda.graph(other, stream=s):
        x = torch.zeros(8, device="cuda")
        with pytest.raises(RuntimeError, match="being captured"):
            g.sim.step(1.0 / 60.0, s.cuda_stream)
    other.replay()
    g.sim.step(1.0 / 60.0, s.cuda_stream)
    torch.cuda.synchronize()
    np.testing.assert_array_equal(g.positions(), want[3])


def test_other_solves_beside_a_step_on_a_captured_stream(cuda):
    """A step that runs at once on a stream under capture leaves the other
    cloths' solves on other streams as they are."""
    import torch
    kw = dict(tol=0.0, max_iter=20)
    ref = make_sim(mesh(130), **kw)
    for _ in range(3):
        ref.sim.step(1.0 / 60.0)
    a, b = make_sim(mesh(130), **kw), make_sim(mesh(130), **kw)
    s, t = torch.cuda.Stream(), torch.cuda.Stream()
    for g, q in ((a, s), (b, t)):
        g.sim.step(1.0 / 60.0, q.cuda_stream)
        g.sim.last_solve_stats()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        x = torch.zeros(8, device="cuda")
        a.sim.step(1.0 / 60.0, s.cuda_stream)
    b.sim.step(1.0 / 60.0, t.cuda_stream)
    b.sim.step(1.0 / 60.0, t.cuda_stream)
    a.sim.step(1.0 / 60.0, s.cuda_stream)
    torch.cuda.synchronize()
    for g in (a, b):
        np.testing.assert_array_equal(g.positions(), ref.positions())
