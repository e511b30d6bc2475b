"""Host-side rules of the one-launch solves, compiled from their headers and run
on the CPU; no GPU is used."""

import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "ai-phyiscs_amd", "csrc")
NATIVE = os.path.join(ROOT, "tests", "native")


@pytest.fixture
def compiled(tmp_path):
    def build(name, *sources):
        exe = tmp_path / name
        subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-I" + CSRC,
                        os.path.join(NATIVE, name + ".cpp"), *(os.path.join(CSRC, s) for s in sources), "-o", str(exe)],
                       check=True)
        return subprocess.run([str(exe)], check=True, capture_output=True, text=True, timeout=120).stdout
    return build


def test_every_batch_comes_to_run(compiled):
    """No order of events leaves all started workgroups waiting for ones that cannot start."""
    rows = {r.split()[0]: [int(v) for v in r.split()[1:]] for r in compiled("places").splitlines()}
    assert len(rows) == 11
    for name, (by_start, stuck, _) in rows.items():
        assert stuck == 0, name
    # places in the order of starting do get stuck where the rule avoids them
    assert rows["two198"][0] == 0 and rows["two198"][2] > 0
    assert rows["sixteen130"][2] > 0
    assert rows["uneven16"][0] == 1 and rows["one256"][0] == 1


def test_batches_that_the_streaming_kernels_solve_faster(compiled):
    """What fits at once always goes in one launch; beyond, it depends on the use of the compute units."""
    rows = {r.split()[0]: [int(v) for v in r.split()[1:]] for r in compiled("min_iters").splitlines()}
    never = 2 ** 31 - 1
    for name in ("1x256", "5x44", "2000x1"):
        assert rows[name] == [0, 0]
    for name in ("3x130", "8x130", "16x130", "8x176"):  # measured 0.65 to 0.87 times as fast at 50 iterations
        assert rows[name] == [never, 2]
    for name in ("2x130", "16x64", "64x32", "128x20", "8x256", "4096x2"):  # 1.08 to 1.7 times as fast at 50
        assert 1 < rows[name][0] <= 25 and rows[name][1] == 2


def test_solves_in_flight_together_leave_room(compiled):
    """Launches that may be under way together never hold a whole XCD with waiting workgroups."""
    assert compiled("gate").startswith("ok ")


def test_steps_held_after_workgroups_did_not_meet(compiled):
    """None at first, then 1024 and twice as many at each miss, up to 65536; 1024 again after as many have met."""
    assert [int(v) for v in compiled("hold").split()] == [0, 1024, 2048, 4096, 8192, 16384, 32768, 65536, 65536, 65536, 1024]
