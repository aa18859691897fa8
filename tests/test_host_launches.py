"""The host side of the step calls on a HIP runtime that runs nothing and
writes down what it is asked for (tests/fake_hip): what is launched, captured,
replayed and waited for.  No GPU and no GPU code: the results of captured and
of direct steps are compared on the device by test_gpu_graph_lengths.py."""
import json
import os
import shutil
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")

pytestmark = pytest.mark.skipif(shutil.which("g++") is None, reason="no host compiler")


@pytest.fixture(scope="module")
def run(tmp_path_factory):
    lib = str(tmp_path_factory.mktemp("fake_hip") / "libfake_hip.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-pthread", "-D__HIP_PLATFORM_AMD__",
                    f"-I{ROCM}/include", os.path.join(HERE, "fake_hip", "fake_hip.cpp"), "-o", lib], check=True)

    def go(script):
        r = subprocess.run([sys.executable, os.path.join(HERE, "fake_hip", "launches.py"), lib], input=script,
                           capture_output=True, text=True, timeout=120)
        assert r.returncode == 0, r.stderr[-4000:]
        return json.loads(r.stdout)

    return go


# launches a step, steps a graph, launches before a call's first step
SHAPE = {"periodic": (3, 16, 0), "slab": (3, 16, 0), "reference": (3, 16, 2), "weno7": (5, 9, 0),
         "heat13": (1, 48, 0)}
DIRECT = 50  # graphs' worth of steps launched before a capture
# steps of a call long enough to be captured (heat7: 4 steps a launch)
LONG = {**{k: (DIRECT + 1) * per + 4 for k, (_, per, _) in SHAPE.items()}, "heat7": (DIRECT + 1) * 48 * 4 + 11}


@pytest.mark.parametrize("kind", LONG)
def test_short_call_waits_for_another_threads_capture(run, kind):
    """Two host threads on one stream: steps that one launches must not be
    recorded into the graph that the other captures."""
    log = run(f"""
fake.fake_hold_captures(400)
t = threading.Thread(target=call, args=({kind!r}, {LONG[kind]}))
t.start()
while not fake.fake_captures_open() and t.is_alive():
    time.sleep(0.001)
opened = fake.fake_captures_open()
rc = call({kind!r}, 3)
t.join()
out = [opened, rc, log()]
""")
    assert log[:2] == [1, 0] and "n" in log[2]
    assert "x" not in log[2]


@pytest.mark.parametrize("n", [0, 3, 16, 18])
@pytest.mark.parametrize("kind", ["batch", "serial"])
def test_batch_calls_with_a_graph_return_when_the_steps_have_ended(run, kind, n):
    with_graph, without = run(f"""
assert call({kind!r}, {n}) == 0
a = log()
assert call({kind!r}, {n}, graph=0) == 0
out = [a, log()]
""")
    assert with_graph.endswith("W")
    assert "W" not in without


@pytest.mark.parametrize("kind", [*LONG, "batch", "serial"])
def test_graph_calls_are_refused_while_the_caller_captures(run, kind):
    """Whatever their length, and without a trace in the caller's capture;
    without a graph the same steps are recorded into it."""
    out = run(f"""
def under_capture(n, graph):
    g = ctypes.c_void_p()
    fake.hipStreamBeginCapture(0x77, 0)
    rc = call({kind!r}, n, graph)
    fake.hipStreamEndCapture(0x77, ctypes.byref(g))
    return rc, log()
out = [under_capture(2, 1), under_capture(250, 1), under_capture(2, 0)]
""")
    assert out[0] == [3, "[]"] and out[1] == [3, "[]"]  # MGAD_ERR_HIP
    assert out[2][0] == 0 and "n" in out[2][1]


@pytest.mark.parametrize("kind", SHAPE)
def test_runs_are_captured_after_fifty_graphs_of_direct_steps(run, kind):
    """Short runs never capture; a longer one does while the device still has
    work, in whichever call it gets there, and replays from then on."""
    per_step, per, pre = SHAPE[kind]
    lead = DIRECT * per
    calls = [lead - 2, per + 6, per + 4, 1]
    *log, other, short = run(f"""
out = []
for n in {calls}:
    assert call({kind!r}, n) == 0
    out.append(log())
assert call({kind!r}, {lead + 2 * per + 4}, u=0x800000) == 0
out.append(log())
for _ in range({DIRECT + 2}):
    assert call({kind!r}, {per - 1}, u=0x900000) == 0
out.append(log())
""")
    def direct(steps):
        return "L" * (steps * per_step)

    head, nodes = "L" * pre, per * per_step
    graph, replay = "[" + "n" * nodes + "]", f"R{nodes};"
    assert log[0] == head + direct(lead - 2)
    assert log[1] == head + direct(2) + graph + replay + direct(4)
    assert log[2] == head + replay + direct(4)
    assert log[3].count("L") == pre + per_step and "R" not in log[3]
    assert other == head + direct(lead) + graph + 2 * replay + direct(4)
    assert "[" not in short


@pytest.mark.parametrize("kind,per_step", [("batch", 3), ("serial", 6)])
def test_batch_call_captures_only_what_it_replays_itself(run, kind, per_step):
    lead = DIRECT * 48
    short, long, execs = run(f"""
assert call({kind!r}, {lead // per_step}) == 0
a = log()
assert call({kind!r}, {(lead + 192) // per_step + 1}) == 0
out = [a, log(), fake.fake_live_execs()]
""")
    assert short == "L" * lead + "W"
    assert long == "L" * lead + "[" + "n" * 48 + "]" + 4 * "R48;" + "L" * per_step + "W"
    assert execs == 0


def test_full_cache_makes_room(run):
    """Keys without a graph go without a wait; graphs are destroyed after one."""
    one, kept, full, execs = run(f"""
for i in range(100):
    assert call("periodic", 20, u=0x1000000 + 0x1000 * i) == 0
a = log()
for i in range(33):
    assert call("periodic", {LONG["periodic"]}, u=0x2000000 + 0x1000 * i) == 0
b = log()
assert call("periodic", 20) == 0
out = [a, b, log(), fake.fake_live_execs()]
""")
    assert set(one) == {"L"}
    assert kept.count("[") == 33 and "D" not in kept
    assert full == "D" + "L" * 60 and execs == 0


def test_heat7_graph_does_not_grow_with_the_call(run):
    """One graph of 48 launches whatever the number of steps, kept for calls of
    any other number."""
    first, second, third = run("""
assert call("heat7", 100003) == 0
a = log()
assert call("heat7", 50000) == 0
b = log()
assert call("heat7", 195) == 0
out = [a, b, log()]
""")
    graph = "[" + "n" * 48 + "]"
    assert first.count("[") == 1 and graph in first and first.count("L") < (DIRECT + 2) * 48
    assert "[" not in second and second.startswith("R48;") and second.count("L") < 2 * 48
    assert "C" not in first + second  # an even number of launches: nothing to copy back
    assert "[" not in third


@pytest.mark.parametrize("nx,ny", [(n, 1) for n in (2**31 - 1, 2**31 - 34, 2**31 - 35)]
                         + [(1, n) for n in (2**31 - 1, 2**31 - 32)] + [(7, 2**31 // 7), (3, 2), (100, 100)])
def test_small_tiles_of_any_accepted_side(nx, ny):
    """The 256-thread tile of a grid (WENO7 takes sides up to 2^31 - 1): at most
    256 columns, sides that sum to at most 42, and blocks that cover the grid."""
    import ctypes

    from multigpu_advectiondiffusion_amd import _capi

    tx, ty = ctypes.c_int(), ctypes.c_int()
    _capi.lib()._ZN4mgad10small_tileEiiRiS0_(nx, ny, ctypes.byref(tx), ctypes.byref(ty))
    x, y = tx.value, ty.value
    assert 1 <= x <= 34 and 1 <= y <= 34 and x * y <= 256 and x + y <= 42
    assert -(-nx // x) * -(-ny // y) <= -(-nx // 16) * -(-ny // 16)


@pytest.mark.parametrize("shape,groups", [((16, 16, 200), 100), ((27, 11, 441), 222), ((32, 32, 512), 512),
                                          ((16, 16, 64), 64), ((32, 32, 32), 128)])
def test_thin_periodic_grids_fill_the_device(run, shape, groups):
    """Columns of more than 128 one-plane bands get the next depth."""
    assert run(f"""
assert call("periodic", 1, graph=0, **dict(zip(("nx", "ny", "nz"), {shape}))) == 0
out = fake.fake_last_groups()
""") == groups
