"""Who holds a second set of fields, and what becomes of it when memory is
short: the engine's host code on a runtime in host memory with a limit
(cpp/fake_hip.cpp), a process a test.  The kernels do nothing there, so what
a download brings back is what was uploaded."""
import os
import subprocess
import sys
import textwrap

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)

PROLOGUE = """
import ctypes, sys
fake = ctypes.CDLL({fake!r}, mode=ctypes.RTLD_GLOBAL)
fake.fake_limit.argtypes = [ctypes.c_size_t]
fake.fake_used.restype = ctypes.c_size_t
sys.path.insert(0, {root!r})
import numpy as np
import xfdtd_cuda_amd as xf
FIELDS = ("ex", "ey", "ez", "hx", "hy", "hz")

def scene(n, seed=0, rows=0, pml=3):
    s = xf.Simulation(1e-3, 1e-3, 1e-3, 0.9)
    s.add_cube("domain", (0, 0, 0), (n * 1e-3,) * 3, xf.Material.air())
    for q in range(rows):  # a coefficient row each
        s.add_cube(f"c{{q}}", ((q % n) * 1e-3, (q // n % n) * 1e-3, 0), (1e-3,) * 3, xf.Material.dielectric(1.5 + 0.01 * q))
    if pml:
        s.add_pml_all(pml)
    s.set_coefficient_layout("dense" if rows else "compact")
    s.init(20)
    rng = np.random.default_rng(seed)
    for f in FIELDS:
        a = s.array(f)
        a[...] = rng.uniform(-1, 1, a.shape)
    return s

def saved(s):
    return [s.array(f).copy() for f in FIELDS]

def cost(make):
    fake.fake_limit(1 << 40)
    before = fake.fake_used()
    x = make()
    bytes = fake.fake_used() - before
    x.close()
    assert fake.fake_used() == before
    return bytes

def step3(x):
    return " step3=1" in x.describe()
"""


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("fake") / "fake_hip.so")
    r = subprocess.run([os.environ.get("CXX", "g++"), "-std=c++17", "-O1", "-shared", "-fPIC", "-o", out,
                        os.path.join(HERE, "cpp", "fake_hip.cpp")], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    return out


def _run(fake, code):
    r = subprocess.run([sys.executable, "-c", PROLOGUE.format(fake=fake, root=ROOT) + textwrap.dedent(code)],
                       capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr


def test_batch_that_fits_without_second_sets_is_uploaded(fake):
    """Grids' second sets come after every grid's own arrays: a batch that
    fits without them is never refused because of them."""
    _run(fake, """
    def batch(split=True):
        b = xf.Batch([scene(20 + q, q) for q in range(6)])
        if not split:
            b.set_tuning(tile_y=1)
        return b.upload()
    bare = cost(lambda: batch(False))
    full = cost(batch)
    assert full > 1.5 * bare, (bare, full)
    for room in (bare + 4096, int(1.3 * bare), int(2 * bare), 8 * bare):
        fake.fake_limit(room)
        sims = [scene(20 + q, q) for q in range(6)]
        want = [saved(s) for s in sims]
        b = xf.Batch(sims).upload()
        assert step3(b) == (room == 8 * bare), b.describe()
        b.run(3).run(2).download()
        for s, w in zip(sims, want):
            assert all(np.array_equal(x, y) for x, y in zip(saved(s), w))
        b.close()
    """)


def test_no_second_set_where_the_tiling_rules_it_out(fake):
    _run(fake, """
    bare = cost(lambda: xf.Engine(scene(24), tile_y=1).upload())
    full = cost(lambda: xf.Engine(scene(24)).upload())
    assert full > 1.6 * bare, (bare, full)
    s = scene(24)
    want = saved(s)
    start = fake.fake_used()
    e = xf.Engine(s, tile_y=1).upload()
    assert not step3(e)
    e.set_tiling()
    assert step3(e) and fake.fake_used() - start == full
    e.run(3)  # the fields are in the second set now, which has to be the one that stays
    e.set_tiling(tile_y=2)
    assert not step3(e) and fake.fake_used() - start == bare
    e.run(2).download()
    assert all(np.array_equal(x, y) for x, y in zip(saved(s), want))
    e.set_tiling()
    assert step3(e) and fake.fake_used() - start == full
    e.autotune(2)
    e.run(2).download()
    assert all(np.array_equal(x, y) for x, y in zip(saved(s), want))
    e.close()
    assert fake.fake_used() == start
    """)


def test_no_second_set_in_a_batch_with_a_grid_that_lacks_the_form(fake):
    _run(fake, """
    def batch(hand):
        b = xf.Batch([scene(20), scene(18, rows=300), scene(22)])
        return (b.set_tuning(tile_y=1) if hand else b).upload()
    assert cost(lambda: batch(False)) == cost(lambda: batch(True))
    sims = [scene(20), scene(22)]
    want = [saved(s) for s in sims]
    b = xf.Batch(sims, use_graph=True).upload()
    assert step3(b)
    held = fake.fake_used()
    b.run(3)
    b.set_tuning(tile_y=1)
    assert not step3(b) and fake.fake_used() < held
    b.run(3).download()
    best = b.autotune(2)
    b.run(3).download()
    for s, w in zip(sims, want):
        assert all(np.array_equal(x, y) for x, y in zip(saved(s), w))
    # uploaded again, it takes them again
    assert step3(b)
    b.upload().run(1)
    assert step3(b) and fake.fake_used() == held
    b.close()
    """)


def test_a_failing_allocation_has_idle_handles_give_theirs_back(fake):
    """Handles that fit the device without second sets all fit it, whichever
    came first, and go on stepping."""
    _run(fake, """
    bare = cost(lambda: xf.Engine(scene(24), tile_y=1).upload())
    fake.fake_limit(int(8.2 * bare))
    sims = [scene(24, q) for q in range(9)]
    want = [saved(s) for s in sims]
    e = [xf.Engine(sims[0], use_graph=True).upload(), xf.Engine(sims[1]).upload()]
    assert step3(e[0]) and step3(e[1])
    e[0].run(3)  # its fields are in the second set, which stays
    e[1].run(2)
    b = xf.Batch(sims[2:4]).upload()
    assert step3(b) == (2 * bare < (8.2 - 5.5) / 4 * bare)
    for s in sims[4:8]:
        e.append(xf.Engine(s).upload())
    assert not step3(e[0]) and not step3(e[1]) and not step3(e[-1])
    try:
        xf.Engine(sims[8]).upload()
        raise SystemExit("nine grids cannot fit")
    except xf.XFError as err:
        assert "status 5" in str(err), err
    for x in e + [b]:
        x.run(3).run(2).download()
    for s, w in zip(sims[:8], want):
        assert all(np.array_equal(x, y) for x, y in zip(saved(s), w))
    e.pop().close()
    e[0].set_tiling()  # room again
    fake.fake_limit(1 << 40)
    e[0].set_tiling()
    assert step3(e[0])
    """)


def test_a_batch_gives_its_sets_back(fake):
    _run(fake, """
    bare = cost(lambda: xf.Batch([scene(24, q) for q in range(3)]).set_tuning(tile_y=1).upload())
    sims = [scene(24, q) for q in range(6)]
    want = [saved(s) for s in sims]
    fake.fake_limit(5 * bare)
    b = xf.Batch(sims[:3], use_graph=True).upload()
    assert step3(b)
    b.run(3)
    fake.fake_limit(int(2.1 * bare))
    c = xf.Batch(sims[3:]).upload()
    assert not step3(b) and not step3(c)
    b.run(2).run(3).download()
    c.run(2).download()
    for s, w in zip(sims, want):
        assert all(np.array_equal(x, y) for x, y in zip(saved(s), w))
    c.close()
    # its own snapshots come before its second sets
    fake.fake_limit(5 * bare)
    b.upload()
    assert step3(b)
    fake.fake_limit(int(2.1 * bare))
    b.autotune(2)
    assert not step3(b)
    b.run(3).download()
    for s, w in zip(sims[:3], want):
        assert all(np.array_equal(x, y) for x, y in zip(saved(s), w))
    """)


def test_threads_fill_the_device(fake):
    """Handles made, run and closed by several threads under a limit that is
    short of second sets for all."""
    _run(fake, """
    import threading
    bare = cost(lambda: xf.Engine(scene(16), tile_y=1).upload())
    fake.fake_limit(int(5.5 * bare))
    errors = []
    def work(q):
        try:
            for turn in range(12):
                s = scene(16, q)
                w = saved(s)
                e = xf.Engine(s).upload()
                e.run(3).describe()
                e.run(2).download()
                assert all(np.array_equal(x, y) for x, y in zip(saved(s), w))
                e.close()
        except Exception as err:
            errors.append(repr(err))
    ts = [threading.Thread(target=work, args=(q,)) for q in range(4)]
    for t in ts: t.start()
    for t in ts: t.join()
    assert not errors, errors
    """)
