"""A tuning run that fails (here: the watchdog finds an overflowed 16-bit
field in the first trial; the random state and the source stay below 4e3 in
the run's own steps and pass that storage's 65504 within thirty) leaves the
handle as it was: the same tiling, graphs and state, and later steps equal
those of a handle that was never tuned, bit for bit."""
import numpy as np
import pytest

import xfdtd_cuda_amd as xf
from conftest import FIELDS

pytestmark = pytest.mark.gpu
RUN = 6


def _box(seed, steps=100, n=16):
    s = xf.Simulation(5e-3, 5e-3, 5e-3, 0.9)
    s.add_cube("domain", (0.0, 0.0, 0.0), (n * 5e-3,) * 3, xf.Material.air())
    s.add_pml_all(4)
    f = 4e9
    s.add_point_source(2, (12, 12, 12), xf.Waveform.cosine_modulated_gaussian(1 / f, 2 / f, f), 1e5)
    s.init(steps)
    rng = np.random.default_rng(seed)
    for q in FIELDS:
        a = s.array(q)
        a[...] = rng.uniform(-1, 1, a.shape) * (1.0 if q[0] == "e" else 2e-3)
    return s


def _untuned(seed, hand, runs):
    s = _box(seed)
    e = xf.Engine(s, precision="fp16").upload()
    if hand:
        e.set_tiling(tile_y=2)
    for n in runs:
        e.run(n)
    e.download()
    e.close()
    return s


def _same(a, b):
    for n in FIELDS:
        x, y = a.array(n), b.array(n)
        assert np.isfinite(x).all() and np.array_equal(x, y), n


@pytest.mark.parametrize("graph", [False, True])
@pytest.mark.parametrize("hand", [False, True])
def test_batch(gpu_available, hand, graph):
    print(f"case: failing autotune, batch, hand={hand} graph={graph}", flush=True)
    sims = [_box(1), _box(2)]
    b = xf.Batch(sims, precision="fp16", watchdog=1, use_graph=graph)
    if hand:
        b.set_tuning(tile_y=2, planes=3)
    b.upload().run(3)
    before = b.describe(), b.tuning()
    assert ("step3=0" if hand else "step3=1") in before[0]
    with pytest.raises(xf.XFError, match=r"status 6\).*non-finite"):
        b.autotune(trial_steps=60)
    assert (b.describe(), b.tuning()) == before
    b.run(2).run(1).download()
    b.close()
    for q, s in enumerate(sims):
        _same(s, _untuned(q + 1, hand, (RUN,)))


@pytest.mark.parametrize("graph", [False, True])
@pytest.mark.parametrize("hand", [False, True])
def test_engine(gpu_available, hand, graph):
    print(f"case: failing autotune, engine, hand={hand} graph={graph}", flush=True)
    s = _box(3)
    e = xf.Engine(s, precision="fp16", watchdog=1, use_graph=graph).upload()
    if hand:
        e.set_tiling(tile_y=2)
    e.run(3)
    before = e.describe()
    with pytest.raises(xf.XFError, match=r"status 6\).*non-finite"):
        e.autotune(trial_steps=60)
    assert e.describe() == before
    e.run(2).run(1).download()
    e.close()
    _same(s, _untuned(3, hand, (RUN,)))
