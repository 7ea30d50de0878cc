"""Grids that the engine steps in two passes though they have the one-pass
form: the default tiling there, and the one-pass step beside it, against the
oracle, bit for bit."""
import numpy as np
import pytest

import oracle
import xfdtd_cuda_amd as xf
from test_gpu_step3 import _box, _random, _same

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cells,pml,tfsf", [
    ((150, 150, 31), 0, False),
    ((150, 150, 12), 4, True),
    ((120, 120, 58), 4, True),
    ((3, 320, 320), 0, False),
    ((320, 2, 320), 0, False),
])
def test_default_of_a_slab_bit_identical_to_oracle(gpu_available, cells, pml, tfsf):
    steps = 5
    print(f"case: slab {cells} {pml} {tfsf}", flush=True)
    c = _box(cells, (pml,) * 6, steps, tfsf=tfsf, material=False)
    _random(c, 6)
    oracle.run(c.scene_ptr(), steps)
    for graph in (False, True):
        g = _box(cells, (pml,) * 6, steps, tfsf=tfsf, material=False)
        _random(g, 6)
        e = xf.Engine(g, use_graph=graph).upload()
        assert "step3=0" in e.describe()
        e.run(1).run(steps - 1).download()
        e.close()
        _same(g, c, f"{cells} graph={graph}")


def test_default_of_a_batch_of_slabs_matches_grids_alone(gpu_available):
    steps = 7
    print("case: batch of slabs, FP32", flush=True)
    build = lambda: [_box((150, 150, 12), (4,) * 6, steps, material=False),
                     _box((151, 149, 13), (4,) * 6, steps, material=False),
                     _box((150, 150, 14), (4,) * 6, steps, material=False)]
    sims, alone = build(), build()
    for q, (a, b) in enumerate(zip(sims, alone)):
        _random(a, 30 + q)
        _random(b, 30 + q)
    b = xf.Batch(sims, precision="fp32").upload()
    assert "step3=0" in b.describe()
    b.run(3).run(steps - 3).download()
    b.close()
    for q, (a, s) in enumerate(zip(sims, alone)):
        e = xf.Engine(s, precision="fp32").upload()
        assert "step3=1" in e.describe()
        e.run(steps).download()
        e.close()
        _same(a, s, f"grid {q}")
