"""Parity at the benchmarked sizes on the paths that a default run no longer
takes there: the 536^3 FP64 sphere by the two passes' own default tiling
(z-face CPML at the end of each 3-plane, 32-lane tile), and the 64-grid batch
by the two passes; both against the CPU oracle, bit for bit, from a random
state.  That the default is the one-pass step at these sizes is asserted here
too."""
import pytest

import oracle
import xfdtd_cuda_amd as xf
from xfdtd_cuda_amd import scenes
from test_gpu_full_size import _assert_same, _randomise

pytestmark = pytest.mark.gpu


def test_full_size_sphere_two_pass_z_tail(gpu_available):
    steps = 3
    print("case: 536^3 FP64 sphere, random state, 3 steps, two passes with the z tail", flush=True)
    g, c = (scenes.large_sphere(n=512, pml=12, steps=steps + 1, layout="compact") for _ in range(2))
    _randomise([g, c], 22)
    e = xf.Engine(g).upload()
    assert " step3=1 step3_chunk=32 " in e.describe(), e.describe()
    e.set_tiling(chunks_x=179, pml_ztail=True, k32=True)
    d = e.describe()
    assert " step3=0" in d and " pml_ztail=1" in d and " klanes=32" in d and " chunk=3 " in d, d
    e.run(1).run(steps - 1).download()
    e.close()
    oracle.run(c.scene_ptr(), steps)
    assert _assert_same(g, c, "536^3 z tail") > 6 + 24


def test_full_size_batch_two_pass(gpu_available):
    steps = 2
    print("case: 64-grid batch FP64, random state, 2 steps, two passes", flush=True)
    gs, cs = (scenes.batch_spheres(count=64, steps=steps + 1) for _ in range(2))
    for q, (g, c) in enumerate(zip(gs, cs)):
        _randomise([g, c], 200 + q)
    b = xf.Batch(gs, precision="fp64").upload()
    assert " step3=1" in b.describe(), b.describe()
    b.set_tuning()
    assert " step3=0" in b.describe(), b.describe()
    b.run(steps).download()
    b.close()
    for c in cs:
        oracle.run(c.scene_ptr(), steps)
    for q, (g, c) in enumerate(zip(gs, cs)):
        _assert_same(g, c, f"batch grid {q}")
