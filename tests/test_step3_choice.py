"""Which grids step in one pass: the rule's two sides at each of its lines,
the tuner's finding above the rule, and that finding kept by a new upload.
The engine's host code on a runtime in host memory (cpp/fake_hip.cpp), whose
device has 256 CUs and whose every run takes the same time, so that a tuner
keeps its first candidate, the one-pass step."""
import pytest

from test_second_sets import _run, fake  # noqa: F401

SCENE = """
def slab(cells, pml=0, tfsf=False):
    s = xf.Simulation(3e-3, 3e-3, 3e-3, 0.95)
    half = [c * 1.5e-3 for c in cells]
    s.add_cube("domain", [-h for h in half], [2 * h for h in half], xf.Material.air())
    if pml:
        s.add_pml_all(pml)
    if tfsf:
        s.add_tfsf3d((pml + 3,) * 3, 0.5, 0.9, 0.2, xf.Waveform.gaussian(1e-10, 2e-10))
    s.set_coefficient_layout("compact")
    s.init(4)
    return s
"""


@pytest.mark.parametrize("precision,cells,pml,tfsf,one_pass", [
    # at most 32 nodes along z in FP64, from six rounds of blocks on
    ("fp64", (150, 150, 31), 0, False, False),
    ("fp64", (150, 150, 32), 0, False, True),
    ("fp64", (100, 100, 20), 0, False, True),
    ("fp32", (150, 150, 20), 0, False, True),
    # the first of two tiles meets both ends' CPML: 65 to 68 nodes for 4 layers
    ("fp64", (150, 150, 55), 4, False, True),
    ("fp64", (150, 150, 56), 4, False, False),
    ("fp64", (150, 150, 64), 4, False, True),
    # FP32: a single tile too, if it is not full or has the TF/SF faces
    ("fp32", (240, 240, 39), 4, False, False),
    ("fp32", (240, 240, 40), 4, False, True),
    ("fp32", (240, 240, 40), 4, True, False),
    ("fp32", (200, 200, 39), 4, False, True),
    # narrow storage: TF/SF without CPML
    ("fp16", (160, 160, 160), 0, True, False),
    ("bf16c", (160, 160, 160), 0, True, False),
    ("fp16", (160, 160, 160), 0, False, True),
    ("fp16", (130, 130, 130), 0, True, True),
    # ... and large grids whose first tile meets both ends
    ("fp16", (280, 280, 56), 4, True, False),
    ("bf16c", (280, 280, 56), 4, True, True),
    # a few nodes across
    ("fp64", (3, 320, 320), 0, False, False),
    ("fp64", (4, 320, 320), 0, False, True),
    ("fp64", (320, 2, 320), 0, False, False),
    ("fp64", (320, 3, 320), 0, False, True),
])
def test_rule(fake, precision, cells, pml, tfsf, one_pass):  # noqa: F811
    _run(fake, SCENE + f"""
e = xf.Engine(slab({cells}, {pml}, {tfsf}), precision={precision!r}).upload()
assert step3(e) == {one_pass}, e.describe()
e.autotune(2)  # all take the same time here: the first it tries
assert step3(e), e.describe()
e.upload()
assert step3(e), e.describe()
e.set_tiling(tile_y=1)
assert not step3(e)
""")


@pytest.mark.parametrize("precision,one_pass", [("fp32", False), ("fp64", True), ("fp16", True)])
def test_rule_of_a_batch(fake, precision, one_pass):  # noqa: F811
    _run(fake, SCENE + f"""
b = xf.Batch([slab((150, 150, 20), 4) for q in range(3)], precision={precision!r}).upload()
assert step3(b) == {one_pass}, b.describe()
b.run(1)
b.autotune(2)
assert step3(b), b.describe()
b.upload().run(1)
assert step3(b), b.describe()
# most of the work is in the other kind of grid
b = xf.Batch([slab((150, 150, 20), 4)] + [slab((150, 150, 60), 4) for q in range(2)], precision={precision!r}).upload()
assert step3(b), b.describe()
""")
