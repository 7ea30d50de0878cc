"""The one-pass step over long marches and large coefficient tables.

The chunk is picked by the engine: the grids have so many tiles across y and z
that one round of blocks takes their whole length along x, up to the 32 planes
a block holds, with both x CPML faces in one march, its x0 to x1 hand-over, the
TF/SF box's x, y and z faces, the full rows of the profile, projection and
z-job tables and the psi values read a plane ahead.  The tables go to the 256
rows (64 with dispersive media) that a block holds, whose LDS passes 64 KiB.
FP64 against the oracle, the other types against the two passes, bit for bit.
"""
import re

import numpy as np
import pytest

import oracle
import xfdtd_cuda_amd as xf
from conftest import FIELDS
from test_gpu_step3 import DL, _box, _random, _same

pytestmark = pytest.mark.gpu

# cells, CPML, planes of a march
MARCHES = [
    ((19, 390, 370), (6,) * 6, 32),            # 32 planes: one march, both x faces in it
    ((18, 391, 365), (5, 7, 6, 6, 6, 6), 31),  # 31
    ((26, 390, 370), (6, 0, 6, 6, 6, 6), 7),   # 33 planes in marches of 7, the last of 5
    ((4, 390, 370), (2, 2, 6, 6, 6, 6), 9),    # 9: faces two planes thick, five between them
]
# materials, dispersive, rows of the table (pairs of E and H rows; 0: more than
# a block's table holds, the two passes run)
TABLES = [(50, False, 51), (200, False, 201), (255, False, 256), (256, False, 0), (62, True, 64), (63, True, 0)]


def _march(e, planes):
    d = e.describe()
    assert " step3=1" in d and f" step3_chunk={planes} " in d, d


@pytest.mark.parametrize("cells,pml,planes", MARCHES)
def test_marches_bit_identical_to_oracle(gpu_available, cells, pml, planes):
    steps = 5
    print(f"case: march {cells} {pml}", flush=True)
    tfsf = min(cells) > 10
    g, c = (_box(cells, pml, steps, tfsf=tfsf) for _ in range(2))
    _random(g, 1)
    _random(c, 1)
    e = xf.Engine(g).upload()
    _march(e, planes)
    e.run(1).run(steps - 1).download()
    e.close()
    oracle.run(c.scene_ptr(), steps)
    _same(g, c, f"{cells}")


@pytest.mark.parametrize("precision", ["fp32", "fp16", "bf16", "bf16c"])
@pytest.mark.parametrize("cells,pml,planes", MARCHES[:2])
def test_marches_match_two_passes(gpu_available, precision, cells, pml, planes):
    steps = 6
    print(f"case: march {precision} {cells} {pml}", flush=True)
    sims = []
    for one_pass in (True, False):
        s = _box(cells, pml, steps)
        _random(s, 2)
        e = xf.Engine(s, precision=precision).upload()
        if one_pass:
            _march(e, planes)
        else:
            e.set_tiling(tile_y=1, pml_split=False)
            assert " step3=0" in e.describe()
        e.run(2).run(steps - 2).download()
        e.close()
        sims.append(s)
    _same(sims[0], sims[1], precision)


def _tables(materials, steps, ade):
    """A box of `materials` cells of a row each, with CPML and a source."""
    s = xf.Simulation(DL, DL, DL, 0.9)
    n = 20
    s.add_cube("domain", (0, 0, 0), (n * DL,) * 3, xf.Material.air())
    if ade:
        s.add_sphere("d", (12 * DL, 12 * DL, 14 * DL), 4 * DL, xf.Material.drude(1.0, [1.2e10], [1.2e9]))
    for q in range(materials):
        s.add_cube(f"c{q}", (q % 18 * DL, q // 18 * DL, 2 * DL), (DL, DL, 3 * DL),
                   xf.Material.dielectric(1.5 + 0.01 * q, 1.0 + 0.002 * (q % 7), 1e-3 * (q % 3), 0.0))
    s.add_pml_all(4)
    s.add_point_source(2, (10, 9, 11), xf.Waveform.sine(3e9))
    s.set_coefficient_layout("dense")
    s.init(steps)
    return s


def _rows(e):
    return int(re.search(r" step3_rows=(\d+)", e.describe()).group(1))


@pytest.mark.parametrize("materials,ade,rows", TABLES)
def test_table_sizes(gpu_available, materials, ade, rows):
    steps = 12
    print(f"case: {materials} materials, ade={ade}", flush=True)
    g, c = _tables(materials, steps, ade), _tables(materials, steps, ade)
    e = xf.Engine(g).upload()
    if rows:
        assert _rows(e) == rows, e.describe()
    else:
        assert " step3=0" in e.describe(), e.describe()
    e.run(5).run(steps - 5).download()
    e.close()
    oracle.run(c.scene_ptr(), steps)
    for n in FIELDS:
        assert np.array_equal(g.array(n), c.array(n)), n
    if ade or not rows:
        return
    sims = []
    for one_pass in (True, False):
        s = _tables(materials, steps, ade)
        e = xf.Engine(s, precision="fp32").upload()
        if not one_pass:
            e.set_tiling(tile_y=1)
        assert (" step3=1" in e.describe()) == one_pass
        e.run(steps).download()
        e.close()
        sims.append(s)
    for n in FIELDS:
        assert np.array_equal(sims[0].array(n), sims[1].array(n)), n
