"""The one-pass 3-D step (k_step3) against the oracle and the two-pass kernels.

The one-pass step forms every node's H and E with the two-pass kernels' own
expressions in their order, so FP64 must equal the oracle bit for bit, and
every other storage type the two-pass engine (an explicit tiling) bit for
bit.  The grids sit where the decomposition can go wrong: rows of j around
multiples of the six a block owns, k around multiples of its 64 lanes, chunks
of one plane and of all, more chunk remainders, grids smaller than a tile.
"""
import re

import numpy as np
import pytest

import oracle
import xfdtd_cuda_amd as xf
from xfdtd_cuda_amd import scenes
from conftest import FIELDS

pytestmark = pytest.mark.gpu

PSI = ("ea_psi_hb", "eb_psi_ha", "ha_psi_eb", "hb_psi_ea")
DL = 3e-3


def _box(cells, pml, steps, tfsf=True, kappa=1.0, material=True, angles=(0.5, 0.9, 0.2)):
    """A box of cells[d] interior cells along each axis with pml[f] CPML cells
    on face f, a lossy sphere, an oblique plane wave and a surface."""
    s = xf.Simulation(DL, DL, DL, 0.95)
    half = [c * DL / 2 for c in cells]
    s.add_cube("domain", [-h for h in half], [2 * h for h in half], xf.Material.air())
    if material:
        s.add_sphere("s", (0.3 * DL, -0.2 * DL, 0.1 * DL), 0.22 * min(cells) * DL,
                     xf.Material.dielectric(3.5, 1.3, 0.02, 0.5))
    for face, size in zip(xf.FACES, pml):
        if size:  # kappa stretches one face: each of its layers has rows of its own
            s.add_pml(size, face, kappa_max=kappa if face == "YP" else 1.0)
    m = max(pml)
    if tfsf:
        tau = 20 * DL / 6e8
        s.add_tfsf3d((m + 3,) * 3, *angles, xf.Waveform.gaussian(tau, 2.0 * tau))
        s.add_nf2ff_fd((m + 2,) * 3, [1e9, 2e9])
    s.set_coefficient_layout("compact" if not material else "dense")
    s.init(steps)
    return s


def _names(sim):
    names = list(FIELDS)
    for p in range(6):
        try:
            sim.array(f"pml.{p}.{PSI[0]}")
        except xf.XFError:
            break
        names += [f"pml.{p}.{m}" for m in PSI]
    for f in range(2):
        for face in xf.FACES:
            for c in ("ja", "jb", "ma", "mb"):
                try:
                    sim.array(f"nf2ff.0.{f}.{face}.{c}")
                except xf.XFError:
                    continue
                names.append(f"nf2ff.0.{f}.{face}.{c}")
    return names


def _random(sim, seed):
    """Every field value and every psi random (a state in which nothing is
    zero by symmetry), walls included."""
    rng = np.random.default_rng(seed)
    for n in _names(sim):
        a = sim.array(n)
        if a.size and not n.startswith("nf2ff"):
            a[...] = rng.uniform(-1, 1, a.shape) * (1.0 if n[0] == "e" else 1e-3)


def _same(a, b, label):
    for n in _names(b):
        x, y = a.array(n), b.array(n)
        assert np.array_equal(x, y), f"{label}: {n} differs at {int(np.sum(x != y))} of {x.size}"


@pytest.mark.parametrize("cells,pml", [
    ((20, 17, 51), (4, 4, 4, 4, 4, 4)),    # ny + 1 = 26, nz + 1 = 60
    ((19, 15, 55), (4, 4, 4, 4, 4, 4)),    # ny + 1 = 24: whole blocks; nz + 1 = 64: one tile
    ((21, 16, 56), (4, 4, 4, 4, 4, 4)),    # nz + 1 = 65: one lane in the second tile
    ((23, 22, 120), (3, 5, 4, 4, 2, 6)),   # nz + 1 = 129
    ((17, 19, 119), (4, 4, 4, 4, 4, 4)),   # nz + 1 = 128: the last tile is full
    ((16, 40, 16), (4, 0, 0, 3, 0, 5)),    # faces on some sides only
    ((40, 16, 18), (0, 0, 0, 0, 0, 0)),    # none
])
def test_step3_bit_identical_to_oracle(gpu_available, cells, pml):
    steps = 11
    print(f"case: step3 {cells} {pml}", flush=True)
    g, c = _box(cells, pml, steps), _box(cells, pml, steps)
    _random(g, 1)
    _random(c, 1)
    e = xf.Engine(g).upload()
    assert "step3=1" in e.describe()
    e.run(1).run(4).run(steps - 5).download()
    e.close()
    oracle.run(c.scene_ptr(), steps)
    _same(g, c, f"{cells}")


@pytest.mark.parametrize("cells,pml", [((1, 1, 1), 0), ((2, 5, 3), 0), ((5, 2, 70), 1), ((3, 7, 63), 1)])
def test_step3_small_grids(gpu_available, cells, pml):
    """Grids smaller than a tile, without a source."""
    steps = 9
    print(f"case: step3 small {cells}", flush=True)
    faces = (0, 0, 0, 0, 0, 0) if not pml else (pml, pml, 0, 0, pml, pml)
    g = _box(cells, faces, steps, tfsf=False, material=False)
    c = _box(cells, faces, steps, tfsf=False, material=False)
    _random(g, 2)
    _random(c, 2)
    e = xf.Engine(g).upload()
    assert "step3=1" in e.describe()
    e.run(steps).download()
    e.close()
    oracle.run(c.scene_ptr(), steps)
    _same(g, c, f"{cells}")


@pytest.mark.parametrize("precision", ["fp32", "fp16", "bf16", "bf16c"])
@pytest.mark.parametrize("cells,pml", [((20, 17, 51), (4, 4, 4, 4, 4, 4)), ((13, 27, 57), (4, 0, 3, 4, 0, 4))])
def test_step3_precisions_match_two_pass(gpu_available, precision, cells, pml):
    steps = 12
    print(f"case: step3 {precision} {cells}", flush=True)
    sims = []
    for one_pass in (True, False):
        s = _box(cells, pml, steps)
        _random(s, 3)
        e = xf.Engine(s, precision=precision).upload()
        if not one_pass:
            e.set_tiling(tile_y=1, pml_split=False)
        assert ("step3=1" in e.describe()) == one_pass
        e.run(5).run(steps - 5).download()
        e.close()
        sims.append(s)
    _same(sims[0], sims[1], precision)


def test_step3_graph_and_change_of_tiling(gpu_available):
    """Odd runs of a captured step (the two sets have a graph each), and runs
    that change between the one-pass and the two-pass kernels."""
    build = lambda: _box((18, 21, 30), (4,) * 6, 40, kappa=2.0)
    c = build()
    _random(c, 4)
    oracle.run(c.scene_ptr(), 29)
    for graph in (False, True):
        g = build()
        _random(g, 4)
        e = xf.Engine(g, use_graph=graph).upload()
        e.run(3).run(4)
        e.download()
        e.set_tiling(tile_y=2)
        e.run(5)
        e.set_tiling()
        assert "step3=1" in e.describe()
        e.run(7).run(10).download()
        e.close()
        _same(g, c, f"graph={graph}")


def test_step3_dispersive_and_wall_sources(gpu_available):
    steps = 30
    g, c = (scenes.dispersive_sphere(n=26, pml=5, steps=steps, freqs=(1e9,)) for _ in range(2))
    e = xf.Engine(g).upload()
    assert "step3=1" in e.describe()
    e.run(13).run(steps - 13).download()
    e.close()
    oracle.run(c.scene_ptr(), steps)
    for n in FIELDS + ("ade.jx", "ade.jy", "ade.jz"):
        assert np.array_equal(g.array(n), c.array(n)), n

    # sources on an outer wall: a node no pass updates keeps what it gains
    def walls():
        s = xf.Simulation(DL, DL, DL, 0.9)
        s.add_cube("domain", (0, 0, 0), (12 * DL, 13 * DL, 14 * DL), xf.Material.air())
        w = xf.Waveform.sine(3e9)
        s.add_point_source(2, (0, 0, 3), w).add_point_source(0, (4, 13, 14), w, 0.5)
        s.add_point_source(1, (6, 5, 7), w)
        s.init(steps)
        return s

    g, c = walls(), walls()
    e = xf.Engine(g).upload()
    e.run(7).run(steps - 7).download()
    e.close()
    oracle.run(c.scene_ptr(), steps)
    _same(g, c, "walls")


@pytest.mark.parametrize("graph", [False, True])
def test_step3_batch_matches_grids_alone(gpu_available, graph):
    """Grids of different sizes, CPML and sources in one launch, against the
    oracle grid by grid."""
    steps = 21
    shapes = [((20, 17, 51), (4,) * 6, True), ((5, 9, 12), (0,) * 6, False), ((13, 27, 57), (4, 0, 3, 4, 0, 4), True)]
    sims = [_box(c, p, steps, tfsf=t) for c, p, t in shapes]
    ref = [_box(c, p, steps, tfsf=t) for c, p, t in shapes]
    for q, (a, b) in enumerate(zip(sims, ref)):
        _random(a, 10 + q)
        _random(b, 10 + q)
    b = xf.Batch(sims, use_graph=graph).upload()
    assert "step3=1" in b.describe()
    b.run(4).run(7)
    b.download()
    b.set_tuning(tile_y=1)
    assert "step3=0" in b.describe()
    b.run(steps - 11).download()
    b.close()
    for q, (x, y) in enumerate(zip(sims, ref)):
        oracle.run(y.scene_ptr(), steps)
        _same(x, y, f"grid {q}")


def test_step3_table_limit(gpu_available):
    """More coefficient rows than the block's table holds: the two-pass kernels
    run, with the same results."""
    def build():
        s = xf.Simulation(DL, DL, DL, 0.9)
        s.add_cube("domain", (0, 0, 0), (12 * DL, 12 * DL, 12 * DL), xf.Material.air())
        for q in range(270):
            i, j, k = q % 12, (q // 12) % 12, q // 144 * 4
            s.add_cube(f"c{q}", (i * DL, j * DL, k * DL), (DL, DL, 4 * DL), xf.Material.dielectric(1.5 + 0.01 * q))
        s.add_point_source(2, (6, 5, 7), xf.Waveform.sine(3e9))
        s.init(20)
        return s

    g, c = build(), build()
    e = xf.Engine(g).upload()
    rows = int(re.search(r"etab=(\d+)", e.describe()).group(1))
    assert rows > 256 and "step3=0" in e.describe(), e.describe()
    e.run(20).download()
    e.close()
    oracle.run(c.scene_ptr(), 20)
    _same(g, c, "table limit")
