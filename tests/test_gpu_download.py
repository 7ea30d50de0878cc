"""What xf_download brings back, through both kinds of staging (ordinary
memory below 48 MiB, pinned slots above) and cut at slot ends: the state as
uploaded, to the rounding of its storage type."""
import threading

import numpy as np
import pytest

import xfdtd_cuda_amd as xf

pytestmark = pytest.mark.gpu
DL = 1e-2
FIELDS = ("ex", "ey", "ez", "hx", "hy", "hz")
PSI = ("ea_psi_hb", "eb_psi_ha", "ha_psi_eb", "hb_psi_ea")


def _scene(cells, pml):
    s = xf.Simulation(DL, DL, DL, 0.95)
    half = [c * DL / 2 for c in cells]
    s.add_cube("domain", [-h for h in half], [2 * h for h in half], xf.Material.air())
    for face in ("XN", "YP", "ZP"):
        if pml:
            s.add_pml(pml, face)
    s.set_coefficient_layout("compact")
    s.init(4)
    return s


def _names(pml):
    return list(FIELDS) + [f"pml.{p}.{m}" for p in range(3 if pml else 0) for m in PSI]


def _round_trip(cells, pml, precision, seed):
    s = _scene(cells, pml)
    rng = np.random.default_rng(seed)
    want = {}
    for n in _names(pml):
        a = s.array(n)
        a[...] = rng.uniform(-1, 1, a.shape)
        want[n] = a.copy() if precision == "fp64" else a.astype(np.float32).astype(np.float64)
    e = xf.Engine(s, precision=precision).upload()
    for n in want:
        s.array(n)[...] = np.nan
    e.download()
    e.close()
    return [n for n in want if not np.array_equal(s.array(n), want[n])]


# 100 x 90 x 120 in FP64 is 52 MiB: pinned slots; 40^3 and less: ordinary memory
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("cells,pml", [((1, 1, 1), 0), ((3, 9, 5), 2), ((40, 33, 41), 4), ((94, 90, 120), 6), ((200, 100, 100), 5)])
def test_state_comes_back(cells, pml, precision):
    assert _round_trip(cells, pml, precision, 3) == []


def test_two_downloads_at_once():
    bad = {}
    ts = [threading.Thread(target=lambda q=q: bad.__setitem__(q, _round_trip((94, 90, 118 + q), 5, "fp64", q))) for q in range(3)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert bad == {0: [], 1: [], 2: []}
