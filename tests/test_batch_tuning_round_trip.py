"""A batch's tuning says whether it steps in one pass, and set again, on this
batch or another, it selects the same step.  The engine's host code on a
runtime in host memory (cpp/fake_hip.cpp), whose tuner keeps the one-pass step
(every run takes the same time there, and it is tried first)."""
from test_second_sets import _run, fake  # noqa: F401


def test_tuning_round_trip(fake):  # noqa: F811
    _run(fake, """
    def again(b, t):
        return b.set_tuning(**{k: v for k, v in t.items() if k != "step_ms"})
    sims = [scene(20, q) for q in range(2)]
    want = [saved(s) for s in sims]
    b = xf.Batch(sims, use_graph=True).upload()
    assert step3(b)
    b.run(1)
    mine = b.tuning()
    again(b, mine)
    assert step3(b) and b.tuning() == mine
    best = b.autotune(2)
    assert best["pml_split"] == 3 and step3(b) and b.tuning() == best
    b.run(1)
    for up in (False, True):  # another batch, tuned before and after its upload
        c = xf.Batch([scene(18, 5)])
        if up:
            c.upload().set_tuning(tile_y=2, planes=3)
            assert not step3(c)
            assert (c.tuning()["tile_y"], c.tuning()["planes"], c.tuning()["pml_split"]) == (2, 3, 1)
        again(c, best)
        c.upload().run(1)
        assert step3(c), c.describe()
        c.close()
    # a tuning of the two passes stays one
    b.set_tuning(tile_y=2, planes=3, pml_split=False)
    two = b.tuning()
    assert not step3(b) and two["pml_split"] == 0
    again(b, two)
    assert not step3(b) and b.tuning() == two
    # ... and back; an engine's finding does as well
    again(b, xf.Engine(scene(16)).upload().autotune(2))
    assert step3(b)
    b.run(2).download()
    for s, w in zip(sims, want):
        assert all(np.array_equal(x, y) for x, y in zip(saved(s), w))
    # without the form: the two passes, and the tuning says so
    b = xf.Batch([scene(18, rows=300)]).upload()
    again(b, best)
    assert not step3(b) and b.tuning()["pml_split"] == 1
    for bad in (-1, 4):
        t = xf.simulation.XfTuning(1, 4, 0, 1, 0, bad, 0, 0.0)
        assert b._lib.xf_batch_set_tuning(b._h, ctypes.byref(t)) != 0
    """)
