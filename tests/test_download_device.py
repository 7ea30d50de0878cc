"""A download from a handle whose device is not the calling thread's current
one: the staging slots' events belong to the handle's stream.  The engine's
host code on a runtime in host memory (cpp/fake_hip.cpp), whose events know
their device; the kernels do nothing there, so what comes back is what was
uploaded."""
from test_second_sets import _run, fake  # noqa: F401


def test_download_takes_the_handle_device(fake):  # noqa: F811
    _run(fake, """
    import threading
    fake.fake_devices(2)
    sims = [scene(20, q) for q in range(3)]
    want = [saved(s) for s in sims]
    handles = [xf.Engine(sims[0], device=1).upload(), xf.Batch(sims[1:], device=1).upload()]
    def download(h):
        fake.hipSetDevice(0)  # as another handle's or the caller's own work leaves it
        try:
            h.download()
        except xf.XFError as err:
            errors.append(str(err))
    errors = []
    for h in handles:
        h.run(3)
        for s in sims:
            for f in FIELDS:
                s.array(f)[...] = 0
        download(h)
        t = threading.Thread(target=download, args=(h,))  # a thread begins on device 0
        t.start()
        t.join()
        for s, w in (list(zip(sims, want))[:1] if h is handles[0] else list(zip(sims, want))[1:]):
            assert errors or all(np.array_equal(x, y) for x, y in zip(saved(s), w))
        h.close()
    assert not errors, errors
    """)
