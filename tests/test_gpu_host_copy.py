"""Host arrays through the library's staged copies, byte for byte: below the
size the runtime copies itself, in one and several pieces of one thread, and in
the pieces of two threads with a last piece of odd size."""
import numpy as np
import pytest

import iroiro_amd as ii

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def idle_slots():
    """A context that has copied enough to have a set of pinned slots: the
    contexts of a test take it from their first copy on."""
    ctx = ii.Context((8, 8, 8, 16))
    u = np.zeros(72 * ctx.V)
    for _ in range(32):
        ctx.upload_gauge(u)
    yield
    ctx.close()


@pytest.mark.parametrize("dims", [(2, 2, 2, 2), (4, 4, 4, 8), (6, 4, 2, 10), (8, 8, 8, 16),
                                  (14, 10, 12, 18), (22, 14, 18, 26)])
def test_field_and_gauge_round_trip(dims):
    ctx = ii.Context(dims)
    f = ii.DeviceField(ctx, "full", 2)
    rng = np.random.default_rng(1)
    a, b = rng.normal(size=f.size), rng.normal(size=f.size)
    f.upload(0, a)
    f.upload(1, b)
    assert np.array_equal(f.download(1), b)
    assert np.array_equal(f.download(0), a)
    u = rng.normal(size=72 * ctx.V)
    ctx.upload_gauge(u)
    assert np.array_equal(ctx.download_gauge(), u)
    ctx.close()


def test_two_contexts_of_a_device_copying_at_once():
    """An upload of one context beside another context's download, each in a
    thread of its own, byte for byte; the slots given up by both and taken
    again."""
    import threading
    dims = (14, 10, 12, 18)  # 5.8 MB a field
    for _ in range(2):
        ctxs = [ii.Context(dims) for _ in range(2)]
        bad = []

        def work(k):
            rng = np.random.default_rng(10 + k)
            f = ii.DeviceField(ctxs[k], "full", 1)
            for i in range(16):  # 186 MB: the second context pins slots of its own on the way
                a = rng.normal(size=f.size)
                f.upload(0, a)
                if not np.array_equal(f.download(0), a):
                    bad.append((k, i))

        ts = [threading.Thread(target=work, args=(k,)) for k in range(2)]
        for t in ts:
            t.start()
        for t in ts:
            t.join()
        for c in ctxs:
            c.close()
        assert not bad
