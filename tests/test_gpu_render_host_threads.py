"""muonx_render_host from several threads on one context, which stages every film
in one device buffer. Bar: each film has the bits of the call made alone."""
import ctypes as C
import threading

import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from muon_amd import Context, DeviceScene, HostScene, scenes  # noqa: E402
from muon_amd import _lib  # noqa: E402


def _render(ds, p):
    film = np.full((p.height, p.width, 3), -1.0, np.float32)
    st = _lib.TraceStatsC()
    _lib.check(_lib.lib.muonx_render_host(ds.h, C.byref(p), film.ctypes.data, C.byref(st)))
    return film


def test_threads_share_the_staging_film():
    """Films of growing sizes, so that the buffer moves, by two integrators."""
    ctx = Context(0)
    jobs = []
    for k, (w, h) in enumerate([(31, 17), (64, 48), (200, 100), (333, 241)]):
        hs = HostScene.from_text(scenes.cornell_text(w, h, 2, 3, seed=k))
        p = hs.params
        p.integrator = 0 if k & 1 else 5  # normals, path tracer
        jobs.append((DeviceScene(ctx, hs), p))
    want = [_render(*j) for j in jobs]
    fresh = Context(0)
    jobs = [(DeviceScene(fresh, HostScene.from_text(scenes.cornell_text(p.width, p.height, 2, 3, seed=k))), p)
            for k, (_, p) in enumerate(jobs)]
    bad = []

    def work(k):
        for rep in range(8):
            j = (k + rep) % len(jobs)
            try:
                if not np.array_equal(_render(*jobs[j]), want[j]):
                    bad.append((k, rep, "film"))
            except Exception as e:  # noqa: BLE001
                bad.append((k, rep, e))

    threads = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
